"""The sampler and the relaxation where the generator's jumps change digits (blocks of 64
stars, steps) and where the radial index has crowded buckets, against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _upload(ctx, cl, o):
    h = cl.copy()
    for k in ("phi", "E", "J", "sigma"):
        h[k] = o[k]
    ctx.upload(h)
    ctx.set_scalars(n_max=o.N, n_max_new=o.N, Mtotal=o.sc("Mtotal"), Rtidal=o.sc("Rtidal"), TidalMassLoss=0.0,
                    TidalMassLoss_old=0.0, OldTidalMassLoss=0.0, Eescaped=0.0, Jescaped=0.0, Etidal=0.0, Dt=0.0,
                    Prev_Dt=0.0, TotalTime=0.0, step=0)


def _orbits(cm, O, cl, step):
    o = O.Oracle(cl.a, cl.n, orbit_r=cl.rtid, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64)
    o.init()
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid, seed=1)) as ctx:
        _upload(ctx, cl, o)
        st = ctx.orbits(step=step)
        d = ctx.download()
    o.s.step = step
    o.orbits()
    assert st["error"] == o.s.error
    N = o.N
    for k in ("rnew", "vrnew", "vtnew", "r_peri", "r_apo", "X", "ntry"):
        assert np.array_equal(d[k][1:N + 1], o[k][1:N + 1]), k
    assert st["n_circular"] == o.sc("n_circular") and st["max_r"] == o.sc("max_r")


@pytest.mark.parametrize("n,step", [(2, 0), (63, 1), (64, 63), (65, 64), (255, 0), (257, 4095), (4095, 4096), (4097, 4097),
                                    (20000, 2 ** 36 + 5), (262143, 0), (262209, 0)])
def test_gpu_orbit_substreams(gpu, O, n, step):
    print("[gpu-test] orbit substreams", n, step, flush=True)
    _orbits(gpu, O, gpu.make_plummer(n, seed=n, kroupa=True), step)


@pytest.mark.parametrize("share,width", [(0.5, 1e-4), (0.9, 1e-7), (0.99, 1e-10)])
@pytest.mark.parametrize("n", [700, 30000])
def test_gpu_orbits_in_crowded_buckets(gpu, O, n, share, width):
    """A shell that holds most stars: its radii share a few buckets of the radial index."""
    print("[gpu-test] crowded buckets", n, share, width, flush=True)
    cl = gpu.make_plummer(n, seed=4, kroupa=True)
    r = np.array(cl["r"][1:n + 1])
    a, b = int(n * (0.5 - share / 2)), int(n * (0.5 + share / 2))
    r[a:b] = r[a] * (1.0 + width * np.linspace(0.0, 1.0, b - a))
    r[b:] = np.maximum(r[b:], r[b - 1] * (1.0 + 1e-6))
    cl["r"][1:n + 1] = np.sort(r)
    _orbits(gpu, O, cl, 3)


@pytest.mark.parametrize("n,step", [(2, 0), (3, 64), (127, 1), (129, 63), (8191, 4095), (8194, 0), (40001, 2 ** 36 + 5),
                                    (524290, 0)])
def test_gpu_relaxation_substreams(gpu, O, n, step):
    print("[gpu-test] relaxation substreams", n, step, flush=True)
    cl = gpu.make_plummer(n, seed=n, kroupa=True)
    o = O.Oracle(cl.a, cl.n, orbit_r=cl.rtid, rng_mode=O.RNG_PER_STAR, libm_mode=O.LIBM_DD)
    o.init()
    dt = O.lib.orc_simul_relax_new(C.byref(o.s))
    with gpu.Context(cl.n, gpu.default_params(cl.n, orbit_r=cl.rtid, seed=1)) as ctx:
        _upload(ctx, cl, o)
        ctx.relax(dt, step=step)
        d = ctx.download()
    o.s.step = step
    o.relax(dt)
    for k in ("vr", "vt", "E", "J"):
        assert np.array_equal(d[k][1:o.N + 1], o[k][1:o.N + 1]), k
    assert np.array_equal(d["Y"][1:o.N], o["Y"][1:o.N])
