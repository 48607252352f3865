"""The glue kernels that one block runs for clusters up to 65536 stars, on both sides of that
size: the tidal stripping loop with several passes and the excess-energy chain, in eager and
captured steps and in the phase calls, against the oracle and each other bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("r", "vr", "vt", "E", "J", "m", "phi")


def _order(d, o):
    gi = {int(i): k + 1 for k, i in enumerate(d["id"][1:o.N + 1])}
    return np.array([gi[int(i)] for i in o["id"][1:o.N + 1]], dtype=np.int64)


# a tidal radius well inside the cluster strips stars pass after pass
@pytest.mark.parametrize("n", [3, 255, 1025, 8193, 65536, 65537])
@pytest.mark.parametrize("cut", [1.0, 0.08])
@pytest.mark.parametrize("graph", [False, True])
def test_gpu_strip_and_excess_vs_oracle(gpu, O, n, cut, graph):
    cm = gpu
    print("[gpu-test] strip", n, cut, graph, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    rt = cl.rtid * cut
    o = O.Oracle(cl.a, cl.n, orbit_r=rt, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64, libm_mode=O.LIBM_DD)
    o.init()
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=rt)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        for _ in range(2):
            (ctx.step_graph if graph else ctx.step)()
            assert o.step() == 0
        d, sc = ctx.download(), ctx.scalars()
    assert sc["n_max"] == o.N and sc["Dt"] == o.sc("Dt")
    idx = _order(d, o)
    for k in FIELDS:
        assert np.array_equal(d[k][idx], o[k][1:o.N + 1]), k
    for k in ("Rtidal", "TidalMassLoss", "Eescaped", "Jescaped"):
        assert sc[k] == pytest.approx(o.sc(k), rel=1e-12, abs=1e-300), k


EVENTS = [(0.0, 1.0), (0.01, 2.0), (0.3, 1.5), (2e-3, 2e3)]


@pytest.mark.parametrize("n,p_ev,scale", [(n, *e) for n in (2, 255, 256, 257, 4097, 65535, 65536, 65537, 262145, 278784)
                                          for e in EVENTS] + [(4194304, 0.01, 2.0), (4200000, 0.01, 2.0)])
def test_gpu_excess_chain_sizes(gpu, O, n, p_ev, scale):
    cm = gpu
    print("[gpu-test] excess chain", n, p_ev, scale, flush=True)
    cl = cm.make_plummer(n, seed=11)
    o = O.Oracle(cl.a, cl.n, orbit_r=cl.rtid)
    o.potential_calculate()
    N = o.N
    rng = np.random.default_rng(n)
    v2 = o["vr"][1:N + 1] ** 2 + o["vt"][1:N + 1] ** 2
    ev = rng.random(N) < p_ev
    o["rOld"][1:N + 1] = o["r"][1:N + 1]
    o["vrold"][1:N + 1] = o["vr"][1:N + 1]
    o["vtold"][1:N + 1] = o["vt"][1:N + 1]
    o["Uoldrold"][1:N + 1] = 0.0
    o["Uoldrnew"][1:N + 1] = np.where(ev, v2 * (1.0 + scale * rng.random(N)), v2 * 0.2 * (rng.random(N) - 0.5))
    h = cm.Cluster(N)
    for k in h.a:
        if k in o.arr:
            h[k] = o[k][:N + 2]
    with cm.Context(N, cm.default_params(N, orbit_r=cl.rtid)) as ctx:
        ctx.upload(h)
        ctx.set_scalars(n_max=N, n_max_new=N, Mtotal=o.sc("Mtotal"))
        ctx.set_velocities3()
        d = ctx.download()
        assert ctx.scalars()["error"] == 0
    O.lib.orc_set_velocities3(C.byref(o.s))
    for k in ("vr", "vt", "vrnew", "vtnew"):
        assert np.array_equal(d[k][1:N + 1], o[k][1:N + 1]), k


@pytest.mark.parametrize("n", [64, 65, 66, 129, 130, 195, 4160, 4225, 4226, 8450, 12675])
def test_gpu_old_potential_search_splits(gpu, O, n):
    """set_velocities3's searches split a range of nodes into 65: the potential at the old
    radii, through 4 steps, where the range is a multiple of 65 and its last part holds some."""
    cm = gpu
    print("[gpu-test] old potential", n, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    rt = cl.rtid * 1e3                                # no star leaves
    o = O.Oracle(cl.a, cl.n, orbit_r=rt, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64, libm_mode=O.LIBM_DD)
    o.init()
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=rt)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        for _ in range(4):
            ctx.step()
            assert o.step() == 0
        d = ctx.download()
    idx = _order(d, o)
    for k in FIELDS:
        assert np.array_equal(d[k][idx], o[k][1:o.N + 1]), k


@pytest.mark.parametrize("n,ave", [(1500000, 20), (1500001, 20), (1500640, 5), (1501283, 4), (1500003, 64), (1600637, 1)])
def test_gpu_step_sigma_of_many_stars(gpu, n, ave):
    """The step's sigma and time step on both sides of 1.5e6 stars and for windows shorter and
    longer than a thread's share of stars, against the phase call's kernels."""
    cm = gpu
    print("[gpu-test] step sigma", n, ave, flush=True)
    cl = cm.make_plummer(n, seed=3, kroupa=True)
    got = []
    for step in (False, True):
        with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid, avekernel=ave)) as ctx:
            ctx.upload(cl)
            ctx.init_cluster()
            dt = None if step else ctx.calc_timestep()
            if step:
                ctx.step()
                dt = ctx.scalars()["Dt"]
            got.append((dt, ctx.download(fields=["sigma"])["sigma"][1:n + 1].copy()))
    assert got[0][0] == got[1][0]
    kept = got[1][1].size                             # stars that leave in the step are not downloaded
    assert kept > 0.99 * n and np.array_equal(got[0][1][:kept], got[1][1])
