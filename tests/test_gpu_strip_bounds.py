"""The step's stripping passes skip blocks of stars by a bound of their apocentres: an apocentre
that is not a number (a circular orbit keeps the one it had) must not hide its neighbours'."""
import ctypes as C

import numpy as np
import pytest

from cases import near_tangent_stars

pytestmark = pytest.mark.gpu


# one block runs the passes up to 65536 stars, grids beyond
@pytest.mark.parametrize("n", [5000, 66005])
@pytest.mark.parametrize("graph", [False, True])
def test_gpu_strip_beside_apocentres_not_a_number(gpu, O, n, graph):
    cm = gpu
    print("[gpu-test] strip beside NaN", n, graph, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    # no kicks, so the first star of a pair keeps a circular orbit; the orbit phase removes no
    # star beyond the tidal radius (set below), the stripping does
    kw = dict(orbit_r=0.02 * cl.rtid, theta_se_max=1e-30)
    o = O.Oracle(cl.a, cl.n, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64, libm_mode=O.LIBM_DD, **kw)
    o.init()
    near_tangent_stars(o, range(65, o.N - 64, 64), rel_j=(0.0,), vr_choices=(0.0,))
    o["r_apo"][1:o.N + 1] = np.nan
    o.s.Rtidal = 1e9
    h = cm.Cluster(n)
    for k in h.a:
        if k in o.arr:
            h[k] = o[k][:n + 2]
    with cm.Context(n, cm.default_params(n, **kw)) as ctx:
        ctx.upload(h)
        ctx.set_scalars(n_max=n, n_max_new=n, Mtotal=o.sc("Mtotal"), Rtidal=1e9, Etot=o.sc("Etot"), Ekin=o.sc("Ekin"),
                        Epot=o.sc("Epot"), step=0)
        (ctx.step_graph if graph else ctx.step)()
        d, sc = ctx.download(), ctx.scalars()
    assert o.step() == 0
    N = o.N
    assert np.isnan(o["r_apo"][1:N + 1]).sum() > n // 128 and N < 0.97 * n     # the case is what it is meant to be
    assert sc["n_max"] == N
    assert sc["TidalMassLoss"] == pytest.approx(o.sc("TidalMassLoss"), rel=1e-12)
    gi = {int(i): k + 1 for k, i in enumerate(d["id"][1:N + 1])}
    idx = np.array([gi[int(i)] for i in o["id"][1:N + 1]], dtype=np.int64)
    for k in ("r", "vr", "vt", "m", "phi"):
        assert np.array_equal(d[k][idx], o[k][1:N + 1]), k
