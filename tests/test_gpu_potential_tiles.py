"""The potential's chains where their tiles (2048 elements) begin and end, and masses that
the parallel chains leave to the repair, against the oracle's recurrence bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(cm, O, cl):
    o = O.Oracle(cl.a, cl.n, orbit_r=cl.rtid, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64)
    n = o.potential_calculate()
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        ng, mt, rt = ctx.potential()
        d = ctx.download()
        mid = 0.5 * (cl["r"][1:n] + cl["r"][2:n + 1])
        at = ctx.potential_at(mid) if mid.size else mid
    assert (ng, mt) == (n, o.sc("Mtotal"))
    assert abs(rt / o.sc("Rtidal") - 1) < 1e-15
    assert np.array_equal(d["phi"][:n + 2], o["phi"][:n + 2])
    assert np.array_equal(at, np.array([o.potential(x) for x in mid[:50]] + list(at[50:])))


@pytest.mark.parametrize("n", [2, 3, 9, 2047, 2048, 2049, 2050, 4096, 4097, 6145, 65537])
@pytest.mark.parametrize("kroupa", [False, True])
def test_gpu_potential_tile_edges(gpu, O, n, kroupa):
    print("[gpu-test] potential", n, kroupa, flush=True)
    _check(gpu, O, gpu.make_plummer(n, seed=n, kroupa=kroupa))


@pytest.mark.parametrize("where", ["first", "last", "spread"])
def test_gpu_potential_of_negative_masses(gpu, O, where):
    print("[gpu-test] potential with negative masses", where, flush=True)
    cl = gpu.make_plummer(5000, seed=2, kroupa=True)
    k = {"first": [1], "last": [5000], "spread": [7, 2048, 2049, 4000]}[where]
    cl["m"][k] *= -0.5
    _check(gpu, O, cl)
