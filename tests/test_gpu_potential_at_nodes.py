"""potential_at between nodes over the whole cluster, at the places where the potential's tiles
(2048 elements, counted from the outermost star) meet, against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 50, 2048, 2049, 4097, 20000, 65537])
def test_gpu_potential_at_tile_edges(gpu, O, n):
    cm = gpu
    print("[gpu-test] potential_at", n, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    o = O.Oracle(cl.a, cl.n, orbit_r=cl.rtid, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64)
    N = o.potential_calculate()
    edges = [N - 2048 * t + s for t in range(N // 2048 + 1) for s in (-2, -1, 0, 1, 2)]
    k = np.array(sorted(set(edges) | set(np.linspace(1, N - 1, 60).astype(int)) | {1, 2, N - 2, N - 1}))
    k = k[(k >= 1) & (k < N)]
    r = cl["r"]
    x = np.concatenate([0.5 * (r[k] + r[k + 1]), r[k], [0.5 * r[1], 2.0 * r[N], 1e8]])
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        assert ctx.potential()[0] == N
        got = ctx.potential_at(x)
    assert np.array_equal(got, np.array([o.potential(float(v)) for v in x]))
