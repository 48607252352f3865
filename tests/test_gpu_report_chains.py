"""The reports' chains run side by side: at the edges of their tiles (2048 elements) and
through the fallback paths, against the oracle; the network's gradient where the ordered sum
over block partials changes its batches of loads; queries from several threads."""
import os
import sys
import threading

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as M  # noqa: E402

pytestmark = pytest.mark.gpu

PC = np.array([1e-4, 1e-3, 1e-3, 0.05, 0.3, 0.5, 0.5, 0.9, 0.99, 0.999, 0.9999])


@pytest.mark.parametrize("n", [40, 2047, 2048, 2049, 4097, 20481])
@pytest.mark.parametrize("drop", [0, 40, 60])
def test_gpu_reports_at_tile_edges(gpu, O, n, drop):
    cm = gpu
    print("[gpu-test] reports", n, drop, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    o = O.Oracle(cl.a, cl.n, orbit_r=cl.rtid)
    o.init()
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid, seed=1)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        ctx.test_hook(cm.HOOK_CHAIN_K_DROP, drop)
        a, c = ctx.comp_mass_percent(PC), ctx.central_calculate()
        b = ctx.comp_mass_percent(PC)                       # the workspace after other chains
    want, central = o.comp_mass_percent(PC), o.central_calculate()
    for d in (a, b):
        assert d["reached"] == int(np.sum(want["no_star_r"] >= 0))
        for k in ("no_star_r", "mass_r", "ave_mass_r", "ke_rad_r", "ke_tan_r", "v2_rad_r", "v2_tan_r"):
            assert np.array_equal(d[k], want[k], equal_nan=True), k
        x, y = d["densities_r"], want["densities_r"]
        fin = ~np.isnan(y)
        assert np.array_equal(np.isnan(x), ~fin) and np.all(np.abs(x[fin] - y[fin]) <= 2 * np.spacing(np.abs(y[fin])))
    assert c["nave"] == central["nave"]
    for k, v in central.items():
        assert c[k] == v, k


@pytest.mark.parametrize("n", [64 * 31 + 1, 64 * 32, 64 * 32 + 1, 64 * 64, 64 * 64 + 1, 64 * 255 + 3, 20001])
def test_gpu_network_gradient_batches(gpu, n):
    """Tolerances of the gradient test: every block within 2e-4 of its largest gradient."""
    print("[gpu-test] gradient", n, flush=True)
    rng = np.random.default_rng(n)
    rows = rng.normal(size=(n, 8)).astype(np.float32)
    nr = np.concatenate([rng.normal(size=6), rng.uniform(0.5, 2.0, 6), rng.normal(size=2),
                         rng.uniform(0.5, 2.0, 2)]).astype(np.float32)
    with gpu.Context(1000, gpu.default_params(1000)) as ctx:
        ctx.mlp_init(seed=11, max_rows=1024)
        th, _ = ctx.mlp_params()
        ctx.mlp_set_params(th, nr)
        loss, g = ctx.mlp_loss_grad(rows)
    x = (rows[:, :6].astype(np.float64) - nr[:6]) / nr[6:12]
    t = (rows[:, 6:].astype(np.float64) - nr[12:14]) / nr[14:16]
    lo, go = M.loss_and_grad(th.astype(np.float64), x, t)
    assert abs(loss - lo) <= 1e-5 * abs(lo) + 1e-7
    bounds = [M.OFF_W1, M.OFF_B1, M.OFF_W2, M.OFF_B2, M.OFF_W3, M.OFF_B3, M.NPARAM]
    for a, b in zip(bounds[:-1], bounds[1:]):
        assert np.max(np.abs(g[a:b] - go[a:b])) <= 2e-4 * (np.max(np.abs(go[a:b])) + 1e-12), (a, b)


def test_gpu_queries_from_threads_and_growing_batches(gpu, O):
    cm = gpu
    print("[gpu-test] queries from threads", flush=True)
    cl = cm.make_plummer(20000, seed=5, kroupa=True)
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        d = ctx.download()
        E = d["E"] + np.where(d["r"] > 0, d["m"] / np.maximum(d["r"], 1e-300), 0.0) / cl.n
        want = {c: ctx.apsides(100, E[100:100 + c], d["J"][100:100 + c]) for c in (1, 300, 7000)}
        pot = ctx.potential_at(d["r"][1:7001])
        alone = ctx.apsides(100, E[100:140], d["J"][100:140], noalloc=True)
        for k, v in alone.items():
            assert np.array_equal(v, want[300][k][:40]), k
        bad = []

        def work(c):
            for _ in range(5):
                got = ctx.apsides(100, E[100:100 + c], d["J"][100:100 + c])
                bad.extend(k for k in got if not np.array_equal(got[k], want[c][k]))
                if not np.array_equal(ctx.potential_at(d["r"][1:7001]), pot):
                    bad.append("potential")

        threads = [threading.Thread(target=work, args=(c,)) for c in (1, 300, 7000, 300)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not bad


@pytest.mark.parametrize("count", [32767, 32768, 32769])
def test_gpu_apsides_batches_packed_and_apart(gpu, count):
    cm = gpu
    print("[gpu-test] apsides batch", count, flush=True)
    cl = cm.make_plummer(40000, seed=5, kroupa=True)
    with cm.Context(cl.n, cm.default_params(cl.n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        d = ctx.download()
        s = slice(7, 7 + count)
        E, J = d["E"][s] + d["m"][s] / d["r"][s] / cl.n, d["J"][s]
        got = ctx.apsides(7, E, J)
        for a in range(0, count, 20000):
            part = ctx.apsides(7 + a, E[a:a + 20000], J[a:a + 20000], noalloc=True)
            for k, v in part.items():
                assert np.array_equal(got[k][a:a + 20000], v), k


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 127, 129, 1000, 80000, 80001])
def test_gpu_network_predictions_at_block_edges(gpu, n):
    """Every row's prediction is its own: a batch of any size gives what rows one by one give,
    and the float64 oracle within 1e-4 of the outputs' scale (FP32 sums of 64 terms)."""
    print("[gpu-test] predictions", n, flush=True)
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, 6)).astype(np.float32)
    nr = np.concatenate([rng.normal(size=6), rng.uniform(0.5, 2.0, 6), rng.normal(size=2),
                         rng.uniform(0.5, 2.0, 2)]).astype(np.float32)
    with gpu.Context(1000, gpu.default_params(1000)) as ctx:
        ctx.mlp_init(seed=5, max_rows=1024)
        th, _ = ctx.mlp_params()
        ctx.mlp_set_params(th, nr)
        y = ctx.mlp_predict(x)
        for k in {0, n // 2, n - 1}:
            assert np.array_equal(ctx.mlp_predict(x[k:k + 1])[0], y[k])
    yo, _ = M.forward(th.astype(np.float64), (x.astype(np.float64) - nr[:6]) / nr[6:12])
    yo = yo * nr[14:16] + nr[12:14]
    assert np.max(np.abs(y - yo)) <= 1e-4 * (1 + np.max(np.abs(yo)))
