"""The bucket sort where its tiles, buckets and LDS capacities end: star counts around
them, radii that fill one bucket far beyond its capacity, and a step whose radii were not
in order, each against numpy's lexsort of (r, id) or the invariants of a sorted state."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-test]", *a, flush=True)


def _radii(kind, n, rng):
    if kind == "spread":                       # 12 decades, some stars of the SF_INFINITY tail
        r = 10.0 ** rng.uniform(-8, 4, n)
        r[rng.random(n) < 0.03] = 1e10
    elif kind == "clumped":                    # most radii within a few ulps: one key range, many ties
        r = 1.0 + 2.0 ** -50 * rng.integers(0, 40, n)
        r[: n // 8] = rng.uniform(0.1, 10.0, n // 8)
    elif kind == "equal":
        r = np.full(n, 0.75)
    else:                                      # two clumps, one sub-range of keys each
        r = np.where(rng.random(n) < 0.6, 1e-3, 5.0) * (1.0 + 1e-9 * rng.random(n))
    return rng.permutation(r)


@pytest.mark.parametrize("kind", ["spread", "clumped", "equal", "two"])
@pytest.mark.parametrize("n", [1, 2, 63, 511, 513, 1024, 1025, 2049, 4097, 16385, 131072, 131073, 300001])
def test_gpu_sort_edges(gpu, n, kind):
    cm = gpu
    say("sort", n, kind)
    rng = np.random.default_rng(n)
    cl = cm.Cluster(n)
    cl["r"][1:n + 1] = _radii(kind, n, rng)
    cl["id"][1:n + 1] = rng.permutation(n) - n // 2          # negative ids too
    for k in ("m", "vr", "vt", "E", "J", "rnew", "vrnew", "vtnew", "X", "Y", "r_peri", "r_apo", "rOld", "Uoldrold",
              "Uoldrnew", "vrold", "vtold", "EI"):
        cl[k][1:n + 1] = rng.random(n)
    order = 1 + np.lexsort((cl["id"][1:n + 1], cl["r"][1:n + 1]))
    order = order[cl["r"][order] < 1e10]
    with cm.Context(n, cm.default_params(n)) as ctx:
        ctx.upload(cl)
        assert ctx.sort_by_r() == order.size
        d = ctx.download()
    for k in ("r", "id", "m", "vr", "vt", "E", "J", "rnew", "vrnew", "vtnew", "X", "Y", "r_peri", "r_apo", "rOld",
              "Uoldrold", "Uoldrnew", "vrold", "vtold", "EI"):
        assert np.array_equal(d[k][1:order.size + 1], cl[k][order]), k


@pytest.mark.parametrize("n", [3000, 140000])
def test_gpu_step_with_radii_out_of_order_still_sorts(gpu, n):
    """A step that starts from radii out of order reports what it likes about the orbits,
    but ends sorted, with every star once."""
    cm = gpu
    say("step from unordered radii", n)
    cl = cm.make_plummer(n, seed=3)
    with cm.Context(n, cm.default_params(n, orbit_r=cl.rtid, seed=3)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        i, j = n // 3, 2 * n // 3
        d = ctx.download()
        d["r"][[i, j]] = d["r"][[j, i]]
        ctx.upload(d, fields=["r"])
        ctx.step(check=False)
        ctx.set_scalars()                                  # clears the error the bad orbits may have raised
        a = ctx.download()
        m = a.n
        assert np.all(a["r"][1:m] <= a["r"][2:m + 1])
        assert np.unique(a["id"][1:m + 1]).size == m and m > 0.9 * n
        ctx.sort_by_r()
        b = ctx.download()
    assert np.array_equal(a["id"][1:m + 1], b["id"][1:m + 1])
