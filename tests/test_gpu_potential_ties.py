"""The potential's chains where many elements round to even: equal masses m / N whose mantissa
ends in zeros tie over a whole binade of the enclosed mass, more of them than a block's LDS
lists; against the oracle's recurrence bit for bit, and in time.  (With chain_k_drop the widened
bound makes such lists of ordinary masses.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _zeros(n_star):
    """Trailing zeros of the mantissa of 1 / n_star."""
    m = int(np.ldexp(np.frexp(1.0 / n_star)[0], 53))
    return (m & -m).bit_length() - 1


def _check(cm, O, cl, n_star, ctx):
    o = O.Oracle(cl.a, cl.n, n_star=n_star, orbit_r=cl.rtid, rng_mode=O.RNG_PER_STAR, q_mode=O.Q_FP64)
    n = o.potential_calculate()
    ctx.upload(cl)
    ng, mt, _ = ctx.potential()
    d = ctx.download(fields=["phi"])
    assert (ng, mt) == (n, o.sc("Mtotal"))
    assert np.array_equal(d["phi"][:n + 2], o["phi"][:n + 2])


# ties: about 2 ** zeros of them
@pytest.mark.parametrize("n_star,zeros", [(204800, 0), (201911, 11), (209563, 12), (211990, 13), (209716, 14), (201961, 15),
                                          (246241, 16), (262145, 17)])
def test_gpu_potential_of_tied_masses(gpu, O, n_star, zeros):
    cm = gpu
    print("[gpu-test] tied masses", n_star, zeros, flush=True)
    if zeros:
        assert _zeros(n_star) == zeros
    cl = cm.make_plummer(n_star, seed=1)
    assert np.all(cl["m"][1:n_star + 1] == cl["m"][1])
    cl["m"][1:n_star + 1] = 1.0
    with cm.Context(cl.n, cm.default_params(n_star, orbit_r=cl.rtid)) as ctx:
        _check(cm, O, cl, n_star, ctx)


@pytest.mark.parametrize("n", [4096, 20000, 70000])
@pytest.mark.parametrize("drop", [20, 30, 34, 38])
def test_gpu_potential_of_long_lists(gpu, O, n, drop):
    cm = gpu
    print("[gpu-test] long lists", n, drop, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    with cm.Context(n, cm.default_params(n, orbit_r=cl.rtid)) as ctx:
        ctx.test_hook(1, drop)
        _check(cm, O, cl, n, ctx)


def test_gpu_potential_of_tied_masses_stays_parallel(gpu):
    """2e5 ties among 1e6 stars: 5.1 ms; 28 when one thread ran the three chains, 0.09 without ties."""
    cm = gpu
    ms = {}
    for n_star in (1048581, 1048580):
        cl = cm.make_plummer(n_star, seed=1)
        cl["m"][1:n_star + 1] = 1.0
        with cm.Context(cl.n, cm.default_params(n_star, orbit_r=cl.rtid)) as ctx:
            ctx.upload(cl)
            ctx.timer_enable(True)
            t = []
            for _ in range(4):
                ctx.timer_reset()
                ctx.potential()
                t.append(ctx.timer_get("potential")[0])
            ms[n_star] = min(t[1:])
    print("[gpu-test] potential ms", ms, flush=True)
    assert _zeros(1048580) == 17 and _zeros(1048581) < 4
    assert ms[1048580] < 150 * ms[1048581]
