"""The reports on masses some of which are negative, so that the enclosed mass is not monotone
and a fraction's first star is no bisection's answer: against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PC = np.array([1e-3, 0.01, 0.05, 0.1, 0.2, 0.3, 0.31, 0.32, 0.4, 0.5, 0.6, 0.7, 0.8, 0.9, 0.95, 0.99, 1.2])


@pytest.mark.parametrize("n", [61, 500, 20000])
@pytest.mark.parametrize("where", ["inner", "outer", "many"])
def test_gpu_reports_of_negative_masses(gpu, O, n, where):
    cm = gpu
    print("[gpu-test] negative masses", n, where, flush=True)
    cl = cm.make_plummer(n, seed=n, kroupa=True)
    m = cl["m"]
    if where == "inner":
        m[n // 5:n // 5 + n // 20] *= -5.0
    elif where == "outer":
        m[int(0.6 * n):int(0.7 * n)] *= -4.0
    else:
        m[1 + np.random.default_rng(n).integers(0, n, n // 3)] *= -1.0
    o = O.Oracle(cl.a, n, orbit_r=cl.rtid)
    o.potential_calculate()
    want = [o.comp_mass_percent(PC, bh_include=b) for b in (0, 1)]
    try:
        cen = o.central_calculate()
    except Exception:
        cen = None
    with cm.Context(n, cm.default_params(n, orbit_r=cl.rtid)) as ctx:
        ctx.upload(cl)
        ctx.potential()
        got = [ctx.comp_mass_percent(PC, bh_include=b) for b in (0, 1)]
        try:
            dev = ctx.central_calculate()
        except cm.CmcgError:
            dev = None
        cl["m"][1:n + 1] = np.abs(cl["m"][1:n + 1])              # the next call is an ordinary one again
        ctx.upload(cl)
        ctx.potential()
        plain = ctx.comp_mass_percent(PC)
        ctx.central_calculate()
    for g, w in zip(got, want):
        assert g["reached"] == int(np.sum(w["no_star_r"] >= 0))
        for k in ("no_star_r", "mass_r", "ave_mass_r", "ke_rad_r", "ke_tan_r", "v2_rad_r", "v2_tan_r"):
            assert np.array_equal(g[k], w[k], equal_nan=True), k
    if dev is not None:                                          # negative terms are refused
        assert cen is not None and dev["nave"] == cen["nave"] and dev["rh"] == cen["rh"]
    o2 = O.Oracle(cl.a, n, orbit_r=cl.rtid)
    o2.potential_calculate()
    assert np.array_equal(plain["no_star_r"], o2.comp_mass_percent(PC)["no_star_r"])
