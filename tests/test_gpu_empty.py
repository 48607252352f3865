"""A cluster that has lost its last star: the phase calls still answer."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3])
def test_gpu_phases_of_an_empty_cluster(gpu, n):
    cm = gpu
    print("[gpu-test] empty", n, flush=True)
    cl = cm.make_plummer(n, seed=n)
    with cm.Context(n, cm.default_params(n, orbit_r=0.02 * cl.rtid)) as ctx:
        ctx.upload(cl)
        ctx.init_cluster()
        for _ in range(3):
            ctx.step_graph()
        assert ctx.scalars()["n_max"] == 0
        for _ in range(2):
            assert ctx.potential() == (0, 0.0, 0.0)
            assert ctx.sort_by_r() == 0
            ctx.calc_timestep()
            ctx.sigma_r()
            ctx.energy_conservation1()
            ctx.energy_conservation2()
            ctx.tidally_strip_stars()
            ctx.set_velocities3()
            ctx.compute_energy()
        s = ctx.scalars()
        assert s["error"] == 0 and s["n_max"] == 0 and s["Ekin"] == 0.0
