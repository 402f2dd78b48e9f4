"""Ghost cells written by the cell update against the fill of their own.

Captured steps let the thread that updates a cell write the ghost cells that copy it;
set_graph(False) fills them before each stage.  Both write the same numbers, so everything agrees
bit for bit: where one cell serves several sides (blocks two cells wide), at walls of skewed
grids, at exchanges, inflows and outflows, in one run and over several with steps
of a given size or single stages in between."""
import numpy as np
import pytest

from gdtk_amd import cases

pytestmark = pytest.mark.gpu


def _blocks(kind):
    if kind == "tube":  # slip walls all round, some blocks two cells wide
        c = cases.perturb_vertices(cases.sod_2d(37, 21), amp=0.2, seed=4)
        return 2, cases.split_block(c, (0, 2, 19, 35, 37), (0, 2, 4, 21))
    if kind == "box":  # inflow and outflow, skewed
        c = cases.perturb_vertices(cases.mach6_box(70, 9, 1, seed=5, dims=2), amp=0.15, seed=6)
        return 2, cases.split_block(c, (0, 33, 68, 70), (0, 2, 9))
    c = cases.mach6_box(9, 8, 7, seed=8)  # 3-D: filled, whichever way
    c.bc = [c.bc[0], c.bc[1]] + [cases.BC_SLIP_WALL] * 4
    return 3, cases.split_block(c, (0, 2, 9), (0, 5, 8), (0, 2, 4, 7))


@pytest.mark.parametrize("kind", ["tube", "box", "duct"])
@pytest.mark.parametrize("flux", ["ausmdv", "efm", "adaptive_hanel_ausmdv"])
def test_pushed_ghosts_equal_filled(kind, flux):
    from gdtk_amd import Simulation
    dims, blocks = _blocks(kind)
    sims = []
    for graph in (True, False):
        s = Simulation(dims, flux=flux, fused=False, dt_init=1e-6, cfl_count=4)
        for b in blocks:
            s.add_block(b)
        s.set_graph(graph)
        sims.append(s)
    a, b = sims

    def same():
        assert a.state() == b.state()
        for q in range(len(blocks)):
            for name in ("rho", "vx", "vy", "vz", "u", "p", "T", "a"):
                x = a.get(q, name)
                assert np.isfinite(x).all() and np.array_equal(x, b.get(q, name)), (q, name)
            assert np.array_equal(a.get_U(q), b.get_U(q)), q

    for n in (1, 11, 3):
        assert a.run(n) == b.run(n)
        same()
    for s in sims:  # steps of their own and single stages between two runs
        s.step_fixed_dt(0.5 * s.state()["dt"])
    same()
    assert a.run(6) == b.run(6)
    same()
    dt = b.state()["dt"]
    assert [a.stage(k, dt) for k in (1, 2)] == [b.stage(k, dt) for k in (1, 2)]
    assert a.run(5) == b.run(5)
    same()
