"""A queue of steps that ends early leaves what the failing step alone would have left.

Steps are queued behind a step whose outcome the host does not know yet.  The same failure is
met with nothing behind it (one step asked for) and with steps behind it, and both runs report
the same error and hold the same state, bit for bit."""
import numpy as np
import pytest

from gdtk_amd import cases
from gdtk_amd import data as gdata

pytestmark = pytest.mark.gpu

AIR = [0.767, 0.233, 0.0, 0.0, 0.0]


def _fields(s, nb):
    names = ["rho", "vx", "vy", "u", "p", "T"] + [300 + k for k in range(s.nsp)]
    return [s.get(q, n) for q in range(nb) for n in names] + [s.get_U(q) for q in range(nb)]


def _same(a, b, nb):
    assert a.state() == b.state()
    for x, y in zip(_fields(a, nb), _fields(b, nb)):
        assert np.array_equal(x, y)


def _resting_columns(numerics):
    """A box of 8 x 4 cells a kilometre wide, at rest at one pressure, so that a step of 1 us
    moves nothing and its chemistry alone changes the cells.  Column 3 (N2 and O at 20000 K)
    dissociates next to frozen columns of N2 and of N2 and O: from then on the Eilmer 5
    reconstruction, which takes the species one by one, has mass fractions on the face between
    columns 2 and 3 that sum to 0.75.  Column 6 (air at 12000 K) is what the integrator fails
    on."""
    from gdtk_amd import Simulation
    from gdtk_amd.chem import Chemistry, mech_record
    rec = cases.air5_gas()
    v = cases.box_vertices(8, 4, 1, 8.0e3, 4.0e3, 0.0, dims=2)
    c = cases.BlockCase(2, 8, 4, 1, v, None, None, None, [cases.BC_SLIP_WALL] * 6)
    mixed = [0.5, 0.0, 0.0, 0.0, 0.5]
    Y = [[1.0, 0.0, 0.0, 0.0, 0.0]] * 2 + [mixed] * 3 + [AIR] * 3
    T = [300.0, 300.0, 300.0, 20000.0, 300.0, 300.0, 12000.0, 300.0]
    c.massf, c.T = np.tile(Y, (4, 1)), np.tile(T, 4)
    c.p, c.vel = np.full(32, 1.0e5), np.zeros((32, 3))
    c.inflow, c.inflow_massf = np.zeros((6, 5)), np.tile(AIR, (6, 1))
    s = Simulation(2, tpg=rec, numerics=numerics, dt_init=1e-6, cfl_count=40)
    s.add_block(c)
    s.set_chemistry(Chemistry(rec, mech_record(gdata.load("park-air-5sp-1T"))))
    s.set_dt(1.0e-6, 1)
    return s


@pytest.mark.parametrize("numerics", ["eilmer4", "lmr"])
@pytest.mark.parametrize("steps", [2, 9, 30])
def test_failed_chemistry_with_steps_behind_it(numerics, steps):
    alone, queued = _resting_columns(numerics), _resting_columns(numerics)
    for s, n in ((alone, 1), (queued, steps)):
        with pytest.raises(Exception, match="thermochemical_increment"):
            s.run(n)
    assert alone.state()["time"] == 1.0e-6
    N2 = alone.get(0, 300)
    assert N2[3] < 1.0e-4 and abs(N2[2] - 0.5) < 1.0e-6  # the contrast is there
    _same(alone, queued, 1)


def _cylinder(queue, cfl):
    from gdtk_amd import Simulation
    blocks, rec, _ = cases.cylinder_blocks(24, 10, 2)
    s = Simulation(2, tpg=rec, dt_init=1e-9, dt_max=1e-6, cfl_count=40, max_attempts_for_step=5)
    for b in blocks:
        s.add_block(b)
    s.set_graph(queue)
    s.set_chemistry(_air_chemistry(rec))
    s.run(7)
    s.set_dt(cfl * min(s.block_dt(q, 1.0, 1.0, False)[0] for q in range(2)), s.state()["step"])
    return s, rec


def _air_chemistry(rec):
    from gdtk_amd.chem import Chemistry, mech_record
    return Chemistry(rec, mech_record(gdata.load("park-air-5sp-1T")))


@pytest.mark.parametrize("cfl", [0.4, 100.0])
def test_reactor_refused_inside_a_queue(cfl):
    """The reactor is closed and the run goes on: the step's flux update is taken (after repeats
    at a smaller dt where the Courant number is too large), its chemistry refused.  Queued or
    step by step, the simulation is left in the same state and goes on from it the same way
    once it has a reactor again."""
    sims = []
    for queue in (True, False):
        s, rec = _cylinder(queue, cfl)
        before = s.state()
        s._chem[0].close()
        with pytest.raises(Exception, match="handle"):
            s.run(12)
        after = s.state()
        assert after["step"] == before["step"] and after["time"] == before["time"] + after["dt"]
        assert (after["attempts"] > 1) == (cfl > 1.0)
        sims.append((s, rec))
    _same(sims[0][0], sims[1][0], 2)
    for s, rec in sims:
        s.set_chemistry(_air_chemistry(rec))
        s.set_dt(1.0e-9, s.state()["step"])
        s.run(20)
    _same(sims[0][0], sims[1][0], 2)
    for q in range(2):
        assert np.array_equal(sims[0][0].get(q, "dt_chem"), sims[1][0].get(q, "dt_chem"))
