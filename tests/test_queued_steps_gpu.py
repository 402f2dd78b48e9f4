"""Steps queued without the host between them against steps checked one by one.

set_graph(False) runs the stages kernel by kernel with the host's checks after each; the two
paths launch the same kernels on the same numbers, so fields, time, dt and step agree bit for
bit: over queues that end at a time-step estimate, at the last step and at max_time; where a
step in the middle of a queue fails and is repeated at a smaller dt (a Courant number above the
scheme's limit); and where a run is given up."""
import numpy as np
import pytest

from gdtk_amd import cases
from gdtk_amd import data as gdata

pytestmark = pytest.mark.gpu


def _sim(kind, graph, **kw):
    from gdtk_amd import Simulation
    from gdtk_amd.chem import Chemistry, mech_record
    if kind == "tube":
        c = cases.sod_2d(60, 30)
        blocks = cases.split_block(c, (0, 17, 41, 60), (0, 13, 30))
        s = Simulation(2, fused=False, dt_init=1e-6, **kw)
    elif kind == "fused":
        blocks = [cases.sod_2d(60, 30)]
        s = Simulation(2, dt_init=1e-6, **kw)
    elif kind == "shock":
        blocks = [cases.wedge_2d(24, 20)]
        s = Simulation(2, flux="adaptive_hanel_ausmdv", dt_init=1e-6, **kw)
    else:
        blocks, rec, _ = cases.cylinder_blocks(24, 10, 2)
        s = Simulation(2, tpg=rec, dt_init=1e-9, dt_max=1e-6, **kw)
    for b in blocks:
        s.add_block(b)
    if kind == "reacting":
        s.set_chemistry(Chemistry(rec, mech_record(gdata.load("park-air-5sp-1T"))))
    s.set_graph(graph)
    return s, len(blocks)


def _fields(s, nb):
    names = ["rho", "vx", "vy", "u", "p", "T"] + [300 + k for k in range(s.nsp if s.nsp > 1 else 0)]
    return [s.get(q, n) for q in range(nb) for n in names] + [s.get_U(q) for q in range(nb)]


def _same(a, b, nb):
    assert a.state() == b.state()
    for x, y in zip(_fields(a, nb), _fields(b, nb)):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("kind", ["tube", "fused", "shock", "reacting"])
@pytest.mark.parametrize("cfl_count", [1, 7, 40])
def test_queues_of_any_length_equal_single_steps(kind, cfl_count):
    (a, nb), (b, _) = (_sim(kind, g, cfl_count=cfl_count) for g in (True, False))
    for n in (1, 5, 23):
        assert a.run(n) == b.run(n)
        _same(a, b, nb)
    t = b.state()["time"] + 3.5 * b.state()["dt"]  # reached inside a queue
    ra, rb = a.run(100, t), b.run(100, t)
    assert ra == rb and ra[0] == 4
    _same(a, b, nb)


@pytest.mark.parametrize("kind", ["tube", "fused", "shock", "reacting"])
@pytest.mark.parametrize("cfl", [2.0, 4.0, 6.0])
def test_a_failed_step_inside_a_queue_is_repeated(kind, cfl):
    """dt starts at a Courant number too large for the flow that develops and holds for 40
    steps unless a step fails; some of these runs meet too many bad cells and end there."""
    out, sims = [], []
    for graph in (True, False):
        s, nb = _sim(kind, graph, cfl_count=40, max_attempts_for_step=5)
        dt = cfl * min(s.block_dt(q, 1.0, 1.0, False)[0] for q in range(nb))
        s.set_dt(dt, 1)
        try:
            out.append(s.run(30))
        except Exception as e:
            out.append(str(e))
        sims.append(s)
    assert out[0] == out[1]
    assert sims[0].state()["dt"] < 0.9 * dt  # some step was repeated
    assert sims[0].state() == sims[1].state()
    if not isinstance(out[0], str):
        _same(sims[0], sims[1], nb)


def test_a_run_that_cannot_be_saved_is_given_up():
    (a, nb), (b, _) = (_sim("tube", g, max_attempts_for_step=1) for g in (True, False))
    for s in (a, b):
        s.set_dt(40.0 * s.block_dt(0, 1.0, 0.5, False)[0], 1)
        with pytest.raises(Exception, match="giving up"):
            s.run(8)
    _same(a, b, nb)
    dt = 0.2 * a.block_dt(0, 1.0, 0.5, False)[0]
    for s in (a, b):  # and the simulation goes on from where the step started
        s.step_fixed_dt(dt)
    _same(a, b, nb)
