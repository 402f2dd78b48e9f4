"""Fields of a block as the host gets them: cells in order, over the chunks (2^19 cells) that
a plane is brought over in, on both sides of a chunk's end, with remainders."""
import numpy as np
import pytest

from gdtk_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(2, 2, 1), (1024, 512, 1), (1021, 514, 1), (83, 80, 79), (129, 128, 96)])
def test_fields_in_cell_order_over_chunks(n):
    from gdtk_amd import Simulation
    dims = 3 if n[2] > 1 else 2
    case = cases.mach6_box(*n, seed=3, dims=dims)
    s = Simulation(dims, flux="adaptive_hanel_ausmdv")
    s.add_block(case)
    # before any step the state is the one given: p, T exactly as encoded and decoded (a few
    # roundings), every cell with a value of its own, so a misplaced one shows
    for name, want in (("p", case.p), ("T", case.T), ("vx", case.vel[:, 0])):
        assert np.max(np.abs(s.get(0, name) - want) / np.abs(want)) <= 1e-14, name
    assert np.max(np.abs(s.get_U(0)[:, 0] - s.get(0, "rho"))) == 0.0
    assert np.array_equal(s.get(0, "S"), np.zeros(case.ncells))
    assert np.max(np.abs(s.get(0, "volume") - 1.0)) <= 1e-12
