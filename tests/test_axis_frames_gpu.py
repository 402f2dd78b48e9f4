"""Faces of grids along the axes against the rotations of the general path.

The face kernel of a grid whose lines follow the axes exchanges the velocity components
instead of rotating them.  What the exchange leaves out are products with one and sums with
zero, so the two agree bit for bit (a signed zero compares equal).  Two general paths are at
hand: the fused stage kernel, which rotates with every face's own frame (AUSMDV and EFM with the
Eilmer 4 numerics; the other calculators run the face kernel on both sides of that comparison),
over the right-handed turns of the axes, block extents from the smallest up
to past a wavefront, stretched spacings, a transverse velocity in every direction, and where one
vertex off the lines sends a direction the general way; and the face kernel itself on a grid
bent at one corner, which sends all its faces the general way, in the cells that the bend has
not reached."""
import numpy as np
import pytest

from gdtk_amd import cases

pytestmark = pytest.mark.gpu

TURNS = {
    "xyz": [[1, 0, 0], [0, 1, 0], [0, 0, 1]],
    "quarter": [[0, -1, 0], [1, 0, 0], [0, 0, 1]],
    "half": [[-1, 0, 0], [0, -1, 0], [0, 0, 1]],
    "cyclic": [[0, 0, 1], [1, 0, 0], [0, 1, 0]],
    "flipped": [[0, 0, -1], [0, -1, 0], [-1, 0, 0]],
}


def _case(dims, n, turn, bent):
    case = cases.mach6_box(*n, seed=17, dims=dims)
    rng = np.random.default_rng(5)
    case.vel += 120.0 * rng.standard_normal(case.vel.shape) * (np.arange(3) < dims)
    v = case.vertices
    for q in range(dims):
        v[:, q] += 0.03 * v[:, q] ** 2 / n[q]
    if bent:  # the last vertex of all: outside, so the faces next to it only
        v[-1, :dims] += 0.07
    P = np.array(TURNS[turn], dtype=float)
    case.vertices = v @ P.T
    case.vel = case.vel @ P.T
    case.inflow[:, 2:5] = case.inflow[:, 2:5] @ P.T
    return case


@pytest.mark.parametrize("dims,n,turn", [
    (2, (2, 2, 1), "xyz"), (2, (70, 5, 1), "quarter"), (2, (9, 67, 1), "half"),
    (3, (2, 2, 2), "cyclic"), (3, (17, 9, 6), "xyz"), (3, (5, 66, 3), "quarter"),
    (3, (13, 4, 9), "cyclic"), (3, (6, 7, 8), "flipped")])
@pytest.mark.parametrize("flux", ["ausmdv", "hanel", "adaptive_hanel_ausmdv", "adaptive_efm_ausmdv", "efm"])
@pytest.mark.parametrize("bent", [False, True])
def test_exchanged_components_equal_rotated(dims, n, turn, flux, bent):
    from gdtk_amd import Simulation
    case = _case(dims, n, turn, bent)
    a, b = (Simulation(dims, flux=flux, fused=f, dt_init=1e-6) for f in (False, True))
    for s in (a, b):
        s.add_block(case)
        s.run(4)
    assert a.state() == b.state()
    for name in ("rho", "vx", "vy", "vz", "u", "p", "T", "a"):
        x = a.get(0, name)
        assert np.isfinite(x).all() and np.array_equal(x, b.get(0, name)), name
    assert np.array_equal(a.get_U(0), b.get_U(0))


@pytest.mark.parametrize("dims,n,turn", [
    (2, (24, 19, 1), "xyz"), (2, (18, 70, 1), "quarter"), (2, (67, 21, 1), "half"),
    (3, (18, 19, 17), "xyz"), (3, (17, 16, 33), "quarter"), (3, (66, 16, 17), "cyclic"), (3, (16, 18, 20), "flipped")])
@pytest.mark.parametrize("flux", ["ausmdv", "hanel", "adaptive_hanel_ausmdv"])
@pytest.mark.parametrize("numerics", ["eilmer4", "lmr"])
def test_exchanged_components_equal_a_bent_grids(dims, n, turn, flux, numerics):
    """Bending the last vertex gives the faces around it a frame of their own in every direction,
    so no direction of that block exchanges components.  What the last cell's shape changes
    travels two cells a stage (a face reads two cells to either side, and the indicators of its own
    two cells, which their neighbours decide): eight cells in two steps of two stages, counted
    along the axes."""
    from gdtk_amd import Simulation
    out = []
    for bent in (False, True):
        s = Simulation(dims, flux=flux, numerics=numerics, fused=False, dt_init=1e-6)
        s.add_block(_case(dims, n, turn, bent))
        for _ in range(2):
            s.step_fixed_dt(2.0e-5)
        out.append(s)
    from_first = np.indices(n[dims - 1::-1]).sum(axis=0).reshape(-1)
    far = from_first < sum(n[:dims]) - dims - 8
    assert far.sum() > 0.8 * far.size
    for name in ("rho", "vx", "vy", "vz", "u", "p", "T", "a"):
        x, y = out[0].get(0, name), out[1].get(0, name)
        assert np.isfinite(x).all() and np.array_equal(x[far], y[far]), name
        assert name == "vz" and dims == 2 or not np.array_equal(x, y), name
    assert np.array_equal(out[0].get_U(0)[far], out[1].get_U(0)[far])
