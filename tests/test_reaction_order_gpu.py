"""Mechanisms of five species whose reactions come in another order than the shipped ones.

The rate code with a mechanism's structure is chosen by its rows in their order, so the same
reactions in another order, or more or fewer of them, take the row walk with a bound of 5, 6 or 8
reactions.  The chemistry of the reordered mechanism is compared with that of the shipped one:
the two differ by the rounding of sums alone, and the bars are those of the other walks (1e-12
for the state, for the suggested step 1e-10 with alpha-QSS and 1e-8 with RKF).  The
two-temperature reactor is compared with the oracle on the same reordered mechanism, with the
bars of its parity test: identical status and counts, and no field further off than 10 times
what last bits of the input move the oracle."""
import copy

import numpy as np
import pytest

from gdtk_amd import chemcases
from gdtk_amd import data as gdata
from gdtk_amd.chem import Chemistry, gas_record, mech_record
from gdtk_amd.two_temp import TwoTemperatureReactor
from tests.parity import TOL
from tests.test_tt_gpu import FIELDS, _cell_errors, _cells, _setup

pytestmark = pytest.mark.gpu


def _ordered(md, order):
    return dict(md, reactions=[copy.deepcopy(md["reactions"][k]) for k in order])


@pytest.mark.parametrize("method,tight", [("alpha-qss", False), ("alpha-qss", True), ("rkf", False)])
@pytest.mark.parametrize("n", [1, 63, 320])
def test_air_reactions_in_another_order(method, tight, n):
    gas, shipped = gas_record(gdata.load("tpg-air-5sp")), gdata.load("park-air-5sp-1T")
    c = chemcases.air_cells(n, seed=n, T_hi=8500.0, p_hi=2.0e5)
    c["dt_chem"] = np.where(np.arange(n) % 3 == 0, -1.0, 2.0e-9)
    out = []
    for md in (shipped, _ordered(shipped, (4, 2, 0, 3, 1))):
        ch = Chemistry(gas, mech_record(md, method=method, errTol=1.0e-3, tightTempCoupling=int(tight)))
        r = ch.step(c["rho"], c["T"], c["u"], c["p"], c["massf"], c["dt_chem"], 2.0e-8)
        out.append((r, ch.substeps(n)))
        ch.close()
    (a, sub_a), (b, sub_b) = out
    assert np.all(a["status"] == 0) and np.array_equal(a["status"], b["status"]) and np.array_equal(sub_a, sub_b)
    bar = {"dt_chem": 1.0e-10 if method == "alpha-qss" else 1.0e-8}
    for k in ("T", "u", "p", "massf", "dt_chem"):
        scale = np.maximum(np.abs(a[k]), 1.0e-8 * np.max(np.abs(a[k])))
        assert np.max(np.abs(a[k] - b[k]) / scale) <= bar.get(k, 1.0e-12), k


@pytest.mark.parametrize("order", [(5, 3, 1, 0, 2, 4), (0, 1, 2, 3), (3, 0, 1, 2, 4, 5, 5, 5)])
def test_two_temperature_reactions_in_another_order(order):
    """Six reactions in another order, four of them, and eight (the last one's rate in thirds)."""
    from oracle import oracle as O
    _, shipped, gas, _, prm, mol, A = _setup()
    md = _ordered(shipped, order)
    for r in md["reactions"]:
        parts = sum(q["reactants"] == r["reactants"] and q["products"] == r["products"] for q in md["reactions"])
        for k in ("frc", "brc"):
            r[k]["A"] /= parts
    mech = mech_record(md)
    n, dt = 512, 1.0e-7
    c = _cells(n, seed=len(order))

    def oracle(c):
        return O.tt_step_batch(gas, mech, mol, A, c["rho"], c["T"], c["Tv"], c["u"], c["uv"], c["p"], c["massf"],
                               c["dt_chem"], dt, nthreads=16)
    r = TwoTemperatureReactor(gas, mech, prm)
    g = r.step(c["rho"], c["T"], c["Tv"], c["u"], c["uv"], c["p"], c["massf"], c["dt_chem"], dt)
    st = r.stats()
    r.close()
    o = oracle(c)
    moved = [oracle(dict(c, T=c["T"] * (1.0 + 1e-15))), oracle(dict(c, T=c["T"] * (1.0 - 1e-15))),
             oracle(dict(c, uv=c["uv"] * (1.0 + 1e-15)))]
    assert np.array_equal(g["status"], o["status"])
    assert st["substeps_total"] == int(o["substeps"].sum()) and st["attempts_total"] == int(o["attempts"].sum())
    ok = o["status"] == 0
    for q in moved:
        ok &= q["status"] == 0
    assert ok.mean() > 0.95
    for k in FIELDS:
        e = _cell_errors(g[k], o[k], n)[ok]
        e_self = np.max([_cell_errors(q[k], o[k], n)[ok] for q in moved], axis=0)
        assert e.max() <= max(TOL, 10.0 * float(e_self.max())), k
        assert np.count_nonzero(e > TOL) <= 2 * np.count_nonzero(e_self > TOL) + 0.01 * n, k
