"""The surrogate's kernels at the edges of their workgroups: inference and routing.

Inference: cell counts around a wave's 16 cells and a workgroup's 128 (64 for the small
network) give, cell by cell, the values of one large call bit for bit (a cell's arithmetic does
not depend on its place), and those agree with float64 arithmetic on the same BF16 operands.
Routing: the list of network cells (any order) and the paths are those of the rule, for counts
around a workgroup's 1024 cells, with none, some and all of the cells on the list."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tests.test_surrogate_gpu import _bf16_forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,n_hidden", [(64, 2), (256, 3)])
@pytest.mark.parametrize("n_in,n_out", [(8, 5), (1, 1), (32, 16)])
def test_inference_does_not_depend_on_place(hidden, n_hidden, n_in, n_out):
    import torch
    from gdtk_amd.surrogate import Mlp
    net = Mlp(n_in, n_out, hidden=hidden, n_hidden=n_hidden, seed=5)
    lay, _ = MO.layout(n_in, hidden, n_hidden, n_out)
    dev = torch.device("cuda:0")
    N = 1100
    X = np.random.default_rng(2).normal(size=(N, n_in)).astype(np.float32)

    def run(rows):
        xs = torch.tensor(np.ascontiguousarray(X[rows].T), device=dev)
        ys = torch.full((n_out, len(rows)), 7.0, dtype=torch.float32, device=dev)
        net.infer(len(rows), xs.data_ptr(), ys.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return ys.cpu().numpy().T

    whole = run(np.arange(N))
    ref = _bf16_forward(net.get_params().astype(np.float64), lay, X)
    # a BF16 activation one rounding away (2^-8 of it) in one of the layers' sums of `hidden`
    # terms of random sign: a few 1e-3 of the output's size
    assert np.max(np.abs(whole - ref)) <= 2e-2 * max(1.0, np.max(np.abs(ref)))
    for n in (1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 1023):
        rows = np.random.default_rng(n).permutation(N)[:n]
        assert np.array_equal(run(rows), whole[rows]), n


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("route_T", [1.0e9, 5000.0, 0.0])
def test_routing_around_a_workgroup(n, route_T):
    import torch
    from gdtk_amd import data as gdata
    from gdtk_amd.chem import Chemistry, gas_record, mech_record
    from gdtk_amd.chemcases import air_cells
    from gdtk_amd.surrogate import Mlp, Surrogate, SurrogateCfg, air_element_matrix, integrator_samples
    gd = gdata.load("tpg-air-5sp")
    ch = Chemistry(gas_record(gd), mech_record(gdata.load("park-air-5sp-1T")))
    nets = [Mlp(8, 5, hidden=64, n_hidden=2, seed=3) for _ in range(2)]
    E = air_element_matrix(gd["species"], gd["M"])
    cfg = SurrogateCfg(x_abs_max=1.0e6, disagree_tol=1.0, n_elem=E.shape[0], route_ratio=10.0, route_T=route_T)
    for k in range(8):
        cfg.x_inv_std[k] = 1.0
    for e in range(E.shape[0]):  # y_scale 0: the networks' answer is no change
        for k in range(5):
            cfg.elem[e][k] = E[e, k]
    sur = Surrogate(ch, nets[0], nets[1], cfg)
    c = air_cells(n, seed=n)
    c["T"][: n // 5] = 250.0
    want = np.where(c["T"] <= 300.0, 2, np.where(c["T"] > route_T, 0, 1))
    dev = torch.device("cuda:0")
    t_in = integrator_samples(ch, c, 1.0e-9, dev)[0]
    out = {k: torch.empty_like(t_in[k]) for k in ("T", "u", "p", "massf")}
    dtc = torch.full((n,), -1.0, dtype=torch.float64, device=dev)
    dto = torch.empty_like(dtc)
    st, path = (torch.full((n,), 9, dtype=torch.int32, device=dev) for _ in range(2))
    sur.step_device(n, t_in["rho"].data_ptr(), t_in["T"].data_ptr(), t_in["u"].data_ptr(), t_in["p"].data_ptr(),
                    t_in["massf"].data_ptr(), dtc.data_ptr(), 1.0e-9, out["T"].data_ptr(), out["u"].data_ptr(),
                    out["p"].data_ptr(), out["massf"].data_ptr(), dto.data_ptr(), st.data_ptr(), path.data_ptr(),
                    torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert np.array_equal(path.cpu().numpy(), want)
    assert (st.cpu().numpy() == 0).all()
    s = sur.stats()
    assert s["network_cells"] == (want == 0).sum() and s["fallback"] == 0
    # no change to the cells of the list, each of them and no other
    Y0, Y = t_in["massf"].cpu().numpy().reshape(5, n), out["massf"].cpu().numpy().reshape(5, n)
    assert np.array_equal(Y[:, want == 0], Y0[:, want == 0])
