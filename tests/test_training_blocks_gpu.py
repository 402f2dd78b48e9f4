"""The training kernels at the edges of their cell blocks, row blocks and batch shares.

k_mlp_pass works on 16 cells and 16 rows at a time and k_mlp_weight_grad on 64 x 64 tiles over
shares of the batch, so batches and widths on both sides of those sizes are compared with the
float64 oracle.  Every value is a chain of FP32 sums of at most 256 products a layer: for the
output and the loss a relative error of a few hundred roundings of 6e-8 at worst, 1e-5 with the
activations' own error; for the gradients, sums over layers of such factors, 1e-4 of the
largest entry."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


def _data(n, n_in, n_out, seed=1):
    rng = np.random.default_rng(seed)
    return rng.normal(size=(n, n_in)).astype(np.float32), rng.normal(size=(n, n_out)).astype(np.float32)


@pytest.mark.parametrize("hidden,n_hidden", [(64, 2), (256, 3)])
@pytest.mark.parametrize("batch", [1, 15, 16, 17, 64, 65, 1009])
@pytest.mark.parametrize("n_in,n_out", [(1, 1), (16, 16), (17, 4), (32, 5)])
def test_gradients_over_block_edges(hidden, n_hidden, batch, n_in, n_out):
    from gdtk_amd.surrogate import Mlp
    net = Mlp(n_in, n_out, hidden=hidden, n_hidden=n_hidden, seed=7)
    lay, _ = MO.layout(n_in, hidden, n_hidden, n_out)
    p = net.get_params().astype(np.float64)
    X, Y = _data(batch, n_in, n_out)
    y_ref = MO.forward(p, lay, X.astype(np.float64))[0]
    y = net.forward(X)
    assert np.max(np.abs(y - y_ref)) <= 1e-5 * max(1.0, np.max(np.abs(y_ref)))
    loss_ref, g_ref = MO.loss_grad(p, lay, X.astype(np.float64), Y.astype(np.float64))
    loss, g = net.loss_grad(X, Y)
    assert abs(loss - loss_ref) <= 1e-5 * loss_ref
    assert np.max(np.abs(g - g_ref)) <= 1e-4 * np.max(np.abs(g_ref))
    # a smaller batch in the buffers of a larger one
    if batch > 16:
        loss, g2 = net.loss_grad(X[:16], Y[:16])
        loss_ref, g_ref = MO.loss_grad(p, lay, X[:16].astype(np.float64), Y[:16].astype(np.float64))
        assert abs(loss - loss_ref) <= 1e-5 * loss_ref
        assert np.max(np.abs(g2 - g_ref)) <= 1e-4 * np.max(np.abs(g_ref))


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("n,batch", [(40, 40), (100, 33), (2000, 1000)])
def test_training_steps_are_adam_on_the_batch_gradients(bf16, n, batch):
    """train() gathers rows by index and adds the batch shares inside the update; the same
    steps from loss_grad() with Adam in float64 on the host.  One batch is the whole set in
    some order, so the gradient does not depend on the shuffle; with more, the losses of the
    epoch bound what a wrong gather would change."""
    import torch
    from gdtk_amd.surrogate import Mlp
    X, Y = _data(n, 8, 5, seed=3)
    dev = torch.device("cuda:0")
    xs, ys = (torch.tensor(np.ascontiguousarray(a.T), device=dev) for a in (X, Y))
    torch.cuda.synchronize()
    net, ref = Mlp(8, 5, seed=9), Mlp(8, 5, seed=9)
    for m in (net, ref):
        m.set_bf16_training(bf16)
    p0 = net.get_params().astype(np.float64)
    hist = net.train(n, xs.data_ptr(), ys.data_ptr(), batch=batch, epochs=1, lr=1e-3, seed=4)
    p1 = net.get_params().astype(np.float64)
    if batch == n:
        loss, g = ref.loss_grad(X, Y)
        assert abs(hist[0] - loss) <= 1e-6 * loss
        g = g.astype(np.float64)
        step = 1e-3 * g / (np.abs(g) + 1e-8)  # the first step of Adam: m / c1 = g, v / c2 = g^2
        # an entry's step differs where its gradient is within rounding (1e-6 of the largest) of 0
        sure = np.abs(g) > 1e-3 * np.max(np.abs(g))
        assert np.max(np.abs(p1 - (p0 - step))[sure]) <= 1e-5 * 1e-3 + 1e-7
    assert np.all(np.abs(p1 - p0) <= 1.01e-3 * (n // batch) + 1e-7) and np.isfinite(p1).all()
    # the update leaves the rounded weights as a fresh rounding does
    ref.set_params(net.get_params())
    assert np.array_equal(net.forward(X[:64]), ref.forward(X[:64]))
    assert np.array_equal(net.loss_grad(X, Y)[1], ref.loss_grad(X, Y)[1])
