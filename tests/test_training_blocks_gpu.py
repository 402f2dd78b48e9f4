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
    some order, so the gradient does not depend on the shuffle; with more, no entry moves
    further than Adam's steps allow (test_epochs_are_adam_in_float64 follows their values)."""
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


def _adam(p, grad, steps, lr):
    """Adam (Kingma & Ba 2015) in float64 with the gradient function grad(p) -> (loss, g)."""
    m, v, losses = np.zeros_like(p), np.zeros_like(p), []
    for t in range(1, steps + 1):
        loss, g = grad(p)
        losses.append(loss)
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - lr * (m / (1.0 - 0.9 ** t)) / (np.sqrt(v / (1.0 - 0.999 ** t)) + 1.0e-8)
    return p, losses


@pytest.mark.parametrize("hidden,n_hidden", [(64, 2), (256, 3)])
@pytest.mark.parametrize("copies,n,batch,epochs", [(False, 48, 48, 6), (False, 1009, 1009, 3),
                                                   (True, 200, 33, 1), (True, 2100, 1000, 3)])
def test_epochs_are_adam_in_float64(hidden, n_hidden, copies, n, batch, epochs):
    """Several updates in a row against the float64 oracle's gradients: every row the same, so
    that all batches are alike whatever the shuffle (a gather past the rows, stale packed weights
    or shares of another batch in any but the first update move the result), or the whole set as
    the batch.  Gradients agree to 1e-4 of the largest entry (above), so where the first gradient
    is more than 1e-2 of the largest an update, which depends on the ratios of an entry's gradients
    alone, is off by at most 1e-2 lr.  Smaller entries may move by up to lr either way; the loss
    depends on them by their gradient times that, and is held to 1e-4."""
    import torch
    from gdtk_amd.surrogate import Mlp
    lr = 1.0e-3
    X, Y = _data(n, 8, 5, seed=6)
    if copies:
        X[:], Y[:] = X[0], Y[0]
    dev = torch.device("cuda:0")
    xs, ys = (torch.tensor(np.ascontiguousarray(a.T), device=dev) for a in (X, Y))
    torch.cuda.synchronize()
    net = Mlp(8, 5, hidden=hidden, n_hidden=n_hidden, seed=11)
    lay, _ = MO.layout(8, hidden, n_hidden, 5)
    p0 = net.get_params().astype(np.float64)
    hist = net.train(n, xs.data_ptr(), ys.data_ptr(), batch=batch, epochs=epochs, lr=lr, seed=4)
    rows = 1 if copies else n
    grad = lambda p: MO.loss_grad(p, lay, X[:rows].astype(np.float64), Y[:rows].astype(np.float64))  # noqa: E731
    per = n // batch
    want, losses = _adam(p0, grad, per * epochs, lr)
    losses = np.array(losses).reshape(epochs, per)
    # the history holds the losses read back: the last of an epoch and every 16th before it
    assert np.max(np.abs(hist - losses[:, -1]) / losses[:, -1]) <= 1e-4
    g0 = np.abs(grad(p0)[1])
    err = np.abs(net.get_params() - want)
    assert np.max(err[g0 > 1e-2 * g0.max()]) <= 1e-2 * lr * per * epochs
