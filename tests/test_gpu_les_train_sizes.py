"""Training step of the closure network at batch sizes around the edges of its
reduction: one point, one and two 16-point chunks, the sizes where a layer's
gradient goes from one block to two and to the largest number of blocks, and
sizes that fill none of them.  The step's gradient (whatever number of block
partials it was added up from), its loss, the weights after Adam and the
BF16 operands made from them (through a forward pass) are held against the
separate entries: x3d_mlp_gradient, the Adam formula on that gradient, and a
network set to the new weights.

Gradient and loss of the two entries come from the same kernels and are equal
bit for bit; Adam in FP64 on the FP32 gradient differs by FP32 rounding, at
most 1e-6 of a weight's scale; the forward pass of the trained network equals
that of a network given its weights, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

X = pytest.importorskip("incompact3d_amd")


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 1000, 32767, 32768, 32801])
def test_train_step_equals_its_parts(torch_cuda, n):
    import torch
    from incompact3d_amd import les
    X.init(X.make_params(32, 32, 32))
    try:
        g = torch.Generator(device="cuda")
        g.manual_seed(n)
        x = torch.randn((n, 10), device="cuda", generator=g)
        t = torch.randn((n, 6), device="cuda", generator=g)
        w0 = les.init_params(3)
        a, b = X.Mlp(w0), X.Mlp(w0)
        grad, loss_g = b.gradient(x, t)
        loss = a.train_step(x, t, 1e-3)
        assert loss == loss_g and np.isfinite(loss)
        w1 = a.get_params()
        g64 = grad.astype(np.float64)
        ref = w0 - 1e-3 * g64 / (np.abs(g64) + 1e-8)
        assert np.abs(w1 - ref).max() <= 1e-6
        c = X.Mlp(w1)
        assert torch.equal(a.forward(x), c.forward(x))
        loss2 = a.train_step(x, t, 1e-3)
        assert np.isfinite(loss2) and loss2 == c.gradient(x, t)[1]
        for net in (a, b, c):
            net.close()
    finally:
        X.finalize()
