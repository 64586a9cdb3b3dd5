"""Gradients of the surrogate's training kernels at the edges of their batches: one sample, whole and ragged groups of
16 samples and of 256 reduction threads, and batches over which the workgroups walk, against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [1, 15, 16, 17, 255, 257, 4096, 16384 + 5, 65536])
def test_gradient_batch_edges(batch):
    import mlp_oracle as mo

    from chapsim2_amd.initial import heated_channel_table
    from chapsim2_amd.mlp import Surrogate
    from chapsim2_amd.props import PropertyTable

    pt = PropertyTable(heated_channel_table(4096), -1.0)
    net = Surrogate(pt, nsamples=4096, seed=9)
    try:
        rng = np.random.default_rng(batch)
        x = rng.uniform(-1, 1, batch).astype(np.float32)
        t = rng.normal(0, 1, (batch, 5)).astype(np.float32)
        loss, g = net.grad(x, t)
        _, p16 = net.params()
        pw = (p16.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        lref, gref = mo.loss_grad(pw, x.astype(np.float64), t.astype(np.float64))
        assert abs(loss - lref) < 1e-5 * lref
        # up to 256 + 8 FP32 additions per entry, of terms sqrt(batch) larger than their sum at most
        tol = 2.0 ** -24 * (batch / 256 + 24) * max(np.sqrt(batch), 16.0)
        assert np.abs(g - gref).max() < tol * np.abs(gref).max()
    finally:
        net.close()
        pt.close()
