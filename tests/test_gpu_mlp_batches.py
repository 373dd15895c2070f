"""The training kernels at batch sizes around their tiles: a single point, sizes that are not a
multiple of 8 (operands read element by element), of the 64-row tile, of the 512-row column-sum
chunks, and enough for several split-K chunks with a ragged last one.  Against the BF16-emulating
oracle at 2e-3 normwise (the training kernels' bound: isolated activations round to neighbouring
BF16 values)."""
import numpy as np
import pytest
import torch

import oracle.mlp as OM
from test_gpu_mlp import _case, _nrel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 63, 64, 65, 250, 511, 513, 1000, 1544, 2051, 4100])
def test_batch_edges(ssc, n):
    from streamsculptor_amd.mlp import MLP
    p, x, t, w = _case(n=n, seed=n)
    net = MLP(params=p)
    print(f"[mlp batch] {n}", flush=True)
    lo, go, yo = OM.loss_and_grad(p, x, t, w, emulate=True)
    for weight, ref in ((w, (lo, go, yo)), (None, OM.loss_and_grad(p, x, t, None, emulate=True))):
        net.grads.fill_(float("nan"))
        loss, y = net.loss_backward(x, t, weight)
        assert abs(loss.item() - ref[0]) <= 2e-3 * abs(ref[0])
        assert _nrel(y, ref[2]) < 2e-3
        assert _nrel(net.grads, ref[1]) < 2e-3
    # the gradient of a given output cotangent: the loss gradient's own
    dy = (2.0 * w[:, None] * (net.forward(x).cpu().numpy() - t) / w.sum()).astype(np.float32)
    assert _nrel(net.vjp(x, dy), go) < 2e-3


def test_workspace_may_start_anywhere(ssc):
    """A workspace that is not 16-byte aligned gives the same bits."""
    from streamsculptor_amd import _lib
    from streamsculptor_amd.mlp import MLP
    p, x, t, w = _case(n=300, seed=3)
    net = MLP(params=p)
    loss, y = net.loss_backward(x, t, w)
    want = net.grads.clone()
    nbytes = _lib.load().ssc_mlp_workspace_bytes(300)
    net._ws, net._ws_n = torch.empty(nbytes + 4, dtype=torch.uint8, device="cuda")[4:], 300
    net.grads.fill_(float("nan"))
    net.loss_backward(x, t, w)
    assert torch.equal(net.grads, want)
