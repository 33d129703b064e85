"""The gradient pass at the edges of its work split: a wavefront takes 16 samples
an iteration, 256 workgroups of 8 wavefronts an iteration of 32,768
(k_mlp_grad, csrc/k_learned.hip).  Loss and gradient against the oracle's
bf16-mode network at the bars of the other sizes, the same bits on every call,
and Adam's operand tiles (a forward pass after the step) against those packed
from the stepped parameters.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd.block import DeviceArray, Mlp
from test_gpu_learned import random_features, random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 129, 32768, 32769, 65537])
def test_gradient_at_split_edges(oracle, n):
    print("mlp grad n", n, flush=True)
    P = random_params(5)
    X, y = random_features(6, n)
    m = Mlp(P)
    dX, dY = DeviceArray.from_host(X), DeviceArray.from_host(y)
    loss, g = m.loss_grad(dX.ptr, dY.ptr, n, w_pos=4.0, want_grad=True)
    loss2, g2 = m.loss_grad(dX.ptr, dY.ptr, n, w_pos=4.0, want_grad=True)
    assert loss == loss2 and np.array_equal(g, g2)
    loss_o, g_o = oracle.mlp_loss_grad(P, X, y, w_pos=4.0, bf16=True)
    assert loss == pytest.approx(loss_o, rel=1e-5)
    assert np.linalg.norm(g - g_o) <= 1e-3 * np.linalg.norm(g_o)
    m.adam_step(1e-2)
    d_out = DeviceArray((n,))
    m.forward(dX.ptr, n, d_out.ptr)
    fresh = Mlp(m.get_params())  # its tiles packed by set_params
    d_ref = DeviceArray((n,))
    fresh.forward(dX.ptr, n, d_ref.ptr)
    assert np.array_equal(d_out.download(), d_ref.download())
