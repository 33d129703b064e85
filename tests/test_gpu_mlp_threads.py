"""One network used by two threads: the parameters that a call returns are the
parameters, whatever another thread's gradient pass is handing to the host at the
time (both stage through pinned memory of the network, csrc/k_learned.hip).
"""
import threading

import numpy as np
import pytest

from cbns3d_cuda_amd.block import MLP_NPARAM, DeviceArray, Mlp

pytestmark = pytest.mark.gpu


def test_params_and_gradient_from_two_threads():
    rng = np.random.default_rng(5)
    P = (rng.standard_normal(MLP_NPARAM) * 0.3).astype(np.float32)
    for r in range(32):
        P[r * 32 + 30:r * 32 + 32] = 0  # the padding inputs stay zero
    n = 4096
    X = rng.standard_normal((n, 32)).astype(np.float32)
    X[:, 30:] = 0
    y = (rng.random(n) < 0.3).astype(np.float32)
    m = Mlp(P)
    dX, dY = DeviceArray.from_host(X), DeviceArray.from_host(y)
    loss, grad = m.loss_grad(dX.ptr, dY.ptr, n, 4.0, want_grad=True)
    wrong, done = [], threading.Event()

    def gradients():
        while not done.is_set():
            lg, g = m.loss_grad(dX.ptr, dY.ptr, n, 4.0, want_grad=True)
            if lg != loss or not np.array_equal(g, grad):
                wrong.append("gradient")

    t = threading.Thread(target=gradients)
    t.start()
    try:
        for _ in range(3000):
            if not np.array_equal(m.get_params(), P):
                wrong.append("parameters")
    finally:
        done.set()
        t.join()
    print("wrong", len(wrong), set(wrong), flush=True)
    assert not wrong
    m.free()
