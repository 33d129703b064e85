"""Reads below the ring's size go in equal parts below 1 MiB (copy_to_host,
csrc/host_copy.hip): every byte lands where one copy would put it, at sizes around one,
two and four parts and around the ring's least, whose parts are no whole fields.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import F_Q, Block

pytestmark = pytest.mark.gpu


# five fields are 0.998 and 1.026 parts at 21x23x21 and 25x21x20, 3.9 at 39x38x39
@pytest.mark.parametrize("size", [(5, 5, 5), (13, 37, 19), (25, 21, 20), (21, 23, 21), (30, 31, 29),
                                  (37, 38, 39), (39, 38, 39), (61, 60, 61)])
def test_fields_come_back_whole(size):
    b = Block(cases.smooth_box(*size, viscous=0).params)
    try:
        q = np.random.default_rng(3).standard_normal((5,) + tuple(b.shape))
        b.set_field(F_Q, q)
        for n in (1, 2, 3, 4, 5):
            assert np.array_equal(np.asarray(b.get_field(F_Q, n)).reshape((n,) + tuple(b.shape)),
                                  q[:n])
    finally:
        b.free()
