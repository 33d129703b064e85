"""The ring of pinned buffers is made when the blocks of the process have read enough
for it (csrc/host_copy.hip): reads before, at and after that point, one large read,
and a program that makes and frees a block for each of its reads.  Bytes stay bytes.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import F_Q, Block

pytestmark = pytest.mark.gpu


def _block(size, seed):
    b = Block(cases.smooth_box(*size, viscous=0).params)
    q = np.random.default_rng(seed).standard_normal((5,) + tuple(b.shape))
    b.set_field(F_Q, q)
    return b, q


# five fields of 4.2, 15 and 38 MB (whole: no parts), and 83 MB, worth the ring alone
@pytest.mark.parametrize("size,reads", [((38, 40, 40), 18), ((64, 64, 64), 7), ((92, 92, 90), 4),
                                        ((120, 120, 120), 2)])
def test_reads_until_past_the_ring(size, reads):
    b, q = _block(size, 1)
    try:
        for _ in range(reads):
            assert np.array_equal(b.get_field(F_Q, 5), q)
    finally:
        b.free()


def test_a_block_for_every_read():
    for seed in range(6):
        b, q = _block((64, 64, 64), seed)
        try:
            assert np.array_equal(b.get_field(F_Q, 5), q)
        finally:
            b.free()
