"""Fields read back through the shared staging ring (csrc/host_copy.hip).  Bytes
stay bytes, so every comparison is exact.  Five fields of the blocks lie on both
sides of the smallest ring copy (4 MiB) and of the change of piece (32 MiB),
with more pieces than the ring has buffers and a last one that is not full.
"""
import threading

import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import F_MET, F_PRIM, F_Q, F_QP, Block, CbnsError

pytestmark = pytest.mark.gpu

SIZES = [(37, 40, 40), (38, 40, 40), (86, 86, 86), (87, 86, 86), (128, 100, 91)]


def _block(size, seed):
    b = Block(cases.smooth_box(*size, viscous=0).params)
    q = np.random.default_rng(seed).standard_normal((5,) + tuple(b.shape))
    b.set_field(F_Q, q)
    return b, q


@pytest.mark.parametrize("size", SIZES)
def test_fields_come_back_whole(size):
    b, q = _block(size, 1)
    try:
        assert np.array_equal(b.get_field(F_Q, 5), q)
        assert np.array_equal(b.get_field(F_Q + 3), q[3])
        # over the end of an array into the next ones
        b.set_field(F_QP, q[::-1])
        b.set_field(F_PRIM, q + 1.0)
        got = b.get_field(F_Q + 2, F_PRIM + 5 - F_Q - 2)
        assert np.array_equal(got, np.concatenate([q[2:], q[::-1], q + 1.0]))
        with pytest.raises(CbnsError):
            b.get_field(F_MET + 8, 40)  # past the last field
    finally:
        b.free()


def test_blocks_read_by_several_threads():
    blocks = [_block(SIZES[-1], s) for s in range(3)]
    wrong = []

    def read(b, q):
        for _ in range(4):
            if not np.array_equal(b.get_field(F_Q, 5), q):
                wrong.append(b)

    try:
        threads = [threading.Thread(target=read, args=bq) for bq in blocks]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
    finally:
        for b, _ in blocks:
            b.free()
