"""The marches cut a line into chunks whose length depends on the block's size
(march_cut, csrc/k_fused.hip).  Every face is formed from the same values by
the same operations whatever the chunk, given its position along the line
modulo 32, so a periodic block that repeats a
small one of 32 nodes a line along eta and zeta takes the small block's step
bit for bit: the small block runs chunks of 1 node, the larger ones up to 32.
The rows along xi are laid end to end over the wavefronts, so row ends fall on
every lane.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import (BUF_Q, F_MET, F_Q, FORM_FP32, FORM_FP64, FORM_HYBRID, G,
                                   Block)

pytestmark = pytest.mark.gpu

N0 = 32  # nodes of the small block along eta and zeta


def tiled(f, reps):
    """Ghosted periodic fields (n, ...) of the small block -> the larger one's."""
    inner = f[:, G:-G, G:-G, :]
    big = np.tile(inner, (1, reps, reps, 1))
    return np.pad(big, ((0, 0), (G, G), (G, G), (0, 0)), mode="wrap")


def start(case, form, met=None, q=None):
    b = Block(case.params)
    b.calc_metrics(case.x, case.y, case.z, case.period)
    if met is not None:
        b.set_field(F_MET, met)
        b.set_field(F_Q, q)
    else:
        b.set_conservative(cases.q_ref_aos(case))
    b.set_bc_calc_primitive(BUF_Q)
    if form & FORM_HYBRID:
        # a network of zeros flags no face: every face linear
        b.set_indicator(np.zeros(2145, dtype=np.float32), 1.0)
    b.set_form(form)
    return b


@pytest.mark.parametrize("viscous", [0, 1])
@pytest.mark.parametrize("form", [FORM_FP64, FORM_FP32, FORM_FP32 | FORM_HYBRID])
@pytest.mark.parametrize("im,reps", [(67, 2), (67, 3), (67, 5), (67, 8), (5, 3), (58, 2), (129, 2)])
def test_repeated_block_steps_alike(im, reps, form, viscous):
    small = start(cases.smooth_box(im, N0, N0, viscous=viscous), form)
    try:
        met, q = small.get_field(F_MET, 10), small.get_field(F_Q, 5)
        _, dt0 = small.rk3_step(1e9, 0.0)
        ref = small.get_field(F_Q, 5)
    finally:
        small.free()
    big = start(cases.smooth_box(im, N0 * reps, N0 * reps, viscous=viscous), form,
                tiled(met, reps), tiled(q, reps))
    try:
        _, dt1 = big.rk3_step(1e9, 0.0)
        out = big.get_field(F_Q, 5)
    finally:
        big.free()
    assert dt0 == dt1
    assert np.array_equal(out, tiled(ref, reps))
