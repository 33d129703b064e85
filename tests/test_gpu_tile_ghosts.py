"""Periodic blocks that run by tiles write their ghosts with the state while they are
small (stage_wraps, csrc/cbns_internal.hpp: at most 2^20 stored nodes), beyond that by the
fill.  Either way a ghost of Q or of a primitive is the node it wraps to, bit for bit.
Blocks on both sides of the limit, and ragged ones of both shapes of tile; the profile
says who filled: the fill counts a launch a stage.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import (BUF_Q, F_PRIM, F_Q, F_QP, FORM_FP32, FORM_FP64, FORM_HYBRID, G,
                                   Block)

pytestmark = pytest.mark.gpu


def wrapped(f):
    return np.pad(f[:, G:-G, G:-G, G:-G], ((0, 0),) + ((G, G),) * 3, mode="wrap")


@pytest.mark.parametrize("viscous,form", [(0, FORM_FP64), (1, FORM_FP64), (1, FORM_FP32),
                                          (1, FORM_FP32 | FORM_HYBRID)])
@pytest.mark.parametrize("size,fill", [((93, 93, 93), False), ((94, 94, 93), True),
                                       ((67, 61, 53), False), ((33, 50, 29), False)])
def test_ghosts_are_copies(size, fill, viscous, form):
    case = cases.smooth_box(*size, viscous=viscous)
    n = 6 if viscous else 5
    b = Block(case.params)
    try:
        b.calc_metrics(case.x, case.y, case.z, case.period)
        b.set_conservative(cases.q_ref_aos(case))
        b.set_bc_calc_primitive(BUF_Q)
        if form & FORM_HYBRID:
            b.set_indicator(np.zeros(2145, dtype=np.float32), 1.0)
        b.set_form(form)
        b.set_profiling(True)
        for stage in (1, 2, 3):
            b.rk3_stage(1e-4, stage)
            f, prim = b.get_field(F_Q if stage == 3 else F_QP, 5), b.get_field(F_PRIM, n)
            assert np.array_equal(f, wrapped(f)) and np.array_equal(prim, wrapped(prim))
        b.rk3_step(1e9, 0.0)
        f, prim = b.get_field(F_Q, 5), b.get_field(F_PRIM, n)
        assert np.array_equal(f, wrapped(f)) and np.array_equal(prim, wrapped(prim))
        t = b.kernel_times()
        assert t["bc"][1] == (6 if fill else 0)
        assert t["march_eta"][1] == 0
    finally:
        b.free()
