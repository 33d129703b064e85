"""Inside a step of a periodic viscous block the flux pass of stages 2 and 3 takes
u, v, w, T from the stage input's conservative state (flux_pass_from_q,
csrc/cbns_internal.hpp); blocks with boundary rules, and the stages called one by
one, read the primitives.  Both are the same values, so a step equals the three
stages with its dt bit for bit: sizes around the pass's 60-node rows, 4-row tiles
and chunks of 2 and 5 planes, and on either side of the tiles and of the ghosts
that they write.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import (BC_PERIODIC, BC_REF, BUF_Q, F_PRIM, F_Q, FORM_FP32, FORM_FP64,
                                   FORM_HYBRID, Block)

pytestmark = pytest.mark.gpu

P, R = BC_PERIODIC, BC_REF


@pytest.mark.parametrize("form", [FORM_FP64, FORM_FP32, FORM_FP32 | FORM_HYBRID])
@pytest.mark.parametrize("size,bc", [((5, 5, 5), (P, P, P)), ((61, 9, 11), (P, P, P)),
                                     ((60, 61, 60), (P, P, P)), ((119, 130, 120), (P, P, P)),
                                     ((61, 34, 36), (R, P, P))])
def test_step_equals_its_stages(size, bc, form):
    case = cases.smooth_box(*size, viscous=1, bc=bc)
    out = []
    for by_stages in (False, True):
        b = Block(case.params)
        try:
            b.calc_metrics(case.x, case.y, case.z, case.period)
            b.set_conservative(cases.q_ref_aos(case))
            b.set_bc_calc_primitive(BUF_Q)
            if form & FORM_HYBRID:
                b.set_indicator(np.zeros(2145, dtype=np.float32), 1.0)
            b.set_form(form)
            for _ in range(2):
                if by_stages:
                    dt = b.calc_dt()
                    for s in (1, 2, 3):
                        b.rk3_stage(dt, s)
                else:
                    b.rk3_step(1e9, 0.0)
            out.append((b.get_field(F_Q, 5), b.get_field(F_PRIM, 6)))
        finally:
            b.free()
    for a, c in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, c)
