"""Small periodic blocks: the last march of a stage writes the ghosts with the
state (stage_wraps, csrc/cbns_internal.hpp).  They are copies, so every ghost of
Q and of the primitives equals the node it wraps to, bit for bit: blocks of 8
nodes (each one in the ghosts' reach), ragged ones, the largest that takes this
way, and beyond its limits the fill.  A step that ends in NaN leaves them so too.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import (BUF_Q, F_PRIM, F_Q, F_QP, FORM_FP32, FORM_FP64, FORM_HYBRID, G,
                                   Block, CbnsError)

pytestmark = pytest.mark.gpu

FORMS = [FORM_FP64, FORM_FP32, FORM_FP64 | FORM_HYBRID, FORM_FP32 | FORM_HYBRID]


def wrapped(f):
    return np.pad(f[:, G:-G, G:-G, G:-G], ((0, 0),) + ((G, G),) * 3, mode="wrap")


@pytest.mark.parametrize("viscous", [0, 1])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("size", [(8, 8, 8), (9, 13, 8), (70, 8, 11), (56, 56, 56), (57, 56, 56),
                                  (7, 8, 9)])
def test_ghosts_are_copies(size, form, viscous):
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
        q0 = b.get_field(F_Q, 5)
        for stage in (1, 2, 3):
            b.rk3_stage(1e-4, stage)
            f = b.get_field(F_Q if stage == 3 else F_QP, 5)
            assert not np.array_equal(f, q0)
            assert np.array_equal(f, wrapped(f))
            prim = b.get_field(F_PRIM, n)
            assert np.array_equal(prim, wrapped(prim))
        b.rk3_step(1e9, 0.0)
        f, prim = b.get_field(F_Q, 5), b.get_field(F_PRIM, n)
        assert np.array_equal(f, wrapped(f)) and np.array_equal(prim, wrapped(prim))
        prim[4, G + 3, G + 2, G + 1] = np.nan
        f[:, 0] += 1.0  # ghosts of their own: the fill takes them back
        b.set_field(F_PRIM, prim)
        b.set_field(F_Q, f)
        with pytest.raises(CbnsError):
            b.rk3_step(1e9, 0.0)
        after = b.get_field(F_Q, 5)
        assert np.array_equal(after, wrapped(f))
    finally:
        b.free()
