"""Small blocks run a stage by tiles (k_tile4, k_tile16, csrc/k_fused.hip).  Against
the oracle on the same stage inputs: the smallest block, updated ranges that fill
the tiles exactly and that leave one node over along each axis, for both shapes of
tile, and every kind of axis.  1e-12 of each quantity's own scale, as for any stage
(momentum components that are small against the others at the largest one's).
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import BC_PERIODIC, BC_REF, F_PRIM, F_Q, F_QP, Block
from helpers import oracle_block, rel_err_state, update_mask

pytestmark = pytest.mark.gpu

P, R = BC_PERIODIC, BC_REF
# 4-node tiles up to 1024 of them, else 16 x 4 x 4
SIZES = [(5, 5, 5), (8, 4 + 2, 4 + 3), (16, 17, 18), (49, 45, 46), (64, 36, 40), (67, 35, 36)]


@pytest.mark.parametrize("viscous,centered", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("bc", [(P, P, P), (R, P, P), (P, R, P), (P, P, R), (R, R, R)])
@pytest.mark.parametrize("size", SIZES)
def test_stages_match_oracle(oracle, size, bc, viscous, centered):
    case = cases.smooth_box(*size, viscous=viscous, bc=bc, visc_centered=centered)
    o = oracle_block(oracle, case)
    o.bc_primitive()
    b = Block(case.params)
    try:
        b.calc_metrics(case.x, case.y, case.z, case.period)
        m = update_mask(case)
        for s in (1, 2, 3):
            b.set_field(F_Q, o.Q)
            b.set_field(F_QP, o.Qp)
            b.set_field(F_PRIM, o.prim)
            o.rk3_stage(1e-3, s)
            b.rk3_stage(1e-3, s)
            ref = o.Q if s == 3 else o.Qp
            out = b.get_field(F_Q if s == 3 else F_QP, 5)
            assert np.isfinite(out[:, m]).all()
            assert rel_err_state(out[:, m], ref[:, m]) < 1e-12, s
    finally:
        b.free()
