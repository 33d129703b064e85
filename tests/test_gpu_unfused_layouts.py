"""The decomposed calls cut their faces and nodes into 64 x 4 tiles or lay the rows end
to end, by the length of the rows (face_cut, node_cut, csrc/k_unfused.hip).  Against the
oracle on the same inputs at the 1e-12 of the other parity cases: rows around both
rules' limits, of one to five tiles, full and with one node over, and planes whose
rows are no multiple of 4.
"""
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import (BC_PERIODIC, BC_REF, BUF_Q, F_FLUX, F_PRIM, F_Q, F_QP, Block)
from helpers import oracle_block, rel_err, rel_err_state, update_mask
from test_gpu_parity import face_mask

pytestmark = pytest.mark.gpu

P, R = BC_PERIODIC, BC_REF
# faces along xi (periodic / reference): one more / one fewer than nodes
ROWS = [5, 24, 25, 26, 51, 52, 53, 63, 64, 65, 88, 89, 103, 128, 154, 193, 205, 258]


@pytest.mark.parametrize("bc", [(P, P, P), (R, R, R)])
@pytest.mark.parametrize("im", ROWS)
def test_fluxes_and_update_match_oracle(oracle, im, bc):
    case = cases.smooth_box(im, 6 + im % 4, 5 + im % 3, viscous=0, bc=bc)
    o = oracle_block(oracle, case)
    o.bc_primitive()
    b = Block(case.params)
    try:
        b.calc_metrics(case.x, case.y, case.z, case.period)
        b.set_field(F_Q, o.Q)
        b.set_field(F_QP, o.Qp)
        b.set_field(F_PRIM, o.prim)
        ref = o.numerical_flux(o.Q)
        b.calc_numerical_flux(BUF_Q)
        flux = b.get_field(F_FLUX, 15).reshape(ref.shape)
        for d in range(3):
            m = face_mask(case, d)
            assert rel_err(flux[d][:, m], ref[d][:, m]) < 1e-12, d
        o.rk3_stage(1e-3, 1)
        b.update_rk3(1e-3, 1)
        m = update_mask(case)
        assert rel_err_state(b.get_field(F_QP, 5)[:, m], o.Qp[:, m]) < 1e-12
    finally:
        b.free()
