"""The viscous flux pass walks 5 planes a workgroup on blocks that fill the
chip and 2 on smaller ones, and takes one-sided derivatives at the outer layers
of reference axes from loads of their own (dedge, csrc/k_viscous.hip).  Larger
blocks than the other parity cases, with every mix of boundary rules, against
the oracle at its stage bar of 1e-12.
"""
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import BC_PERIODIC, BC_REF, F_PRIM, F_Q, F_QP, Block
from helpers import oracle_block, rel_err_state

pytestmark = pytest.mark.gpu

R, P = BC_REF, BC_PERIODIC


def box(bc, **kw):
    return cases.smooth_box(123, 70, 64, viscous=1, bc=bc, **kw)


CASES = {
    "cgrid": lambda: cases.c_grid_channel(190, 70, 41, viscous=1),
    "rpp": lambda: box((R, P, P)),
    "prp": lambda: box((P, R, P)),
    "ppr_centered": lambda: box((P, P, R), visc_centered=1),
    "ppp": lambda: box((P, P, P)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_stage_matches_oracle(name, oracle):
    case = CASES[name]()
    print("case", case.name, flush=True)
    o = oracle_block(oracle, case)
    o.bc_primitive()
    o.viscous()
    dt = o.calc_dt()
    b = Block(case.params)
    try:
        b.calc_metrics(case.x, case.y, case.z, case.period)
        b.set_field(F_Q, o.Q)
        b.set_field(F_QP, o.Qp)
        b.set_field(F_PRIM, o.prim)
        assert b.calc_dt() == dt
        o.rk3_stage(dt, 1)
        b.rk3_stage(dt, 1)
        assert rel_err_state(b.get_field(F_QP, 5), o.Qp) < 1e-12
    finally:
        b.free()
