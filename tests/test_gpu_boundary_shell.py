"""Boundary rules and ghost fill in one launch (k_shell, csrc/k_bc.hip) against
the oracle's ordered phases (src/primitive_bc_kernel.cu:13-494), bit for bit
over the whole ghosted extent: every mix of rules and periodic axes, the
smallest block, ghosts that no rule writes holding values of their own, and wake
cuts whose mirror images meet the wall, meet each other or are absent.
"""
import itertools

import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import BC_PERIODIC, BC_REF, BUF_Q, F_PRIM, F_Q, Block
from helpers import oracle_params

pytestmark = pytest.mark.gpu

MIXES = list(itertools.product((BC_REF, BC_PERIODIC), repeat=3))
SIZES = [(5, 5, 5), (13, 6, 9), (66, 7, 5)]
# (i_begin, i_end) as parts of IM: none, C-grid, wall over the mirror images,
# wall up to the end, cuts past the middle, all wake
COLUMNS = [(0, 0), (0.25, 0.75), (0.3, 1.0), (0.2, 2.0), (0.7, 0.8), (3.0, 3.0)]


@pytest.mark.parametrize("viscous", [0, 1])
@pytest.mark.parametrize("size", SIZES)
def test_every_mix_bit_exact(oracle, size, viscous):
    for bc, (first, last) in itertools.product(MIXES, COLUMNS):
        if bc[1] == BC_PERIODIC and (first, last) != COLUMNS[0]:
            continue  # no eta = 0 rule
        case = cases.smooth_box(*size, viscous=viscous, bc=bc)
        case.params.i_begin = int(first * size[0])
        case.params.i_end = int(last * size[0])
        o = oracle.Oracle(oracle_params(oracle, case))
        o.set_mesh(case.x, case.y, case.z, case.period)
        rng = np.random.default_rng(5)
        o.Q[...] = 0.1 * rng.standard_normal(o.Q.shape)
        o.Q[0] += 1.0
        o.Q[4] += 20.0
        o.prim[...] = rng.standard_normal(o.prim.shape)
        b = Block(case.params)
        try:
            b.calc_metrics(case.x, case.y, case.z, case.period)
            b.set_field(F_Q, o.Q)
            b.set_field(F_PRIM, o.prim)
            o.bc_primitive()
            b.set_bc_calc_primitive(BUF_Q)
            n = 6 if viscous else 5
            what = "bc %s columns %s" % (bc, (first, last))
            assert np.array_equal(b.get_field(F_Q, 5), o.Q), what
            assert np.array_equal(b.get_field(F_PRIM, n), o.prim[:n]), what
        finally:
            b.free()
