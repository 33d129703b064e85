"""The time-step pass cuts a block into workgroups by its size (dt_chunk,
csrc/k_dt.hip) and one workgroup takes the maximum of their maxima.  The
fastest node decides wherever it lies, bit for bit (src/time_step_kernel.cu:
43-94 on uniform metrics), and a NaN anywhere makes the time step NaN.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import F_MET, F_PRIM, G, Block, CbnsError

pytestmark = pytest.mark.gpu

# one node along k a thread; two with a short last walk; 9 to 13 workgroups a
# thread of the last pass
SIZES = [(5, 5, 5), (24, 20, 16), (65, 37, 301), (130, 66, 128), (64, 8, 5000)]


@pytest.mark.parametrize("size", SIZES)
def test_fastest_node_anywhere(size):
    IM, JM, KM = size
    case = cases.smooth_box(IM, JM, KM, viscous=0)
    b = Block(case.params)
    try:
        b.calc_metrics(case.x, case.y, case.z, case.period)
        shape = (KM + 2 * G, JM + 2 * G, IM + 2 * G)
        met = np.zeros((10,) + shape)
        met[0], met[4], met[8], met[9] = 2.0, 3.0, 5.0, 1.0 / 30.0
        b.set_field(F_MET, met)
        prim = np.zeros((6,) + shape)
        prim[0], prim[4] = 1.0, 1.0
        c = np.sqrt(1.4 * 1.0 / 1.0)
        expect = 0.5 / (((7.0 * 2.0) + c * 2.0) + c * 3.0 + c * 5.0)
        for at in ((0, 0, 0), (KM - 1, JM - 1, IM - 1), (KM // 2, JM // 2, IM // 2),
                   (KM - 1, 0, IM // 3)):
            k, j, i = (a + G for a in at)
            prim[1, k, j, i] = 7.0
            b.set_field(F_PRIM, prim)
            assert b.calc_dt() == expect
            prim[1, k, j, i] = np.nan
            b.set_field(F_PRIM, prim)
            with pytest.raises(CbnsError):
                b.calc_dt()
            prim[1, k, j, i] = 0.0
    finally:
        b.free()
