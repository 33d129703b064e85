"""Stages that run by the marches (k_march, csrc/k_fused.hip) against the oracle on the
same inputs, at the bars of the other parity cases (1e-12 of each quantity's scale; the
precision form 1e-7).  Blocks below about 10^6 nodes go by tiles unless these fit them
badly, so the blocks here are thin, with one node past the tiles along two axes or all
three: long and short rows, chunks from the shortest to the longest, every kind of axis,
and one C-grid of the size that runs.  The profile says which way a stage went: a tile
launch counts as none of the eta march.
"""
import numpy as np
import pytest

from cbns3d_cuda_amd import cases
from cbns3d_cuda_amd.block import (BC_PERIODIC, BC_REF, BUF_Q, F_MET, F_PRIM, F_Q, F_QP, FORM_FP32,
                                   FORM_FP64, FORM_HYBRID, G, MLP_NPARAM, Block)
from helpers import oracle_block, rel_err, rel_err_state

pytestmark = pytest.mark.gpu

P, R = BC_PERIODIC, BC_REF
AXES = [(P, P, P), (R, P, P), (P, R, P), (P, P, R), (R, R, R)]
UPDATED = [(17, 133, 133), (67, 5, 900), (67, 900, 5)]  # updated nodes


def box(updated, bc, viscous, centered=0):
    n = [u if b == P else u + 2 for u, b in zip(updated, bc)]
    return cases.smooth_box(*n, viscous=viscous, bc=bc, visc_centered=centered)


def start(oracle, case):
    o = oracle_block(oracle, case)
    o.bc_primitive()
    if case.params.viscous:
        o.viscous()
    b = Block(case.params)
    b.calc_metrics(case.x, case.y, case.z, case.period)
    b.set_profiling(True)
    return o, b, o.calc_dt()


def put(b, o):
    b.set_field(F_Q, o.Q)
    b.set_field(F_QP, o.Qp)
    b.set_field(F_PRIM, o.prim)


def marched(b):
    return b.kernel_times(reset=True)["march_eta"][1] == 1


def stages_match(oracle, case):
    o, b, dt = start(oracle, case)
    try:
        for s in (1, 2, 3):
            put(b, o)
            o.rk3_stage(dt, s)
            b.rk3_stage(dt, s)
            assert marched(b)
            ref = o.Q if s == 3 else o.Qp
            out = b.get_field(F_Q if s == 3 else F_QP, 5)
            assert np.isfinite(out).all()
            assert rel_err_state(out, ref) < 1e-12, s
            n = 6 if case.params.viscous else 5
            assert rel_err(b.get_field(F_PRIM, 6)[:n], o.prim[:n]) < 1e-12, s
    finally:
        b.free()


@pytest.mark.parametrize("viscous,centered", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("bc", AXES)
@pytest.mark.parametrize("updated", UPDATED)
def test_stages_match_oracle(oracle, updated, bc, viscous, centered):
    stages_match(oracle, box(updated, bc, viscous, centered))


@pytest.mark.parametrize("viscous", [0, 1])
def test_cgrid_matches_oracle(oracle, viscous):
    stages_match(oracle, cases.c_grid_channel(133, 103, 103, viscous=viscous))


@pytest.mark.parametrize("viscous", [0, 1])
@pytest.mark.parametrize("bc", AXES)
@pytest.mark.parametrize("updated", UPDATED)
def test_precision_stage_close_to_oracle(oracle, updated, bc, viscous):
    o, b, dt = start(oracle, box(updated, bc, viscous))
    try:
        b.set_form(FORM_FP32)
        put(b, o)
        o.rk3_stage(dt, 1)
        b.rk3_stage(dt, 1)
        assert marched(b)
        assert rel_err_state(b.get_field(F_QP, 5), o.Qp) < 1e-7
    finally:
        b.free()


def some_faces(seed):
    """A network whose logits lie on both sides of 0 (as in the other hybrid tests)."""
    p = (np.random.default_rng(seed).standard_normal(MLP_NPARAM) * 0.3).astype(np.float32)
    for r in range(32):
        p[r * 32 + 30:r * 32 + 32] = 0
    return p


@pytest.mark.parametrize("form,bar", [(FORM_HYBRID, 1e-12), (FORM_FP32 | FORM_HYBRID, 1e-7)])
@pytest.mark.parametrize("bc", AXES)
@pytest.mark.parametrize("updated", UPDATED)
def test_hybrid_stage_matches_oracle(oracle, updated, bc, form, bar):
    o, b, dt = start(oracle, box(updated, bc, 1))
    try:
        b.set_indicator(some_faces(13), 0.0, full_lists=True)
        b.set_form(form)
        put(b, o)
        b.rk3_stage(dt, 1)
        assert marched(b)
        flags = b.get_flags()
        share = flags.mean()
        print("troubled", share, flush=True)
        assert 0.02 < share < 0.9
        o.rk3_stage_hybrid(dt, 1, flags)
        assert rel_err_state(b.get_field(F_QP, 5), o.Qp) < bar
    finally:
        b.free()


def tiled(f, reps):
    """Ghosted fields (n, ...) repeated along eta and zeta."""
    big = np.tile(f[:, G:-G, G:-G, :], (1, reps, reps, 1))
    return np.pad(big, ((0, 0), (G, G), (G, G), (0, 0)), mode="wrap")


@pytest.mark.parametrize("form", [FORM_FP64, FORM_FP32, FORM_HYBRID, FORM_FP32 | FORM_HYBRID])
@pytest.mark.parametrize("viscous,centered", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("xi", [P, R])
def test_marches_have_the_tiles_bits(xi, viscous, centered, form):
    """A block of 32 nodes along eta and zeta, by tiles, and five of it along each, by
    the marches: the same step, a part of the faces troubled."""
    out = []
    met = q = None
    for n in (32, 160):
        case = cases.smooth_box(67, n, n, viscous=viscous, bc=(xi, P, P), visc_centered=centered)
        b = Block(case.params)
        try:
            b.calc_metrics(case.x, case.y, case.z, case.period)
            if met is None:
                b.set_conservative(cases.q_ref_aos(case))
                b.set_bc_calc_primitive(BUF_Q)
                met, q = b.get_field(F_MET, 10), b.get_field(F_Q, 5)
            else:
                b.set_field(F_MET, tiled(met, 5))
                b.set_field(F_Q, tiled(q, 5))
                b.set_bc_calc_primitive(BUF_Q)
            if form & FORM_HYBRID:
                b.set_indicator(some_faces(13), 0.0, full_lists=True)
            b.set_form(form)
            b.set_profiling(True)
            _, dt = b.rk3_step(1e9, 0.0)
            assert (b.kernel_times()["march_eta"][1] > 0) == (n == 160)
            if form & FORM_HYBRID:
                assert 0.02 < b.get_flags().mean() < 0.9
            out.append((dt, b.get_field(F_Q, 5)))
        finally:
            b.free()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[1][1], tiled(out[0][1], 5))
