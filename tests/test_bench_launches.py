"""The work that bench.py books for a kernel is that of the launches the library makes
(CPU only): the fields and planes of the flux pass, the ghosts' fields and the faces of
a stage that runs by tiles, each counted here by hand.
"""
import json
import os
import sys
from types import SimpleNamespace

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402

P, R = 1, 0
MARCHES = {"march_eta": (1.0, 3), "march_zeta": (1.0, 3)}
TILES = {"march_eta": (0.0, 0), "march_zeta": (1.0, 3)}


def params(n, bc=(P, P, P), viscous=1):
    return SimpleNamespace(IM=n[0], JM=n[1], KM=n[2], bc=bc, viscous=viscous)


def work(name, p, kt=MARCHES):
    return bench.kernel_work(name, p, **bench.as_run(p, kt))


def test_ghost_fields_of_a_viscous_step():
    # periodic: Q alone in stages 1 and 2, with the six primitives in stage 3;
    # boundary rules: u, v, w, T in stages 1 and 2 too
    shell = 24 ** 3 - 16 ** 3
    assert work("bc", params((16,) * 3)) == ("byte", shell * (5 + 5 + 11) * 16 // 3)
    assert work("bc", params((16,) * 3, (R, P, P))) == ("byte", int(shell * (9 + 9 + 11) * 16 / 3))
    assert work("bc", params((16,) * 3, viscous=0)) == ("byte", int(shell * (5 + 5 + 10) * 16 / 3))


def test_maxima_of_the_flux_pass():
    # 260 nodes: 5 tiles of 60, 65 of 4, 52 chunks of 5; the counters' bytes of that
    # launch hold them and little else
    p = params((256,) * 3)
    assert work("dt", p) == ("byte", 5 * 65 * 52 * 8)
    with open(bench.TRAFFIC_FILE) as f:
        measured = json.load(f)["bytes_per_launch"]["dt"]
    assert work("dt", p)[1] == pytest.approx(measured, rel=0.1)
    # fewer than 448 workgroups of 5 planes, and just over 512 with a reference axis: 2
    assert work("dt", params((32,) * 3)) == ("byte", 1 * 9 * 18 * 8)
    assert work("dt", params((193, 61, 33), (R, R, R))) == ("byte", 4 * 17 * 19 * 8)
    assert work("dt", params((193, 61, 33))) == ("byte", 4 * 17 * 8 * 8)


def test_fields_of_the_flux_pass():
    # 10 metrics, 12 fluxes, and u, v, w, T or Q; rho and p of the block's nodes once a step
    ext, n = 20 ** 3, 16 ** 3
    for bc, fields in (((P, P, P), 4 + 5 + 5), ((P, R, P), 4 + 4 + 4)):
        assert work("visc_flux", params((16,) * 3, bc)) == (
            "byte", (ext * (3 * 22 + fields) + n * 2) * 8 // 3)


def test_faces_of_a_stage_by_tiles():
    p = params((16, 17, 18), (P, R, P))
    faces, _ = bench.face_counts(p)
    assert work("march_zeta", p, TILES)[1] == sum(faces) * bench.FLOPS_PER_FACE
    assert work("march_zeta", p)[1] == (faces[0] + faces[2]) * bench.FLOPS_PER_FACE


def test_rate_uses_the_launches_work():
    p = params((64,) * 3)
    run = bench.as_run(p, TILES)
    r = bench.roofline_of("march_zeta", 3.0, 3, p, "tgv", run)
    assert r["achieved"] == pytest.approx(sum(bench.face_counts(p)[0]) * 1580 / 1e-3 / 1e12)
