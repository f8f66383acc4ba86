"""Divisions of the backward that were chosen while a launch's workgroups were counted as if they were dealt evenly to the XCDs, and
that took longer than the undivided kernels (us on an MI355X, whole backward): the plan may not choose them."""
import pytest

from plans import bwd_plan

SLOWER = [
    # heads, Nq, Nk, D, causal, (rows per wave / 32, parts) of dK / dV and of dQ, us undivided, us so divided
    (5, 4270, 4270, 128, False, (2, 3), (2, 3), 219.3, 259.7),      # 33 workgroups on one XCD of 32 CUs
    (7, 4502, 4502, 128, True, (2, 3), (1, 1), 207.5, 242.6),
    (5, 4555, 4555, 128, True, (2, 4), (2, 4), 200.5, 230.5),
    (2, 15368, 15368, 128, True, (2, 3), (2, 3), 635.8, 726.9),
    (8, 3727, 3727, 128, True, (2, 3), (1, 1), 173.2, 197.6),
    (12, 4037, 4037, 128, True, (2, 2), (1, 1), 216.0, 240.2),
    (2, 16351, 16351, 256, True, (1, 4), (1, 4), 1223.8, 1483.8),
    (2, 15938, 15938, 256, True, (1, 4), (1, 4), 1185.5, 1433.7),
    (10, 3567, 3567, 256, True, (1, 1), (1, 3), 296.9, 337.1),
    (9, 3345, 3345, 64, True, (1, 3), (1, 3), 115.4, 122.8),
]


@pytest.mark.parametrize("BH,Nq,Nk,D,causal,dkv,dq,undivided,divided", SLOWER)
def test_slower_division_is_not_chosen(qfa, BH, Nq, Nk, D, causal, dkv, dq, undivided, divided):
    p = bwd_plan(BH, Nq, Nk, D, causal)
    assert ((p.blocks_dkv, p.splits_dkv), (p.blocks_dq, p.splits_dq)) != (dkv, dq), divided / undivided
