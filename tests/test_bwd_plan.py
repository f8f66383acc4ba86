"""Divisions of the backward that took longer than the undivided kernels (us on an MI355X, whole backward): the plan may not choose
them."""
import math
import random

import pytest

from plans import bwd_plan, bwd_plan_within

SLOWER = [
    # heads, Nq, Nk, D, causal, (rows per wave / 32, parts) of dK / dV and of dQ, us undivided, us so divided
    # chosen while a launch's workgroups were counted as if they were dealt evenly to the XCDs
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
    # chosen by an estimate that was fitted to undivided launches of more than 1100 workgroups, and in which parts cost nothing
    (96, 691, 691, 128, True, (2, 1), (2, 2), 94.9, 117.7),
    (107, 227, 1168, 128, True, (2, 1), (2, 3), 97.0, 118.5),
    (74, 942, 942, 128, True, (2, 1), (2, 2), 116.2, 137.6),
    (159, 216, 1186, 128, False, (2, 1), (2, 2), 140.0, 162.0),
    (71, 1014, 1014, 128, False, (2, 1), (2, 2), 160.5, 183.7),
    (75, 975, 975, 128, False, (2, 1), (2, 2), 165.0, 187.3),
    (106, 199, 1034, 128, True, (2, 1), (2, 3), 94.8, 106.9),
    (58, 508, 2568, 128, False, (2, 1), (2, 4), 171.4, 190.9),
    (78, 158, 2145, 128, False, (2, 1), (2, 5), 117.9, 126.2),
    (27, 1513, 5602, 128, False, (2, 1), (2, 3), 365.1, 385.7),
]

FULL = [s[:5] for s in SLOWER[10:]] + [(188, 127, 1876, 128, False), (103, 231, 3686, 128, True), (170, 1056, 1056, 128, False)]


@pytest.mark.parametrize("BH,Nq,Nk,D,causal,dkv,dq,undivided,divided", SLOWER)
def test_slower_division_is_not_chosen(qfa, BH, Nq, Nk, D, causal, dkv, dq, undivided, divided):
    p = bwd_plan(BH, Nq, Nk, D, causal)
    assert ((p.blocks_dkv, p.splits_dkv), (p.blocks_dq, p.splits_dq)) != (dkv, dq), divided / undivided


@pytest.mark.parametrize("BH,Nq,Nk,D,causal", FULL)
def test_a_full_chip_is_not_divided(qfa, BH, Nq, Nk, D, causal):
    """More than 1100 workgroups, of which neither kind by itself is worth dividing."""
    assert BH * ((Nq + 127) // 128 + (Nk + 127) // 128) > 1100
    p = bwd_plan(BH, Nq, Nk, D, causal)
    assert (p.splits_dkv, p.splits_dq, p.part_bytes) == (1, 1, 0)


OTHER_ROWS = [
    # heads, Nq, Nk, causal, rows per wave / 32 of dK / dV and of dQ, us with each kind's own choice, us with this one (in one launch both)
    (53, 415, 2158, False, (2, 2), 125.4, 146.7),
    (118, 355, 3301, True, (2, 1), 343.1, 393.8),
    (119, 378, 4799, True, (2, 1), 486.6, 553.8),
    (87, 380, 5964, False, (2, 1), 474.2, 539.5),
    (94, 345, 3632, False, (2, 1), 328.2, 372.5),
    (102, 145, 1237, False, (2, 2), 88.6, 100.2),
    (126, 364, 5066, False, (2, 1), 541.2, 610.3),
    (22, 1173, 5651, False, (2, 2), 275.0, 307.1),
]


@pytest.mark.parametrize("BH,Nq,Nk,causal,rows,own,joint", OTHER_ROWS)
def test_slower_rows_per_wave_are_not_chosen(qfa, BH, Nq, Nk, causal, rows, own, joint):
    """Many workgroups whose estimate was fitted to sequences of about the same length."""
    p = bwd_plan(BH, Nq, Nk, 128, causal)
    assert (p.blocks_dkv, p.blocks_dq) != rows, joint / own


LONG_CHAINS = [
    # heads, Nq, Nk, causal, us undivided with 32 rows per wave, us with 64 of dK / dV
    (7, 4143, 4143, False, 199.7, 232.5),
    (7, 4192, 4192, False, 203.5, 236.1),
    (7, 4159, 4188, False, 203.7, 233.6),
    (7, 4324, 4324, False, 210.9, 250.5),
    (7, 4288, 4288, True, 161.5, 175.6),
    (7, 4546, 4546, True, 176.2, 187.9),
    (6, 4909, 4909, True, 180.5, 198.6),
]


@pytest.mark.parametrize("BH,Nq,Nk,causal,short,long", LONG_CHAINS)
def test_dkv_stays_at_32_rows_where_it_runs_all_at_once(qfa, BH, Nq, Nk, causal, short, long):
    """Half as many workgroups of twice the length, beside as many of dQ as before."""
    p = bwd_plan(BH, Nq, Nk, 128, causal)
    assert ((p.blocks_dkv, p.splits_dkv), (p.blocks_dq, p.splits_dq)) != ((2, 1), (1, 1)), long / short


def _fields(p):
    return tuple(getattr(p, n) for n, _ in p._fields_)


def test_what_is_planned_is_launched(qfa):
    """With the memory that the size query asks for the launch gets the plan that the query made, also where that is none for parts
    but rows per wave; with less it is undivided, with more the same."""
    rng, undivided = random.Random(5), 0
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    shapes = [(170, 1056, 1056, 128, False), (7, 1542, 4268, 128, False), (15, 782, 2179, 128, True), (6, 5995, 5995, 128, True)]
    for _ in range(5000):
        Nk = log(16, 8192)
        shapes.append((log(1, 800), Nk if rng.random() < 0.6 else log(1, Nk), Nk, rng.choice((64, 128, 128, 256)), rng.random() < 0.5))
    for s in shapes:
        p = bwd_plan(*s)
        assert _fields(bwd_plan_within(*s, p.part_bytes)) == _fields(bwd_plan_within(*s, p.part_bytes + 999)) == _fields(p), s
        if p.part_bytes > 0:
            less = bwd_plan_within(*s, p.part_bytes - 1)
            assert (less.splits_dkv, less.splits_dq, less.part_bytes) == (1, 1, 0), s
        else:
            alone = bwd_plan(*s, may_split=0)   # (each kind's rows per wave as if it had the chip to itself)
            undivided += (p.blocks_dkv, p.blocks_dq) != (alone.blocks_dkv, alone.blocks_dq)
    assert undivided > 20


def test_more_than_one_launch_holds(qfa):
    """2^32 - 1 threads: of so many heads dK / dV and dQ go out one after the other, as long as the staging launch (two tiles a head) fits."""
    for BH, two in ((8388600, 0), (8388601, 1), (8388607, 1)):
        assert 2 * BH * 256 < 2 ** 32
        p = bwd_plan(BH, 1, 1, 64, False)
        assert (p.sum_between, p.part_bytes, p.splits_dkv, p.splits_dq) == (two, 0, 1, 1)
        assert two or 2 * ((BH + 7) // 8 * 8) * 256 < 2 ** 32
