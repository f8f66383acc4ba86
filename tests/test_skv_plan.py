"""Which shared-KV kernel the plan takes where the workgroups of whole heads do not fill the XCDs evenly, or where a workgroup has
few tiles: launches measured with every kernel (us on an MI355X; 16 queries per workgroup, two and four waves side by side on
tiles).  The choice may not cost more than a twentieth over the 16-query kernel."""
import math
import random

import pytest

from plans import skv_tile_dq_plan, skv_tile_fwd_plan
from quant_flash_attn_amd import _lib

FORWARD = [
    # heads, Nq, Nk, D, {kernel: us}
    (81, 173, 513, 256, {0: 32.0, 2: 45.9, 4: 31.2}),    # 33 workgroups on one XCD of 32 CUs with two waves
    (85, 155, 2474, 256, {0: 91.1, 2: 135.7}),
    (1820, 34, 345, 256, {0: 109.2, 2: 139.2}),
    (1207, 137, 612, 256, {0: 318.4, 2: 353.5, 4: 333.3}),
    (430, 42, 1109, 256, {0: 70.1, 2: 77.0}),
    (18, 465, 132, 128, {0: 8.2, 2: 9.8, 4: 10.1}),
    (555, 48, 380, 128, {0: 21.7, 2: 24.7}),
    (1552, 32, 80, 128, {0: 23.6, 2: 27.5}),
    (57, 188, 178, 128, {0: 9.1, 2: 10.2, 4: 10.0}),
    (265, 47, 96, 64, {0: 6.0, 2: 7.7}),
    (158, 65, 257, 64, {0: 8.7, 2: 11.2, 4: 9.7}),
    (330, 35, 134, 64, {0: 7.0, 2: 8.9}),
    (88, 150, 708, 64, {0: 13.2, 2: 16.2, 4: 16.3}),
    (317, 39, 685, 64, {0: 13.1, 2: 16.0}),
    (161, 85, 1550, 64, {0: 25.1, 2: 30.0, 4: 28.9}),
]
DQ = [(84, 347, 546, 256, {0: 175.0, 4: 195.6})]   # (the whole backward)


@pytest.mark.parametrize("plan,BH,Nq,Nk,D,us", [(skv_tile_fwd_plan, *c) for c in FORWARD] + [(skv_tile_dq_plan, *c) for c in DQ])
def test_choice_is_not_slower(qfa, plan, BH, Nq, Nk, D, us):
    p = plan(BH, Nq, Nk, D)
    assert p.splits == 1 and us.get(p.waves, float("inf")) <= 1.05 * us[0], (p.waves, p.splits)


def test_more_than_16_queries_fit_the_built_in_scratch(qfa):
    """qfa_attn_fwd_shared_kv_static accepts every block of more than 16 queries, whichever kernel the plan takes."""
    L, rng = _lib.lib(), random.Random(4)
    log = lambda lo, hi: int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    shapes = [(5, 537, 40160, 256), (83, 50, 10756, 256), (8, 144, 15338, 256)]   # (16 and 18 MB for the 16-query kernel's splits)
    shapes += [(log(1, 1500), log(17, 1100), log(30, 60000), rng.choice((64, 128, 256))) for _ in range(40000)]
    for BH, Nq, Nk, D in shapes:
        assert 0 <= L.qfa_attn_fwd_shared_kv_workspace_bytes(1, BH, Nq, Nk, D) <= 16 << 20, (BH, Nq, Nk, D)


@pytest.mark.parametrize("BH,Nq", [(1, 1 << 40), (5, 537), (1, 17), (1, 16)])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_sizes_beyond_any_memory_are_answered(qfa, BH, Nq, D):
    """The size of a scratch can be asked for with any sizes: 2^40 keys are 2^35 tiles, a number that is 0 in 32 bits."""
    assert 0 <= _lib.lib().qfa_attn_fwd_shared_kv_workspace_bytes(1, BH, Nq, 1 << 40, D)
