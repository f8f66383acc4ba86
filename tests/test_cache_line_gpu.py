"""Query blocks of more than 128 on an INT8 cache that take the short-query kernel because its few launches win there: ragged last
blocks of 16, the last length that may take it and the first that may not, against fp64."""
import pytest
import torch

from test_cache_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,H,Nq,Nk,D", [(1, 4, 129, 1000, 64), (1, 3, 200, 777, 128), (2, 1, 257, 600, 256), (1, 40, 144, 300, 128),
                                         (1, 2, 512, 513, 64), (1, 2, 513, 514, 64)])
def test_long_blocks_on_the_short_kernel(qfa, B, H, Nq, Nk, D, causal):
    _check(qfa, B, H, Nq, Nk, D, causal, torch.float16, torch.float16, seed=Nq)
