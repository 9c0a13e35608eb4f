"""The query-side kernels around 512 groups of eight query blocks, the size of half a round of the chip, at the edges of the topk
ranges that the list registers have: one register of entries per lane up to 32 entries a row, two up to 64."""
import pytest
import torch

import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [4, 32, 36, 48, 64])
def test_topk_ranges(T):
    P.check_op_l1(torch.device("cuda"), B=4, H=4, N=4096, T=T, fused=True, rope=T == 36, smooth=T != 48)


def test_two_levels_largest_topk():
    P.check_op_l2(torch.device("cuda"), B=2, H=2, N=16384, T=64, T2=32, fused=True, rope=True, smooth=True)


@pytest.mark.parametrize("H", [63, 64])
def test_around_the_smallest_grid(H):
    P.check_op_l1(torch.device("cuda"), B=1, H=H, N=1024, T=8, fused=True, rope=True)
