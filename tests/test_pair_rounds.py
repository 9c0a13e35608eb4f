"""A wave takes two sibling query blocks where such waves fill the chip's rounds (768 groups of eight query blocks each), one block
elsewhere: both sides of every line of that rule, and the two-block kernels at the edges of their topk ranges."""
import pytest
import torch

import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [20, 21, 24, 25, 36, 37])   # 32 H groups; two blocks: 21, 24 and 37 heads
def test_lines_of_the_rule(H):
    P.check_op_l1(torch.device("cuda"), B=1, H=H, N=4096, T=4, fused=True, rope=True)   # (16 shared blocks, topk 4: forward as well)


@pytest.mark.parametrize("T", [4, 32, 36, 64])
def test_topk_ranges(T):
    P.check_op_l1(torch.device("cuda"), B=4, H=6, N=4096, T=T, fused=True, rope=T == 36, smooth=T != 64)


def test_two_levels_largest_topk():
    P.check_op_l2(torch.device("cuda"), B=2, H=3, N=16384, T=64, T2=32, fused=True, rope=True, smooth=True)
