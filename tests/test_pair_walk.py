"""The query-side kernels with one query block a wave, at and just below 512 groups of eight query blocks, where their workgroups fill
the chip once: topk up to the 64 entries that a wave's list register holds."""
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
