"""A wave takes two sibling query blocks where such waves fill the chip's rounds (768 groups of eight query blocks each) or pooled
blocks are most of the walk, one block elsewhere: both sides of every line of that rule, and the two-block kernels at the edges of
their topk ranges."""
import ctypes as C

import pytest
import torch

import parity_cases as P
from llsa_amd._lib import get_lib


def _blocks(B, H, N, *topk):
    ask = lambda backward: get_lib().query_blocks_per_wave(B, H, N, (C.c_int32 * len(topk))(*topk), len(topk), backward)
    return ask(0), ask(1)


@pytest.mark.parametrize("B,H,N,topk,blocks", [
    # rounds, few pooled blocks: the forward from 513 groups on, dQ from 641, neither where 31 % of the places or more stay empty
    (1, 16, 4096, (4,), (1, 1)), (1, 17, 4096, (4,), (2, 1)), (1, 9, 8192, (8,), (2, 1)), (1, 20, 4096, (4,), (2, 1)), (1, 21, 4096, (4,), (2, 2)),
    (1, 24, 4096, (4,), (2, 2)), (1, 25, 4096, (4,), (1, 1)), (1, 36, 4096, (4,), (1, 1)), (1, 37, 4096, (4,), (2, 2)),
    # most of the walk in the fine blocks: the forward only on grids of several rounds
    (2, 6, 16384, (16, 16), (1, 2)), (1, 16, 16384, (64, 4), (2, 2)),
    # most of the walk in pooled blocks: from 512 groups on (a large topk: from a full round on), up to 60 % more places than groups
    (1, 1, 65536, (8,), (2, 2)), (1, 1, 65536, (16,), (2, 2)), (1, 2, 65536, (8,), (2, 2)), (1, 2, 32768, (8,), (2, 2)), (1, 2, 32768, (16,), (2, 2)),
    (1, 3, 24576, (8,), (2, 2)), (1, 5, 24576, (8,), (2, 2)), (1, 1, 57344, (8,), (1, 1)), (1, 5, 20480, (8,), (1, 1)), (1, 4, 28672, (8,), (1, 1)),
    (1, 4, 16384, (8,), (2, 2)), (1, 7, 16384, (8,), (1, 1)), (1, 8, 16384, (8,), (2, 2)), (1, 13, 16384, (16,), (2, 2)), (1, 4, 32768, (32,), (2, 2)),
    (1, 1, 65536, (64,), (1, 1)), (1, 2, 65536, (64,), (2, 2)), (1, 2, 32768, (20,), (1, 1)), (1, 8, 16384, (20,), (1, 1)), (1, 1, 262144, (8, 16), (2, 2)),
    # the lists of more than 64 entries have no two-block kernel
    (8, 8, 16384, (68, 16), (1, 1)),
])
def test_rule(B, H, N, topk, blocks):
    assert _blocks(B, H, N, *topk) == blocks


@pytest.mark.gpu
@pytest.mark.parametrize("H", [16, 17, 20, 21, 24, 25, 36, 37])   # 32 H groups; dQ with two blocks: 21, 24 and 37 heads, the forward from 17 to 24 and 37
def test_lines_of_the_rule(H):
    P.check_op_l1(torch.device("cuda"), B=1, H=H, N=4096, T=4, fused=True, rope=True)   # (16 shared blocks, topk 4)


@pytest.mark.gpu
@pytest.mark.parametrize("H,N,T", [(9, 8192, 8), (2, 32768, 8), (3, 24576, 8), (5, 20480, 8), (8, 16384, 16)])      # 576, 512, 576, 800, 1024 groups
def test_pooled_walk(H, N, T):
    P.check_op_l1(torch.device("cuda"), B=1, H=H, N=N, T=T, fused=True)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [4, 32, 36, 64])
def test_topk_ranges(T):
    """dQ with two blocks (768 groups); the forward, with 16 shared blocks, only at topk 4."""
    P.check_op_l1(torch.device("cuda"), B=4, H=6, N=4096, T=T, fused=True, rope=T == 36, smooth=T != 64)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [32, 36, 64])
def test_topk_ranges_of_the_forward(T):
    """Both kernels with two blocks: 2048 groups."""
    assert _blocks(1, 16, 16384, T, 4) == (2, 2)
    P.check_op_l2(torch.device("cuda"), B=1, H=16, N=16384, T=T, T2=4, fused=True, rope=T == 36, smooth=T != 64, slices=[(0, 0), (0, 15)])


@pytest.mark.gpu
def test_two_levels_largest_topk():
    P.check_op_l2(torch.device("cuda"), B=2, H=3, N=16384, T=64, T2=32, fused=True, rope=True, smooth=True)
