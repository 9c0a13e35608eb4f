"""The pooled levels' partial sums past the caches (grids with many of them) against the oracle.  Stored so beyond 80 MiB: 16 heads of 16384
tokens with 20 key blocks a group are just on that line, 17 just beyond; an even share of key blocks a wave, and the fewest.  Read so beyond
64 MiB: 12 heads are below that line, 13 beyond; without lists, 48 heads of 16384 tokens (96 MiB of fp32 sums)."""
import pytest
import torch

import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,T2", [(12, 16), (13, 16), (16, 16), (17, 16), (15, 20), (21, 12)])
def test_grids(H, T2):
    P.check_op_l2(torch.device("cuda"), B=1, H=H, N=16384, T=8, T2=T2, fused=True, rope=True, smooth=True)


def test_one_level():
    P.check_op_l1(torch.device("cuda"), B=8, H=6, N=16384, T=4, fused=True, rope=True)
