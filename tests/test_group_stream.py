"""The pooled levels' partial sums past the caches (grids with many of them) against the oracle: 80 MiB of partial sums is where the line lies, 16
heads of 16384 tokens with 20 key blocks a group are just on it, 17 just beyond; an even share of key blocks a wave, and the fewest."""
import pytest
import torch

import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,T2", [(16, 16), (17, 16), (15, 20), (21, 12)])
def test_grids(H, T2):
    P.check_op_l2(torch.device("cuda"), B=1, H=H, N=16384, T=8, T2=T2, fused=True, rope=True, smooth=True)
