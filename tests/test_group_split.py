"""The group-major pass where the groups of its last round are dealt out to several workgroups, against the oracle.  An XCD has 8 groups per head of
16384 tokens and takes 64 at a time: 1, 4 and 7 heads are one round that is an eighth, half and seven eighths full, 8 fill it, 9, 10 and 12 leave a
second one nearly empty to half full; few key blocks a group (T2 + 4) are dealt out to fewer workgroups or none, many to more waves than
have a share."""
import pytest
import torch

import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,T2", [(1, 4), (1, 8), (1, 16), (1, 32), (4, 16), (7, 16), (8, 16), (9, 4), (9, 8), (9, 20), (9, 32), (10, 16), (12, 24)])
def test_grids(H, T2):
    P.check_op_l2(torch.device("cuda"), B=1, H=H, N=16384, T=8, T2=T2, fused=True, rope=True, smooth=True)
