"""The list form of the dense K-side kernel (level 2 of llsa_l3 on grids that fill the chip) against the oracle: lists of one and of two
workgroups, an owner's range in two pieces and whole; and the largest grid that keeps the group-major pass.  (Lists of level 3, with their
owner's range in sixteen pieces: the four-level case of test_gpu_fullsize.)"""
import pytest
import torch

import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,T3", [(5, 16), (6, 16), (3, 32)])
def test_grids(H, T3):
    P.check_op_l3(torch.device("cuda"), H=H, T=8, T2=4, T3=T3)


def test_whole_ranges():
    P.check_op_l3(torch.device("cuda"), H=12, T=8, T2=4, T3=16, heads=[0, 11])
