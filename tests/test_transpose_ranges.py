"""The one-launch index transpose at the edges of its ranges: key blocks that do not divide into equal ranges, entries read
one and four at a time, the largest list it takes and the smallest it leaves to the kernels for large jobs."""
import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from gpu_time import median_us
from llsa_amd._lib import override_library_for_tests
from llsa_amd.kernel.hip.indices_transpose import transpose_indices

SMALL = [(1, 2, 33, 1, 33, 4), (2, 1, 50, 5, 97, 2), (1, 1, 64, 4, 2100, 3), (1, 1, 12000, 1, 70, 64)]    # (the last: a sum for every fourth word)


@pytest.mark.parametrize("B,H,Mb,T,Kb,chunk", SMALL)
def test_cpu(B, H, Mb, T, Kb, chunk):
    with override_library_for_tests(emu_lib()):
        P.check_transpose(torch.device("cpu"), B=B, H=H, Mb=Mb, T=T, Kb=Kb, chunk=chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Mb,T,Kb,chunk", SMALL + [(1, 3, 4096, 16, 4096, 256), (1, 3, 4112, 16, 4112, 256), (4, 16, 1024, 64, 1024, 64),
                                                       (1, 1, 65536, 1, 500, 64), (1, 6, 8192, 8, 8192, 64), (1, 48, 1024, 16, 1024, 64)])
def test_gpu(B, H, Mb, T, Kb, chunk):
    P.check_transpose(torch.device("cuda"), B=B, H=H, Mb=Mb, T=T, Kb=Kb, chunk=chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("BH,Mb,T", [(6, 8192, 8), (1, 16384, 4), (12, 4096, 8)])
def test_inverse_costs_no_second_set_of_ranges(BH, Mb, T):
    """Lists with their inverse positions take 1.5 to 1.7 times the time of the lists alone.  (With sums that double a key block's LDS, and so the ranges that
    each read all entries, 2.9 to 3.5 times.)"""
    near = torch.rand(Mb, 512, generator=torch.Generator().manual_seed(Mb)).topk(T, -1).indices       # (of key blocks near by, as a selection's are)
    idx = ((torch.arange(Mb)[:, None] // 256 * 256 + near) % Mb).int().expand(1, BH, Mb, T).contiguous().cuda()
    times = [median_us(lambda: transpose_indices(idx, inverse=inverse)) for inverse in (True, False)]
    print(f"{times[0] / times[1]:.2f}")
    assert times[0] < 2.4 * times[1]
