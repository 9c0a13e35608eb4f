"""The one-launch index transpose at the edges of its ranges: key blocks that do not divide into equal ranges, entries read
one and four at a time, the largest list it takes and the smallest it leaves to the kernels for large jobs."""
import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests

SMALL = [(1, 2, 33, 1, 33, 4), (2, 1, 50, 5, 97, 2), (1, 1, 64, 4, 2100, 3)]


@pytest.mark.parametrize("B,H,Mb,T,Kb,chunk", SMALL)
def test_cpu(B, H, Mb, T, Kb, chunk):
    with override_library_for_tests(emu_lib()):
        P.check_transpose(torch.device("cpu"), B=B, H=H, Mb=Mb, T=T, Kb=Kb, chunk=chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Mb,T,Kb,chunk", SMALL + [(1, 3, 4096, 16, 4096, 256), (1, 3, 4112, 16, 4112, 256), (4, 16, 1024, 64, 1024, 64),
                                                       (1, 1, 65536, 1, 500, 64)])
def test_gpu(B, H, Mb, T, Kb, chunk):
    P.check_transpose(torch.device("cuda"), B=B, H=H, Mb=Mb, T=T, Kb=Kb, chunk=chunk)
