"""Dense selection over rows longer than 1024 keys: the forms of the kernel (rows per workgroup, groups per row, key width) at the
edges of their ranges, and rows whose bound lets more keys through than their buffer holds.  Scores are small integers, exact in
bf16, so the result is known exactly: score descending, index ascending, NaN below every number."""
import pytest
import torch

from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests


def expected(pq, pk, T):
    s = torch.matmul(pq.float(), pk.float().transpose(-1, -2))
    s = torch.where(s.isnan(), torch.full_like(s, -1e30), s)
    return torch.sort(s, dim=-1, descending=True, stable=True).indices[..., :T]


def ints(seed, *shape, hi=2):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-(hi - 1), hi, shape, generator=g).bfloat16()


def check(dev, n, T, BH, kind, round_scores=True):
    from llsa_amd.kernel.hip.topk import gen_sparse_indices
    pq, pk = ints(n + T, 1, BH, n, 64), ints(n + T + 1, 1, BH, n, 64)
    if kind == "few groups":            # the best keys at T - 1 of the positions modulo 64
        at = torch.arange(n) % 64 < T - 1
        pk[:, :, at] = ints(n, 1, BH, int(at.sum()), 64, hi=4)
    elif kind == "equal":
        pk[:] = pk[:, :, :1]
    elif kind == "nan":                 # rows without a number, keys without a number, a row of infinities
        pq[:, :, 5, 3] = float("nan")
        pk[:, :, 1::3, 7] = float("nan")
        pk[:, :, 40, :] = 0
        pk[:, :, 40, 0] = float("inf")
        pq[:, :, :, 0] = 1
    got = gen_sparse_indices(pq.to(dev), pk.to(dev), T, round_scores=round_scores).cpu().long()
    assert torch.equal(got, expected(pq, pk, T))


@pytest.mark.parametrize("n,T,kind", [(1040, 1, "plain"), (1088, 16, "few groups"), (1040, 17, "nan"), (1056, 64, "equal")])
def test_cpu(n, T, kind):
    with override_library_for_tests(emu_lib()):
        check(torch.device("cpu"), n, T, 1, kind)


# 16 rows a workgroup: at most 256 sixteens of rows, or an odd number of them; 32: at most 512, n no multiple of 64, or T > 32; 64 beyond
@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "few groups", "equal", "nan"])
@pytest.mark.parametrize("n,T,BH", [(1040, 16, 8), (2048, 32, 2), (4096, 16, 1), (1056, 16, 8), (1056, 33, 9), (2064, 8, 1), (1088, 17, 4), (1088, 16, 8),
                                    (1088, 17, 8), (3072, 32, 3), (1088, 64, 8), (4096, 64, 2)])
def test_gpu(n, T, BH, kind):
    check(torch.device("cuda"), n, T, BH, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "few groups", "equal", "nan"])
@pytest.mark.parametrize("n,T,BH", [(1040, 64, 3), (4096, 8, 2), (1088, 64, 8), (1088, 32, 8)])
def test_unrounded_gpu(n, T, BH, kind):
    check(torch.device("cuda"), n, T, BH, kind, round_scores=False)
