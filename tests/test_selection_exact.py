"""Block selection on small-integer inputs: every score is exact in bf16 and most rows have ties at the threshold, so the
selected blocks and their order (score descending, index ascending) are known exactly.  Sizes at the edges of the
selection kernels' forms: keys in registers up to 1024 per row, streamed beyond; rows that do not fill a wave's tiles; top-k
from 1 to the row's length."""
import pytest
import torch

from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests
from oracle import llsa_oracle as O


def ints(seed, *shape, hi=2):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-(hi - 1), hi, shape, generator=g).bfloat16()


def check_dense(dev, n, T, BH, round_scores, hi=2):
    from llsa_amd.kernel.hip.topk import gen_sparse_indices
    pq, pk = ints(n + T, 1, BH, n, 64, hi=hi), ints(n + T + 1, 1, BH, n, 64, hi=hi)
    got = gen_sparse_indices(pq.to(dev), pk.to(dev), T, round_scores=round_scores).cpu().long()
    ref = O.topk_lowest_index(torch.matmul(pq.float(), pk.float().transpose(-1, -2)), T)
    assert torch.equal(got, ref)


def check_sparse(dev, N1, T, T2, BH, hi=2):
    from llsa_amd.kernel.hip.topk import compute_topk_indices_sparse, gen_sparse_indices, topk_cascade
    pq, pk = ints(N1 + T, 1, BH, N1, 64, hi=hi), ints(N1 + T + 1, 1, BH, N1, 64, hi=hi)
    N2 = N1 // 16
    g = torch.Generator().manual_seed(T2)
    pidx = torch.stack([torch.randperm(N2, generator=g)[:T2] for _ in range(BH * N2)]).reshape(1, BH, N2, T2)
    got = compute_topk_indices_sparse(pq.to(dev), pk.to(dev), pidx.int().to(dev), T, T2).cpu().long()
    score = torch.matmul(pq.float(), pk.float().transpose(-1, -2))
    own = torch.zeros(1, BH, N2, N2).scatter_(-1, pidx, 1.0).repeat_interleave(16, 2).repeat_interleave(16, 3)
    ref = O.topk_lowest_index(torch.where(own > 0, score, torch.full_like(score, -1e30)), T)
    assert torch.equal(got, ref)
    pq2, pk2 = ints(N1 + 7, 1, BH, N2, 64, hi=hi), ints(N1 + 8, 1, BH, N2, 64, hi=hi)
    if N2 <= 256:
        p_got, c_got = topk_cascade(pq2.to(dev), pk2.to(dev), pq.to(dev), pk.to(dev), T, T2)
        p_ref = gen_sparse_indices(pq2.to(dev), pk2.to(dev), T2)
        assert torch.equal(p_got, p_ref)
        assert torch.equal(c_got, compute_topk_indices_sparse(pq.to(dev), pk.to(dev), p_ref, T, T2))


DENSE = [(16, 1, 2), (16, 16, 1), (48, 3, 1), (64, 64, 1), (80, 16, 2), (256, 64, 1), (320, 12, 1), (1024, 16, 1), (1040, 8, 1), (1088, 64, 1)]
SPARSE = [(256, 1, 1, 1), (256, 20, 4, 1), (512, 16, 5, 1), (512, 64, 16, 1), (768, 8, 17, 1), (512, 64, 32, 1)]


@pytest.mark.parametrize("n,T,BH", DENSE)
@pytest.mark.parametrize("round_scores", [True, False])
def test_dense_cpu(n, T, BH, round_scores):
    with override_library_for_tests(emu_lib()):
        check_dense(torch.device("cpu"), n, T, BH, round_scores)


@pytest.mark.parametrize("N1,T,T2,BH", SPARSE)
def test_sparse_cpu(N1, T, T2, BH):
    with override_library_for_tests(emu_lib()):
        check_sparse(torch.device("cpu"), N1, T, T2, BH)


def test_equal_scores_everywhere_cpu():
    with override_library_for_tests(emu_lib()):
        check_dense(torch.device("cpu"), 1088, 16, 1, True, hi=1)        # all zero: indices 0 .. T-1
        check_sparse(torch.device("cpu"), 256, 8, 4, 1, hi=1)


@pytest.mark.gpu
@pytest.mark.parametrize("n,T,BH", DENSE + [(2112, 20, 3), (4096, 8, 8), (4096, 64, 8), (2048, 16, 20)])
@pytest.mark.parametrize("round_scores", [True, False])
def test_dense_gpu(n, T, BH, round_scores):
    check_dense(torch.device("cuda"), n, T, BH, round_scores)
    check_dense(torch.device("cuda"), n, T, BH, round_scores, hi=1)


@pytest.mark.gpu
@pytest.mark.parametrize("N1,T,T2,BH", SPARSE + [(1024, 16, 16, 12), (4096, 32, 24, 2)])
def test_sparse_gpu(N1, T, T2, BH):
    check_sparse(torch.device("cuda"), N1, T, T2, BH)
    check_sparse(torch.device("cuda"), N1, T, T2, BH, hi=1)
