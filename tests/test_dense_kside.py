"""The K side of the dense coarsest level against the oracle where its forms begin and end: groups of 4, 8 and 16 units (a unit is 16
coarsest tokens), the last group full, with idle waves, and almost empty; and the query range cut for one, two and three rounds of the chip."""
import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests
from oracle import llsa_oracle as O


def _run(dev, B, H, N, T=4):
    from llsa_amd.kernel.hip._attention import attn_bwd, attn_fwd
    q, k, v, do = P.randn_inputs(B, H, N, 64, dev, seed=N + H)
    c = [t.cpu() for t in (q, k, v, do)]
    pk, pv = O.mean_pool(c[1]), O.mean_pool(c[2])
    idx = P._hot_indices(B, H, N // 16, N // 16, T, 3, 5)
    args = (pk.to(dev), pv.to(dev), idx.int().to(dev), 16.0)
    o, lse = attn_fwd(q, k, v, *args)
    ref = O.attn_bwd_l1(c[3], c[0], c[1], c[2], pk, pv, o.cpu(), lse.cpu(), idx, 16.0)
    got = attn_bwd(do, q, k, v, *args[:2], o, lse, *args[2:], 1.0)
    for name, a, b in zip(("dq", "dk", "dv", "dpk", "dpv"), got, ref):
        P.close(f"{name} at {N // 256} units", a, b)


@pytest.mark.parametrize("N", [4096, 5120])
def test_dense_cpu(N):
    with override_library_for_tests(emu_lib()):
        _run(torch.device("cpu"), 1, 1, N)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N", [(1, 1, 1024), (1, 2, 3072), (1, 1, 4096), (2, 3, 4096), (1, 2, 5120), (1, 3, 6144), (2, 2, 7168), (1, 2, 9216), (1, 1, 17408),
                                   (1, 8, 32768), (4, 6, 16384), (2, 24, 16384)])          # 4, 5 and 4 long pieces
def test_dense_gpu(B, H, N):
    _run(torch.device("cuda"), B, H, N)
