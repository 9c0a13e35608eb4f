"""The piece length of the fine K-side pass: by the entries of all heads at the short sequences, by the token count beyond; and lists
cut into other pieces give the same gradients."""
import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import LlsaError, override_library_for_tests
from oracle import llsa_oracle as O


@pytest.mark.parametrize("B,H,N,T,chunk", [(1, 1, 1024, 4, 16), (1, 6, 1024, 8, 16), (4, 8, 1024, 8, 16), (4, 8, 1024, 12, 32), (4, 16, 1024, 16, 32),
                                           (4, 16, 1024, 20, 64), (16, 6, 1024, 64, 64), (128, 6, 1024, 64, 64), (1, 1, 2048, 64, 16),
                                           (1, 8, 2048, 64, 32), (1, 9, 2048, 64, 64), (1, 1, 3072, 4, 64), (1, 1, 16384, 4, 64),
                                           (1, 1, 17408, 4, 256), (8, 12, 262144, 16, 256)])
def test_rule(B, H, N, T, chunk):
    import ctypes as C
    lib = emu_lib()
    assert lib.fine_chunk_for(B, H, N, T) == chunk and chunk <= lib.fine_chunk(N)
    # the workspace of many heads does not grow with the cut: 8 KB for each of at most 2 E / chunk + 2 pieces a head
    if N == 1024:
        need = lib.attn_bwd_workspace_bytes(B, H, N, (C.c_int32 * 1)(T), 1)
        assert need <= B * H * (2 * (64 * T // chunk) + 2) * 8192 + B * H * (64 * 128 + 1024 * 128 + 4 * 4 * 8192) + 1024


def _run(dev, B, H, N, T, chunks):
    from llsa_amd.kernel.hip._attention import attn_bwd, attn_fwd
    from llsa_amd.kernel.hip.indices_transpose import transpose_indices
    q, k, v, do = P.randn_inputs(B, H, N, 64, dev, seed=51)
    c = [t.cpu() for t in (q, k, v, do)]
    pk, pv = O.mean_pool(c[1]), O.mean_pool(c[2])
    idx = P._hot_indices(B, H, N // 16, N // 16, T, 3, 7)     # key block 3 is in every list: cut at every chunk
    args = (pk.to(dev), pv.to(dev))
    o, lse = attn_fwd(q, k, v, *args, idx.int().to(dev), 16.0)
    ref = O.attn_bwd_l1(c[3], c[0], c[1], c[2], pk, pv, o.cpu(), lse.cpu(), idx, 16.0)
    for chunk in chunks:
        csr = transpose_indices(idx.int().to(dev), N // 16, chunk or 64)
        got = attn_bwd(do, q, k, v, *args, o, lse, idx.int().to(dev), 16.0, 1.0, csr=csr, chunk=chunk)
        for name, a, b in zip(("dq", "dk", "dv", "dpk", "dpv"), got, ref):
            P.close(f"{name} in pieces of {chunk}", a, b)
    with pytest.raises(LlsaError, match="chunk=8"):
        attn_bwd(do, q, k, v, *args, o, lse, idx.int().to(dev), 16.0, 1.0, csr=csr, chunk=8)
    with pytest.raises(LlsaError, match="chunk=512"):
        attn_bwd(do, q, k, v, *args, o, lse, idx.int().to(dev), 16.0, 1.0, csr=csr, chunk=512)


def test_pieces_cpu():
    with override_library_for_tests(emu_lib()):
        _run(torch.device("cpu"), 1, 1, 1024, 4, (16, 24, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,T", [(1, 2, 1024, 8), (2, 16, 1024, 16), (2, 24, 1024, 64), (1, 1, 2048, 32)])
def test_pieces_gpu(B, H, N, T):
    from llsa_amd._lib import get_lib
    _run(torch.device("cuda"), B, H, N, T, (get_lib().fine_chunk_for(B, H, N, T), 48 if T < 64 else 100, 0, 256))
