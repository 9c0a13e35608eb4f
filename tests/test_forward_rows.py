"""The forward without gradients, which selects by itself at 1024 and 2048 tokens and, at the larger sizes, reads q and v as rows and
normalises and rotates q itself, gives bit for bit what the forward with gradients gives: one and two query blocks a wave, lists of more than one and two registers, RoPE and qk norm, rows of a packed
projection."""
import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import current_lib, override_library_for_tests


def _check(dev, B, H, N, topks, rope, norm, packed, equal=False):
    import llsa_amd
    from llsa_amd.utils.rope_table import rope_table
    g = torch.Generator().manual_seed(N + topks[0])
    if packed:                               # slices of one projection: heads and tokens far apart
        qkv = torch.randn(B, N, 3, H, 64, generator=g).bfloat16().to(dev)
        q, k, v = (t.transpose(1, 2) for t in qkv.unbind(2))
    else:
        q, k, v = (torch.randn(B, H, N, 64, generator=g).bfloat16().to(dev) for _ in range(3))
    if equal:                                # equal scores everywhere, other values in every block
        q, k = torch.ones_like(q), torch.ones_like(k)
    kw = {}
    if rope:
        W = 1
        while W * W < N:
            W *= 2
        kw["rope"] = rope_table(W, dtype=torch.bfloat16)[:N].contiguous().to(dev)
    if norm:
        kw["qk_norm"] = tuple((1.0 + 0.1 * torch.randn(64, generator=g)).to(dev) for _ in range(2)) + (1e-5,)
    with torch.no_grad():
        o = llsa_amd.llsa_lk(q, k, v, topks, 16, **kw)
    ref = llsa_amd.llsa_lk(q.detach().requires_grad_(), k, v, topks, 16, **kw)
    assert torch.equal(o, ref.detach())


def _check_launch(dev, monkeypatch, N, T, T2, rope, norm):
    """The kernel itself, at sizes the operators leave to the tiles."""
    from llsa_amd.kernel.hip._attention import attn_fwd
    from llsa_amd.kernel.hip.mean_pool import mean_pool1d
    from llsa_amd.kernel.hip.rms_norm import my_rms_norm_fn
    from llsa_amd.kernel.hip.rope import my_rope_fn
    from llsa_amd.utils.rope_table import rope_table
    lib = current_lib()
    g = torch.Generator().manual_seed(N + T)
    qkv = torch.randn(1, N, 3, 2, 64, generator=g).bfloat16().to(dev)
    q, k, v = (t.transpose(1, 2) for t in qkv.unbind(2))
    gamma = (1.0 + 0.1 * torch.randn(64, generator=g)).to(dev)
    side = 1 << ((N - 1).bit_length() + 1) // 2
    freq = rope_table(side, dtype=torch.bfloat16)[:N].contiguous().to(dev)
    ready = my_rms_norm_fn(q, gamma, 1e-5) if norm else q
    ready = my_rope_fn(ready, freq) if rope else ready
    pk, pv = mean_pool1d(k, 16), mean_pool1d(v, 16)
    sel = P._hot_indices(1, 2, N // 16, N // 16, T, 3, 11).int().to(dev)
    kw = {}
    if T2:
        kw = {"pk2": mean_pool1d(pk, 16), "pv2": mean_pool1d(pv, 16), "token_weight_2": 256.0,
              "p_indices": P._hot_indices(1, 2, N // 256, N // 256, T2, 1, 12).int().to(dev)}
    ref, _ = attn_fwd(ready, k, v, pk, pv, sel, 16.0, **kw)
    real = lib.attn_fwd

    def on_rows(a, stream):
        f = a._obj
        f.qr = f.vt = f.lse = None
        for n, t in (("q", q), ("v", v)):
            setattr(f, n, t.data_ptr())
            for axis, s in zip("bhn", t.stride()):
                setattr(f, f"s{n}{axis}", s)
        f.freq_q, f.gamma_q, f.eps_q = freq.data_ptr() if rope else None, gamma.data_ptr() if norm else None, 1e-5
        return real(a, stream)

    monkeypatch.setattr(lib, "attn_fwd", on_rows)
    o, _ = attn_fwd(ready, k, v, pk, pv, sel, 16.0, **kw)
    monkeypatch.undo()
    assert torch.equal(o, ref)


@pytest.mark.parametrize("rope,norm", [(False, False), (True, True)])
def test_launch_cpu(monkeypatch, rope, norm):
    with override_library_for_tests(emu_lib()):
        _check_launch(torch.device("cpu"), monkeypatch, 1024, 4, 0, rope, norm)


@pytest.mark.gpu
@pytest.mark.parametrize("rope,norm", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("N,T,T2", [(1024, 4, 0), (2048, 128, 0), (7168, 12, 0), (16384, 8, 4)])
def test_launch_gpu(monkeypatch, N, T, T2, rope, norm):
    _check_launch(torch.device("cuda"), monkeypatch, N, T, T2, rope, norm)


@pytest.mark.parametrize("N,T", [(1024, 4), (2048, 64)])
def test_selecting_cpu(N, T):
    with override_library_for_tests(emu_lib()):
        assert current_lib().attn_fwd_selects(1, 1, N, T, 1)
        _check(torch.device("cpu"), 1, 1, N, (T,), False, False, False)
        _check(torch.device("cpu"), 1, 1, N, (T,), False, False, False, equal=True)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,T", [(1, 6, 1024, 8), (1, 1, 1024, 64), (3, 5, 1024, 12), (8, 16, 1024, 20), (1, 1, 2048, 4), (2, 3, 2048, 64), (4, 6, 2048, 16)])
def test_selecting_gpu(B, H, N, T):
    assert current_lib().attn_fwd_selects(B, H, N, T, 1)
    _check(torch.device("cuda"), B, H, N, (T,), True, False, True)
    _check(torch.device("cuda"), B, H, N, (T,), False, False, False, equal=True)


def test_which_sizes_select():
    with override_library_for_tests(emu_lib()):
        ask = current_lib().attn_fwd_selects
        assert ask(8, 16, 1024, 8, 1) and not ask(3, 43, 1024, 8, 1)
        assert ask(4, 6, 2048, 8, 1) and not ask(5, 5, 2048, 8, 1) and ask(8, 8, 2048, 32, 1) and not ask(5, 13, 2048, 32, 1)
        assert not ask(1, 1, 3072, 8, 1) and not ask(1, 1, 4096, 8, 1) and not ask(1, 1, 16384, 8, 2) and not ask(1, 1, 1024, 6, 1)


# more than 131072 tokens over all heads; one and two query blocks a wave, lists in one and two registers
@pytest.mark.gpu
@pytest.mark.parametrize("rope,norm,packed", [(False, False, False), (True, False, True), (False, True, True), (True, True, False)])
@pytest.mark.parametrize("B,H,N,topks", [(12, 11, 1024, (8,)), (1, 3, 65536, (64,)), (1, 3, 49152, (16, 8)), (8, 6, 16384, (16, 16))])
def test_gpu(B, H, N, topks, rope, norm, packed):
    _check(torch.device("cuda"), B, H, N, topks, rope, norm, packed)
