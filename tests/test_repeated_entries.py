"""Index rows that name a block more than once (a top-k output never does, a caller's own indices may): every entry counts, as in
the reference -- in the transposed lists of all forms of the kernel, in their inverse, and in the K-side gradients."""
import contextlib

import pytest
import torch

import parity_cases as P
from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests
from oracle import llsa_oracle as O


@pytest.fixture(params=["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def dev(request):
    with contextlib.ExitStack() as stack:
        if request.param == "cpu":
            stack.enter_context(override_library_for_tests(emu_lib()))
        yield torch.device(request.param)


def _rows(B, H, Mb, T, Kb):
    """Rows of distinct values, rows with one value twice, rows with one value three times among others, rows of one value."""
    g = torch.Generator().manual_seed(Mb * T + Kb)
    idx = torch.randint(0, Kb // T, (B, H, Mb, T), generator=g) * T + torch.arange(T)        # distinct: one of every residue
    idx = idx.gather(-1, torch.rand(B, H, Mb, T, generator=g).argsort(-1))
    if T > 1:
        idx[:, :, 1::4, T - 1] = idx[:, :, 1::4, 0]
        idx[:, :, 2::8, [T // 2, T - 1]] = idx[:, :, 2::8, :1]
        idx[:, :, 3::16] = idx[:, :, 3::16, :1]
    return idx


def _check(idx, Kb, off, flat, inv):
    B, H, Mb, T = idx.shape
    ro, rf = O.transpose_indices(idx, Kb)
    assert torch.equal(off.cpu().long(), ro), "offsets differ"
    assert torch.equal(flat.cpu().long(), rf), "flat list differs"
    if inv is not None:                                       # every entry its own place, in the order of the key blocks, query blocks, slots
        e = idx.reshape(B, H, -1) * (Mb * T) + torch.arange(Mb * T)
        assert torch.equal(inv.cpu().long().reshape(B, H, -1), e.argsort(-1).argsort(-1)), "inverse positions differ"


@pytest.mark.parametrize("B,H,Mb,T,Kb,chunk", [(1, 2, 64, 8, 64, 4), (2, 1, 50, 5, 97, 2), (1, 1, 300, 12, 300, 16), (1, 1, 64, 1, 40, 0),
                                               (1, 1, 33, 4, 32800, 0),          # one workgroup, sorted afterwards
                                               (1, 1, 4112, 16, 4112, 64)])      # histogram and scatter over many workgroups
def test_lists(dev, B, H, Mb, T, Kb, chunk):
    from llsa_amd.kernel.hip.indices_transpose import transpose_indices
    idx = _rows(B, H, Mb, T, Kb)
    res = transpose_indices(idx.int().to(dev), Kb, chunk, inverse=True)
    _check(idx, Kb, res[0], res[1], res[-1])


@pytest.mark.parametrize("Mb,T,Kb,blocks", [(4096, 16, 4096, 1), (1024, 64, 1024, 3), (4112, 16, 4112, 2)])
def test_few_blocks_named_by_all(dev, Mb, T, Kb, blocks):
    """Segments with tens of thousands of entries, nearly all of them repeats."""
    from llsa_amd.kernel.hip.indices_transpose import transpose_indices
    idx = torch.randint(7, 7 + blocks, (1, 1, Mb, T), generator=torch.Generator().manual_seed(blocks))
    res = transpose_indices(idx.int().to(dev), Kb, 64, inverse=True)
    _check(idx, Kb, res[0], res[1], res[-1])


def test_lists_of_several_levels(dev):
    """A small job beside a large one: workgroups of four waves."""
    from llsa_amd.kernel.hip.indices_transpose import transpose_indices_levels
    sels = [_rows(1, 1, 4112, 16, 4112), _rows(1, 1, 257, 12, 257)]
    for l, (sel, (off, flat, extra)) in enumerate(zip(sels, transpose_indices_levels([s.int().to(dev) for s in sels], 64))):
        _check(sel, sel.shape[2], off, flat, extra if l else None)


@pytest.mark.parametrize("H,N,T", [(2, 1024, 8), pytest.param(64, 1024, 8, marks=pytest.mark.gpu), pytest.param(2, 2048, 64, marks=pytest.mark.gpu)])
def test_gradients(dev, H, N, T):
    from llsa_amd.kernel.hip._attention import attn_bwd, attn_fwd
    if dev.type == "cpu" and (H, N, T) != (2, 1024, 8):
        pytest.skip("GPU sizes")
    q, k, v, do = P.randn_inputs(1, H, N, 64, dev, seed=41)
    c = [t.cpu() for t in (q, k, v, do)]
    pk, pv = O.mean_pool(c[1]), O.mean_pool(c[2])
    idx = _rows(1, H, N // 16, T, N // 16)
    o, lse = attn_fwd(q, k, v, pk.to(dev), pv.to(dev), idx.int().to(dev), 16.0)
    got = attn_bwd(do, q, k, v, pk.to(dev), pv.to(dev), o, lse, idx.int().to(dev), 16.0, 1.0)
    ref = O.attn_bwd_l1(c[3], c[0], c[1], c[2], pk, pv, o.cpu(), lse.cpu(), idx, 16.0)
    for name, a, b in zip(("dq", "dk", "dv", "dpk", "dpv"), got, ref):
        P.close(name, a, b)
