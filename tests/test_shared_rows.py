"""Inputs whose heads, batches or tokens share memory (keys and values expanded over the heads of a group, overlapping windows): outputs and gradients are
those of copies, every gradient with an element of its own for each of its primal's."""
import pytest
import torch

import llsa_amd
from emu_util import emu_lib
from llsa_amd._lib import override_library_for_tests


def _shared(kind, g, B, H, N):
    if kind == "heads":
        return torch.randn(B, 1, N, 64, generator=g).bfloat16().expand(B, H, N, 64)
    if kind == "batches":
        return torch.randn(1, H, N, 64, generator=g).bfloat16().expand(B, H, N, 64)
    if kind == "tokens":
        return torch.randn(B, H, 1, 64, generator=g).bfloat16().expand(B, H, N, 64)
    return torch.randn(B * H * N * 64 + 8 * N, generator=g).bfloat16().as_strided((B, H, N, 64), (H * N * 64, N * 64, 32, 1))     # rows that overlap by half


def _check(dev, B, H, N, topks, kinds):
    g = torch.Generator().manual_seed(N)
    q, do = (torch.randn(B, H, N, 64, generator=g).bfloat16().to(dev) for _ in range(2))

    def moved(t):                                             # (a copy to the device makes rows of its own)
        return t if dev.type == "cpu" else t.as_strided((t.untyped_storage().nbytes() // 2,), (1,)).to(dev).as_strided(t.shape, t.stride())

    shared = [q if kind is None else moved(_shared(kind, g, B, H, N)) for kind in kinds]
    assert [t.stride() for t, kind in zip(shared, kinds) if kind == "heads"] == [(N * 64, 0, 64, 1)] * kinds.count("heads")
    results = []
    for copy in (False, True):
        leaves = [(t.clone(memory_format=torch.contiguous_format) if copy else t).detach().requires_grad_() for t in shared]
        o = llsa_amd.llsa_lk(*leaves, topks, 16)
        results.append([o.detach(), *torch.autograd.grad(o, leaves, do)])
    for name, a, b in zip(("o", "dq", "dk", "dv"), *results):
        assert torch.equal(a, b), name


CASES = [(None, "heads", "heads"), ("heads", None, "batches"), ("tokens", "windows", None)]


@pytest.mark.parametrize("kinds", CASES)
def test_cpu(kinds):
    with override_library_for_tests(emu_lib()):
        _check(torch.device("cpu"), 2, 2, 1024, (4,), kinds)


@pytest.mark.gpu
@pytest.mark.parametrize("kinds", CASES)
@pytest.mark.parametrize("B,H,N,topks", [(2, 3, 1024, (8,)), (2, 6, 16384, (16, 16))])
def test_gpu(B, H, N, topks, kinds):
    _check(torch.device("cuda"), B, H, N, topks, kinds)
