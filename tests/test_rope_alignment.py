"""A rope table that starts at any element of its storage: accepted at every size, with and without gradients, with the results of an aligned one.  The
kernels read the table in 16-byte pieces, so what they are given is 16-byte aligned."""
import ctypes as C

import pytest
import torch

import llsa_amd
from emu_util import emu_lib
from llsa_amd._lib import _SIGNATURES, current_lib, override_library_for_tests
from llsa_amd.utils.rope_table import rope_table


def _inputs(dev, B, H, N, offset):
    g = torch.Generator().manual_seed(N + offset)
    q, k, v = (torch.randn(B, H, N, 64, generator=g).bfloat16().to(dev) for _ in range(3))
    side = 1 << ((N - 1).bit_length() + 1) // 2
    table = rope_table(side, dtype=torch.bfloat16)[:N].contiguous().to(dev)
    moved = torch.zeros(N * 64 + offset, dtype=torch.bfloat16, device=dev)[offset:].view(N, 64)
    assert moved.is_contiguous() and moved.data_ptr() % 16 == 2 * offset
    return q, k, v, table, moved.copy_(table)


def _check(dev, B, H, N, topks, grad, offset):
    q, k, v, table, moved = _inputs(dev, B, H, N, offset)
    results = []
    for rope in (table, moved):
        leaves = [t.detach().clone().requires_grad_(grad) for t in (q, k, v)]
        o = llsa_amd.llsa_lk(*leaves, topks, 16, rope=rope)
        results.append([o.detach(), *(torch.autograd.grad(o, leaves, q) if grad else ())])
    for a, b in zip(*results):
        assert torch.equal(a, b)


class _Aligned:
    """The CPU build of the kernels behind a pooling pass that refuses a table the GPU would have to read across 16-byte pieces (the CPU build cannot)."""

    def __init__(self, lib):
        def pool(items, n, freq, B, H, stream):
            return -1 if (freq or 0) % 16 else lib.pool_pyramid_fwd(items, n, freq, B, H, stream)
        res, args = _SIGNATURES["llsa_pool_pyramid_fwd"]
        self.callback = C.CFUNCTYPE(res, *args)(pool)
        at = {n: C.cast(getattr(lib.cdll, n), C.c_void_p).value for n in _SIGNATURES}
        at["llsa_pool_pyramid_fwd"] = C.cast(self.callback, C.c_void_p).value
        self.host_library = lib.host.Library(at, False)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("offset", [1, 4])
def test_cpu(monkeypatch, grad, offset):
    with override_library_for_tests(emu_lib()):
        lib = current_lib()
        guarded = _Aligned(lib)
        monkeypatch.setattr(lib, "host_library", guarded.host_library)
        _check(torch.device("cpu"), 1, 1, 1024, (4,), grad, offset)


# without gradients: up to 131072 tokens over all heads the forward reads q as tiles, above as rows
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,N,topks,grad", [(1, 2, 1024, (8,), False), (1, 2, 65536, (8,), False), (1, 3, 65536, (8,), False), (3, 3, 16384, (16, 8), False),
                                              (1, 2, 1024, (8,), True), (3, 3, 16384, (16, 8), True)])
@pytest.mark.parametrize("offset", [1, 4])
def test_gpu(B, H, N, topks, grad, offset):
    _check(torch.device("cuda"), B, H, N, topks, grad, offset)
