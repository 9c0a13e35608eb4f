"""What a training forward keeps for its backward: the memory that only the forward needs -- the scratch of lists made from those of the level above --
is not in it, so that no saved-tensor hook moves it and nobody holds it until the backward."""
import ctypes as C

import pytest
import torch

import llsa_amd
from emu_util import emu_lib
from llsa_amd._lib import _SIGNATURES, current_lib, override_library_for_tests


def _saved_bytes(dev, N, topks):
    q = torch.randn(1, 1, N, 64, generator=torch.Generator().manual_seed(N)).bfloat16().to(dev).requires_grad_()
    sizes = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: sizes.append(t.numel() * t.element_size()) or t, lambda t: t):
        o = llsa_amd.llsa_lk(q, q, q, topks, 16)
    if dev.type == "cuda":
        torch.autograd.grad(o, q, o.detach())
    return sum(sizes)


def test_cpu(monkeypatch):
    with override_library_for_tests(emu_lib()):
        lib = current_lib()
        res, args = _SIGNATURES["llsa_transpose_one_launch"]
        sizes = []
        for answer in (1, 0):                                 # the host's plan for lists of one launch, then for longer ones
            one_launch = C.CFUNCTYPE(res, *args)(lambda *_: answer)
            at = {n: C.cast(getattr(lib.cdll, n), C.c_void_p).value for n in _SIGNATURES}
            at["llsa_transpose_one_launch"] = C.cast(one_launch, C.c_void_p).value
            monkeypatch.setattr(lib, "host_library", lib.host.Library(at, False))
            sizes.append(_saved_bytes(torch.device("cpu"), 16384, (4, 4)))
        assert sizes[0] == sizes[1]


@pytest.mark.gpu
def test_gpu():
    """131072 tokens, topk 8 and 12: 65536 entries, which one launch makes, and more, made from the lists of the level above."""
    dev, N = torch.device("cuda"), 131072
    n1, lib = N // 16, current_lib()
    assert lib.transpose_one_launch(n1, n1, 8, 1, 1) and not lib.transpose_one_launch(n1, n1, 12, 1, 1)
    chunk = lib.fine_chunk_for(1, 1, N, 8)
    assert chunk == lib.fine_chunk_for(1, 1, N, 12)
    per_entry = 4 * n1 * 4 * 2                                # selection and list of four more entries a query block ...
    records = 4 * (lib.work_list_len(n1, n1, 12, chunk) - lib.work_list_len(n1, n1, 8, chunk))      # ... and their work records
    more = _saved_bytes(dev, N, (12, 4)) - _saved_bytes(dev, N, (8, 4))
    assert abs(more - per_entry - records) < 4 * 256          # (sections are 256-byte aligned)
