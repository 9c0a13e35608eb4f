"""Token permutation of a (B, N, C) tensor, the form in which the model puts its tokens into
Z-order and back (models/rope_dit_transformer_2d.py:963-965 `hidden_states[:, fwd_perm, :]`,
:1028-1030 `hidden_states[:, bwd_perm, :]`, :1020 after the REPA pooling)."""
from __future__ import annotations

import torch

from ..._lib import current_lib


def gather_tokens(x: torch.Tensor, index: torch.Tensor) -> torch.Tensor:
    """y[:, i, :] = x[:, index[i], :].  x is (B, N, C) with contiguous rows of a multiple of 16
    bytes; index is an integer tensor on x's device (int32 is used as it is)."""
    lib = current_lib()
    return lib.host.gather(lib.host_library, x, index)


class _TracedPermutation(torch.autograd.Function):
    """permute_tokens while torch.jit.trace records: it keeps a Python function's call as one node of the graph, of a native
    call nothing but the output's allocation."""

    @staticmethod
    def forward(ctx, x, perm, inv):
        ctx.save_for_backward(inv)
        return gather_tokens(x, perm)

    @staticmethod
    def backward(ctx, dy):
        inv, = ctx.saved_tensors
        return gather_tokens(dy, inv), None, None


def permute_tokens(x: torch.Tensor, perm: torch.Tensor, inv: torch.Tensor) -> torch.Tensor:
    """x[:, perm, :] for a permutation `perm` whose inverse is `inv`: the gradient is dy[:, inv, :]."""
    if torch._C._get_tracing_state() is not None:
        return _TracedPermutation.apply(x, perm, inv)
    lib = current_lib()
    return lib.host.permute(lib.host_library, x, perm, inv)
