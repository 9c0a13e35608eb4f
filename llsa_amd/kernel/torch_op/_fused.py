"""llsa_l1 / llsa_l2 / llsa_lk as ONE autograd node.

The reference composes the operator from nine Python launchers (six mean pools, two selections,
the attention) and autograd adds the pooled gradients afterwards.  The kernels of this package
fuse most of that work, and at the sizes of interest they finish a whole forward + backward in
less time than it takes Python to issue them, so the sequence of C-ABI calls, its one arena per call and
the autograd node are native (csrc/host/operators.cpp); this module is the door to them."""
from __future__ import annotations

from ..._lib import current_lib


def attend(q, k, v, topks, block_size, freq, qk_norm):
    """topks: one entry per pooled level, (topk1, topk2, ...): the fine blocks a query block keeps, then the blocks of
    pooled level 1, 2, ... its ancestor groups keep; len(topks) = 1 is llsa_l1, 2 is llsa_l2.
    freq: RoPE table or None; qk_norm: (gamma_q, gamma_k, eps) or None."""
    if block_size != 16:
        raise NotImplementedError("block_size must be 16")
    lib = current_lib()
    gq, gk, eps = qk_norm if qk_norm is not None else (None, None, 0.0)
    return lib.host.attend(lib.host_library, q, k, v, topks, freq, gq, gk, eps)


def selection(out):
    """The blocks the forward that produced `out` chose, finest first: (indices (B,H,N/16,T), p_indices
    (B,H,N/256,T2) or None for one level, then one more tensor per further level), int32 views of the arena its
    autograd node holds."""
    views = current_lib().host.selection(out)
    return tuple(views) if len(views) >= 2 else (views[0], None)
