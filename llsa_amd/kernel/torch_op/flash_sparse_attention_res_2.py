"""llsa_l2: two pooled levels.  Mirrors torch_op/flash_sparse_attention_res_2.py of the
reference: `FlashSparseResidualAttentionL2`, `flash_sparse_residual_attention_l2_op`,
`llsa_l2(q, k, v, topk1=8, topk2=8, block_size=16)` with the same positional arguments,
plus the optional `rope=freq` and `qk_norm=(gamma_q, gamma_k, eps)` described in
flash_sparse_attention_res_1.
"""
from __future__ import annotations

import torch
from torch.autograd import Function

from ..hip.mean_pool import mean_pool1d
from ._fused import attend
from ..hip.sparse_attention_res_2 import (sparse_indices_attn_res_2_2_fwd,
                                          sparse_indices_attn_res_scatter_2_2_bwd_v2)
from ..hip.topk import compute_topk_indices_sparse, gen_sparse_indices


class FlashSparseResidualAttentionL2(Function):
    """flash_sparse_attention_res_2.py:10-42."""

    @staticmethod
    def forward(ctx, q, k, v, pq, pk, pv, pq2, pk2, pv2, topk, topk2, token_weight=1, token_weight_2=1,
                block_size=16):
        p_indices = gen_sparse_indices(pq2, pk2, topk2)
        topk2 = p_indices.shape[-1]
        indices = compute_topk_indices_sparse(pq, pk, p_indices, topk, topk2, block_size)
        output, m = sparse_indices_attn_res_2_2_fwd(q, k, v, pk, pv, pk2, pv2, indices, p_indices, topk, topk2,
                                                    token_weight, token_weight_2, int(block_size ** 0.5))
        ctx.save_for_backward(q, k, v, pk, pv, pk2, pv2, output, m, indices, p_indices)
        ctx.topk = topk
        ctx.topk2 = topk2
        ctx.block_size = block_size
        ctx.token_weight = token_weight
        ctx.token_weight_2 = token_weight_2
        return output

    @staticmethod
    def backward(ctx, do):
        q, k, v, pk, pv, pk2, pv2, o, m, indices, p_indices = ctx.saved_tensors
        return *sparse_indices_attn_res_scatter_2_2_bwd_v2(do, q, k, v, pk, pv, pk2, pv2, o, m, indices, p_indices,
                                                           ctx.topk, ctx.topk2, ctx.block_size, ctx.token_weight,
                                                           ctx.token_weight_2), None, None, None, None, None


flash_sparse_residual_attention_l2_op = FlashSparseResidualAttentionL2.apply


def llsa_l2(q, k, v, topk1=8, topk2=8, block_size=16, rope=None, qk_norm=None):
    """flash_sparse_attention_res_2.py:48-59."""
    return attend(q, k, v, (int(topk1), int(topk2)), block_size, rope, qk_norm)


def llsa_lk(q, k, v, topks, block_size=16, rope=None, qk_norm=None):
    """Any number of pooled levels (1 to 4): topks = (topk1, ..., topk_k), the fine blocks a query block keeps and then
    the blocks of pooled level 1, 2, ... that its ancestor groups keep.  The reference has k = 1 (llsa_l1) and k = 2
    (llsa_l2), whose coarsest level every query still reads in full (N/256 tokens, sparse_attention_res_2.py:127-149);
    deeper hierarchies continue the scheme by induction: dense selection over the N/16^k tokens of the coarsest
    level, parent-guided selection level by level down to the fine blocks, and every query reads topk1 fine blocks,
    16 topk_(l+1) tokens of pooled level l < k with weight 16^l, and all N/16^k tokens of level k with weight 16^k.
    N must be a multiple of 64 * 16^k."""
    return attend(q, k, v, tuple(int(t) for t in topks), block_size, rope, qk_norm)


def llsa_l3(q, k, v, topk1=8, topk2=8, topk3=8, block_size=16, rope=None, qk_norm=None):
    """Three pooled levels (llsa_lk with three entries): N a multiple of 262144."""
    return llsa_lk(q, k, v, (topk1, topk2, topk3), block_size, rope, qk_norm)


def llsa_l2_unfused(q, k, v, topk1=8, topk2=8, block_size=16):
    """The reference's own composition: six mean_pool1d calls, then the op."""
    pq1 = mean_pool1d(q, block_size)
    pk1 = mean_pool1d(k, block_size)
    pv1 = mean_pool1d(v, block_size)
    pq2 = mean_pool1d(pq1, block_size)
    pk2 = mean_pool1d(pk1, block_size)
    pv2 = mean_pool1d(pv1, block_size)
    return flash_sparse_residual_attention_l2_op(q, k, v, pq1, pk1, pv1, pq2, pk2, pv2, topk1, topk2, block_size,
                                                 block_size * block_size, block_size)
