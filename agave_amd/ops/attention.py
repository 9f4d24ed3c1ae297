"""Choosing the attention kernel for a step."""
from __future__ import annotations

from typing import Optional

import torch

from ..cache import PAGE
from . import attention_mfma, gemm_mfma, kernels


def attention(q: torch.Tensor, out: torch.Tensor, k_pages: torch.Tensor, v_pages: torch.Tensor,
              table: torch.Tensor, base: torch.Tensor, step, n_heads: int, n_kv: int, head_dim: int,
              scale: float, window: Optional[int], packed: bool = False) -> None:
    """Attention of the step's tokens over their sequences' cache pages (which already hold the
    step's own keys and values).  Pages in the matrix cores' tile order go to the MFMA kernels,
    pages stored row by row to the plain kernel."""
    if packed:
        attention_mfma.attention(q, out, k_pages, v_pages, table, base, step, n_heads, n_kv, head_dim, scale, window)
        return
    one_each = step.is_decode and step.n_tokens == step.n_seqs
    kernels.attn_plain(q, out, k_pages, v_pages, table, base, step.tok_seq, step.tok_pos, n_heads, n_kv, head_dim, scale, window,
                       one_token_each=one_each, span=step.page_span(window) if one_each else 1, workspace=step.workspace, most_seqs=step.most_seqs,
                       most_keys=step.max_len if step.fixed_span is None else PAGE * step.fixed_span)


def adds_slices(step, qkv, head_dim: int) -> bool:
    """Whether a step's q/k work is handed the q/k/v product (a Linear) as 32-bit slices.  From 17 tokens on: one product either fills few
    compute units with tiles or brings all of its rows to every row block (4,096 rows of 2,560, us, one product and four slices: 17 tokens
    8.1 and 7.1, 32 8.8 and 7.4, 64 10.6 and 8.0; a decode step 2.52 and 2.51 ms, 2.59 and 2.55, 2.82 and 2.75; a prompt of 20, 37 and 60 tokens
    2.64 and 2.59, 2.74 and 2.71, 2.90 and 2.83).  Two slices pay as well, though the kernels ask for four (ms, decode steps of 17, 24, 32, 48 and 64
    through 12 layers, one product and two slices: 8,192 rows of 3,840 1.312 1.343 1.378 1.513 1.645 and 1.315 1.340 1.370 1.496
    1.607; 8,192 of 5,376 2.076 2.111 2.164 2.303 2.472 and 2.078 2.102 2.146 2.275 2.432; 1,536 of 1,152 48 and 64 0.657 0.725 and
    0.659 0.720; a prompt of 60 1.568 and 1.534, 2.375 and 2.329, 0.738 and 0.730).  With fewer tokens the plans make one product of it at
    these sizes.  Prompts of several sequences are not recorded, and the host, which the GPU waits for there, has a little more to do with
    slices."""
    n = step.n_tokens
    return (17 <= n <= gemm_mfma.SKINNY_MAX_M and qkv.packed is not None
            and (head_dim in attention_mfma.FUSED_HEAD_DIMS if step.is_decode else step.n_seqs == 1)
            and gemm_mfma.slices_for(n, qkv.out_features, qkv.in_features) <= kernels.QK_MAX_SLICES)


def tokens_apart(step) -> int:
    """How a step's tokens lie for the kernels that take them four positions at a time: 0 if they are one sequence's and begin at
    a multiple of four, else of how many sequences they are."""
    return 0 if step.n_seqs == 1 and step.pos0[0] % 4 == 0 else step.n_seqs


def qk_attention(q: torch.Tensor, k: Optional[torch.Tensor], v: Optional[torch.Tensor], q_rot: torch.Tensor,
                 out: torch.Tensor, q_gain, k_gain, eps_q: float, eps_k: float, inv_freq, pos_scale: float,
                 k_pages: torch.Tensor, v_pages: torch.Tensor, table: torch.Tensor, base: torch.Tensor, step,
                 n_heads: int, n_kv: int, head_dim: int, scale: float, window: Optional[int], packed: bool,
                 partials_ok=None):
    """Head norm and rotation of q and k, k and v into the cache, and attention.  A decode step over
    pages in tile order does all of it in one kernel; otherwise the q/k kernel runs first (q into
    ``q_rot``) and the attention kernel after it.  ``partials_ok``: see
    :func:`agave_amd.ops.attention_mfma.decode_fused`; returns the partial results or None."""
    if packed and step.is_decode:
        if head_dim in attention_mfma.FUSED_HEAD_DIMS:
            return attention_mfma.decode_fused(q, k, v, out, q_gain, k_gain, eps_q, eps_k, inv_freq, pos_scale, k_pages,
                                               v_pages, table, base, step, n_heads, n_kv, head_dim, scale, window,
                                               partials_ok=partials_ok)
    kernels.qk_norm_rope_kv(q, k, v, q_rot, q_gain, k_gain, eps_q, eps_k, inv_freq, pos_scale, step.tok_seq,
                            step.tok_pos, k_pages, v_pages, table, base, n_heads, n_kv, head_dim, packed, tokens_apart(step))
    attention(q_rot, out, k_pages, v_pages, table, base, step, n_heads, n_kv, head_dim, scale, window, packed)
    return None
