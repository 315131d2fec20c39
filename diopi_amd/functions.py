"""Python callers of the seven LLaMA-inference operators, through the C ABI.

Each function mirrors the wrapper of the same name in
``diopi_test/python/conformance/diopi_functions.py`` of the reference
(rotary_emb 7030-7037, rms_norm 7040-7070, rms_norm_backward 7073-7109,
destindex_copy_kv 7896-7902, token_attention 7905-7911,
token_softmax_reducev 7914-7939, context_attention 7942-7948): same argument
order and meaning, outputs allocated by the caller side with the reference's
shape/dtype rules, return code checked with the reference's policy.

Arguments are torch tensors on the GPU; they are wrapped as diopiTensor handles
for the duration of the call.  Without a context the operators run on torch's
current stream.  A context given explicitly brings its own stream; the wrappers
order that stream after torch's current stream on entry and torch's current
stream after it on exit, so results can be used by torch code directly.
"""
from __future__ import annotations

from typing import Optional, Sequence

import math

import torch

from . import runtime as rt
from .runtime import check_returncode

# inv_rms of the last rms_norm call, consumed by rms_norm_backward
# (reference: GLOBAL_STATE["rms_norm_inv_rms"], diopi_functions.py:7069, 7087)
GLOBAL_STATE = {}


class _on_stream:
    """Orders the stream of an explicit context with torch's current stream around a call."""

    def __init__(self, ctx: rt.Context, tensor: torch.Tensor):
        self.ctx = ctx
        self.current = torch.cuda.current_stream() if tensor.is_cuda else None
        # a context on the current stream is in order by itself
        self.other = self.current is not None and ctx.torch_stream is not None and ctx.torch_stream != self.current
        # a context that made its own native stream has no torch stream to order against: the host waits instead, before
        # the call for what torch has queued (fills and copies of the arguments) and after it for the operator
        self.foreign = self.current is not None and ctx.torch_stream is None

    def __enter__(self):
        if self.other:
            self.ctx.torch_stream.wait_stream(self.current)
        elif self.foreign:
            self.current.synchronize()
        return self

    def __exit__(self, *exc):
        if self.other:
            self.current.wait_stream(self.ctx.torch_stream)
        elif self.foreign:
            self.ctx.synchronize()
        # scratch an operator took from the context (partial sums, tile plans, score buffers) belongs to that call:
        # hand it back to the context's pool, as the reference harness does after every case (litert.hpp:268-276);
        # the pool is reused in stream order, so a later call on this context may overwrite it safely
        self.ctx.clear_tensors()
        return False


def _call(name: str, ctx: Optional[rt.Context], tensor: torch.Tensor, *args):
    """Calls an operator by its C name; `tensor` tells whether the call is on the device at all."""
    op = getattr(rt.torch_ops(), name)
    if ctx is None:
        ret = op(None, *args)
    else:
        with _on_stream(ctx, tensor):
            ret = op(ctx.handle.value if ctx.handle else 0, *args)  # 0: a closed context, which the operator refuses
    value = None
    if type(ret) is tuple:  # the operators that answer more than their return code
        ret, value = ret
    if ret:
        check_returncode(ret, name)
    return value


def rotary_emb(input: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, conj: bool, interleaved: bool, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    out = torch.empty_like(input, memory_format=torch.contiguous_format)
    _call("diopiRotaryEmbedding", ctx, input, out, input, cos, sin, bool(conj), bool(interleaved))
    return out


def rotary_emb_v2(query: torch.Tensor, key: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, dim: int, ctx: Optional[rt.Context] = None):
    """In place on query and key, like the reference wrapper (diopi_functions.py:8051-8056)."""
    _call("diopiRotaryEmbeddingV2", ctx, query, query, key, cos, sin, int(dim))
    return query, key


def apply_penalty(logits: torch.Tensor, presence_penalty: torch.Tensor, frequency_penalty: torch.Tensor, p_token_ids: torch.Tensor,
                  p_token_counts: torch.Tensor, p_cumsum_seq_len: torch.Tensor, p_max_len_in_batch: int, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """In place on logits, like the reference wrapper (diopi_functions.py:7851-7895)."""
    _call("diopiApplyPenalty", ctx, logits, logits, presence_penalty, frequency_penalty, p_token_ids, p_token_counts, p_cumsum_seq_len, int(p_max_len_in_batch))
    return logits


def apply_penalty_v2(logits: torch.Tensor, presence_penalty: torch.Tensor, frequency_penalty: torch.Tensor, repetition_penalty: torch.Tensor,
                     p_token_ids: torch.Tensor, p_token_counts: torch.Tensor, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """In place on logits, like the reference wrapper (diopi_functions.py:8019-8049)."""
    _call("diopiApplyPenaltyV2", ctx, logits, logits, presence_penalty, frequency_penalty, repetition_penalty, p_token_ids, p_token_counts)
    return logits


def rms_norm(input: torch.Tensor, normalized_shape: Sequence[int], weight: torch.Tensor, bias: Optional[torch.Tensor], eps: float,
             ctx: Optional[rt.Context] = None, out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    out = torch.empty(input.shape, dtype=out_dtype or input.dtype, device=input.device)
    n = len(normalized_shape)
    inv_shape = list(input.shape)[: input.dim() - n]
    # 16-bit and fp32 inputs keep their statistics in fp32, fp64 inputs in fp64
    inv_dtype = torch.float64 if input.dtype == torch.float64 else torch.float32
    inv_rms = torch.empty(inv_shape, dtype=inv_dtype, device=input.device)
    _call("diopiRMSNorm", ctx, input, out, inv_rms, input, normalized_shape, weight, bias, float(eps))
    GLOBAL_STATE["rms_norm_inv_rms"] = inv_rms
    return out


def rms_norm_backward(grad_outputs: Sequence[torch.Tensor], input: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
                      normalized_shape: Sequence[int], eps: float, ctx: Optional[rt.Context] = None, inv_rms: Optional[torch.Tensor] = None) -> dict:
    grad_input = torch.empty_like(input)
    grad_weight = torch.empty_like(weight)
    grad_bias = torch.empty_like(bias) if bias is not None else None
    if inv_rms is None:
        inv_rms = GLOBAL_STATE.pop("rms_norm_inv_rms")
    _call("diopiRMSNormBackward", ctx, input, grad_input, grad_weight, grad_bias, grad_outputs[0], input, weight, bias, inv_rms, normalized_shape, float(eps))
    out = {"input": grad_input, "weight": grad_weight}
    if bias is not None:
        out["bias"] = grad_bias
    return out


def root_mean_square_norm_inp(inoutput: torch.Tensor, scale: torch.Tensor, eps: float, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """In-place RMS normalisation of every row (functions_lmdeploy.h:31-38 of the reference)."""
    _call("diopiRootMeanSquareNormInp", ctx, inoutput, inoutput, scale, float(eps))
    return inoutput


def fused_add_root_mean_square_norm_inp(inoutput: torch.Tensor, residual: torch.Tensor, bias: Optional[torch.Tensor], scale: torch.Tensor, eps: float,
                                        ctx: Optional[rt.Context] = None):
    """residual += inoutput + bias; inoutput = RMSNorm(residual) * scale (functions_lmdeploy.h:40-49 of the reference)."""
    _call("diopiFusedAddRootMeanSquareNormInp", ctx, inoutput, inoutput, residual, bias, scale, float(eps))
    return inoutput, residual


def fused_decoder_attention_inp(inoutput: torch.Tensor, qkv_weight: torch.Tensor, qkv_bias: Optional[torch.Tensor], workspace: Optional[torch.Tensor],
                                fusion_level: int, key_cache: torch.Tensor, value_cache: torch.Tensor, finished: Optional[torch.Tensor],
                                total_padding_tokens: Optional[torch.Tensor], sequence_lengths: torch.Tensor, step: int, layer_id: int, local_head_num: int,
                                local_kv_head_num: int, size_per_head: int, max_seq_len: int, rotary_embedding: int, rope_theta: float,
                                ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """One decode step of self-attention, from hidden states to attention output (functions_lmdeploy.h:104-135 of the reference).

    `workspace` None allocates one of the size the operator asks for (the header's size query: workspace_size < 0)."""
    shape = (int(fusion_level), key_cache, value_cache, finished, total_padding_tokens, sequence_lengths, int(step), int(layer_id), int(local_head_num),
             int(local_kv_head_num), int(size_per_head), int(max_seq_len), int(rotary_embedding), float(rope_theta))
    name = "diopiFusedDecoderAttentionInp"
    if workspace is None:
        bytes_needed = _call(name, ctx, inoutput, inoutput, qkv_weight, qkv_bias, None, -1, *shape)
        workspace = torch.empty(max(bytes_needed, 16), dtype=torch.int8, device=inoutput.device)
    _call(name, ctx, inoutput, inoutput, qkv_weight, qkv_bias, workspace, workspace.numel() * workspace.element_size(), *shape)
    return inoutput


def destindex_copy_kv(k: torch.Tensor, dest_loc: torch.Tensor, out: torch.Tensor, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    _call("diopiDestIndexCopyKV", ctx, out, out, k, dest_loc)
    return out


def token_attention(q: torch.Tensor, k: torch.Tensor, out: torch.Tensor, b_loc: torch.Tensor, b_start_loc: torch.Tensor, b_seq_len: torch.Tensor,
                    max_input_len: int, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    _call("diopiTokenAttentionInference", ctx, out, out, q, k, b_loc, b_start_loc, b_seq_len, int(max_input_len))
    return out


def token_softmax_reducev(logics: torch.Tensor, v: torch.Tensor, out: torch.Tensor, b_loc: torch.Tensor, b_start_loc: torch.Tensor,
                          b_seq_len: torch.Tensor, max_input_len: int, other_kv_index: int, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    _call("diopiTokenSoftmaxReduceVInference", ctx, out, out, logics, v, b_loc, b_start_loc, b_seq_len, int(max_input_len), int(other_kv_index))
    return out


def context_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out: torch.Tensor, b_start_loc: torch.Tensor, b_seq_len: torch.Tensor,
                      max_input_len: int, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    _call("diopiContextAttentionInference", ctx, out, out, q, k, v, b_start_loc, b_seq_len, int(max_input_len))
    return out


def context_attention_no_alloc(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out: torch.Tensor, b_start_loc: torch.Tensor, b_seq_len: torch.Tensor,
                               max_input_len: int, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """context_attention through the entry point that allocates nothing (no counterpart in the reference): the tile plan
    lives in a static device array of the library, so calls on one device must not overlap: the ones without a context
    all go to the default context's stream."""
    ctx = ctx if ctx is not None else rt.default_context()
    _call("diopiContextAttentionInferenceNoAlloc", ctx, out, out, q, k, v, b_start_loc, b_seq_len, int(max_input_len))
    return out


def flash_attention_varlen(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cu_seqlens_q: torch.Tensor, cu_seqlens_kv: torch.Tensor, alibi_slopes,
                           max_seqlen_q: int, max_seqlen_kv: int, p_dropout: float, softmax_scale, is_causal: bool, window_size_left: int = -1,
                           window_size_right: int = -1, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """diopi_functions.py:7530-7590 of the reference: allocates out and softmax_lse [batch, heads, max_seqlen_q] (kept in
    GLOBAL_STATE["flash_attention_varlen_softmax_lse"]), replaces a missing scale by 1/sqrt(head_dim), returns out."""
    out = torch.empty_like(q)
    batch = cu_seqlens_q.numel() - 1
    lse = torch.zeros(batch, q.shape[1], int(max_seqlen_q), dtype=torch.float32, device=q.device)
    scale = 1.0 / math.sqrt(q.shape[-1]) if not softmax_scale else float(softmax_scale)
    _call("diopiFlashAttentionVarLen", ctx, out, out, lse, None, q, k, v, cu_seqlens_q, cu_seqlens_kv, alibi_slopes, int(max_seqlen_q), int(max_seqlen_kv),
          float(p_dropout), scale, bool(is_causal), int(window_size_left), int(window_size_right))
    GLOBAL_STATE["flash_attention_varlen_softmax_lse"] = lse
    return out


def flash_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, alibi_slopes, p_dropout: float, softmax_scale, is_causal: bool,
                    window_size_left: int = -1, window_size_right: int = -1, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """diopi_functions.py flash_attention of the reference: allocates out and softmax_lse [batch, heads, seq_len] (kept in
    GLOBAL_STATE["flash_attention_softmax_lse"]), replaces a missing scale by 1/sqrt(head_dim), returns out."""
    out = torch.empty_like(q)
    lse = torch.zeros(q.shape[0], q.shape[2], q.shape[1], dtype=torch.float32, device=q.device)
    scale = 1.0 / math.sqrt(q.shape[-1]) if not softmax_scale else float(softmax_scale)
    _call("diopiFlashAttention", ctx, out, out, lse, None, q, k, v, alibi_slopes, float(p_dropout), scale, bool(is_causal), int(window_size_left),
          int(window_size_right))
    GLOBAL_STATE["flash_attention_softmax_lse"] = lse
    return out


def multihead_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, dropout_p: float, is_causal: bool, return_debug_mask: bool, scale,
                        ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """diopi_functions.py:7112-7149 of the reference (softmax_lse kept in GLOBAL_STATE["multihead_attention_softmax_lse"])."""
    out = torch.empty_like(q)
    lse = torch.zeros(q.shape[0], q.shape[2], q.shape[1], dtype=torch.float32, device=q.device)
    softmax_scale = 1.0 / math.sqrt(q.shape[-1]) if not scale else float(scale)
    _call("diopiMultiHeadAttention", ctx, out, q, k, v, float(dropout_p), bool(is_causal), bool(return_debug_mask), softmax_scale, out, lse, None, None)
    GLOBAL_STATE["multihead_attention_softmax_lse"] = lse
    return out


def multihead_attention_varlen(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cu_seqlens: torch.Tensor, max_seqlen: int, dropout_p: float,
                               is_causal: bool, return_debug_mask: bool, scale, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """diopi_functions.py:7195-7250 of the reference (softmax_lse kept in GLOBAL_STATE["multihead_attention_varlen_softmax_lse"])."""
    out = torch.empty_like(q)
    lse = torch.zeros(cu_seqlens.numel() - 1, q.shape[1], int(max_seqlen), dtype=torch.float32, device=q.device)
    softmax_scale = 1.0 / math.sqrt(q.shape[-1]) if not scale else float(scale)
    _call("diopiMultiHeadAttentionVarLen", ctx, out, q, k, v, cu_seqlens, cu_seqlens, int(max_seqlen), int(max_seqlen), float(dropout_p), bool(is_causal),
          bool(return_debug_mask), softmax_scale, out, lse, None, None)
    GLOBAL_STATE["multihead_attention_varlen_softmax_lse"] = lse
    return out


def prompt_flash_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, attenMask: Optional[torch.Tensor], actualSeqLengths: Sequence[int],
                           maxInputLen: int, numHeads: int, numKeyValueHeads: int, dim: int, ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """diopi_functions.py:7951-7981 of the reference."""
    out = torch.empty_like(query)
    _call("diopiPromptFlashAttention", ctx, out, out, query, key, value, attenMask, actualSeqLengths, int(maxInputLen), int(numHeads), int(numKeyValueHeads),
          int(dim))
    return out


def paged_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, attenMask: Optional[torch.Tensor], actualSeqLengths: Sequence[int],
                    numHeads: int, numKeyValueHeads: int, dim: int, blockTable: torch.Tensor, blockSize: int,
                    ctx: Optional[rt.Context] = None) -> torch.Tensor:
    """diopi_functions.py:7984-8016 of the reference."""
    out = torch.empty_like(query)
    _call("diopiPagedAttention", ctx, out, out, query, key, value, attenMask, actualSeqLengths, int(numHeads), int(numKeyValueHeads), int(dim), blockTable,
          int(blockSize))
    return out
