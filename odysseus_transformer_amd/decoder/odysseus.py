"""Odysseus attention block and ZeRO-3 SwiGLU MLP (decoder/odysseus.py of the
reference) on the gfx950 HIP library, plus the module patcher.

Layout of one rank: the residual stream is the sequence shard (1, L/N, d); the
attention block gathers the sequence, projects it onto this rank's heads
(packed [q heads ; k heads ; v heads] rows of the column-split weight), applies
RoPE with the FULL position ids, runs causal attention over the whole sequence,
and row-splits the output projection; the MLP stays on the local tokens.

The reference subclasses transformers' LlamaFlashAttention2, which current
transformers no longer ship.  The class here is self-contained (reads the same
config fields, owns its rotary table) and keeps the reference's constructor
keywords, parameter names and shapes, and return convention.
"""
from __future__ import annotations

import inspect
import warnings
import math
from typing import Optional

import torch
from torch import nn

from .. import ops
from ..parallel_state import get_model_parallel_rank, get_model_parallel_world_size
from ..utils.allgather import allgather_bsz1
from ..utils.linear_tpsp import ColumnParallelLinear, ColumnParallelLinearAG, RowParallelLinearRS
from ..utils.linear_zero3 import LinearZeRO3


def _rope_theta(config) -> float:
    params = getattr(config, "rope_parameters", None)
    if isinstance(params, dict) and "rope_theta" in params:
        return float(params["rope_theta"])
    return float(getattr(config, "rope_theta", 10000.0))


class PackedRoPEAttnFunc(torch.autograd.Function):
    """RoPE + causal GQA attention on the packed projection, without a single copy.

    qkv3 (1, L, (Hq + 2 Hkv) * D) is the output of the packed projection; its first
    Hq + Hkv heads are rotated IN PLACE, attention reads q/k/v as head-axis slices
    of that same buffer.  Backward writes dq/dk/dv straight into the slices of one
    packed gradient buffer and un-rotates its q/k part in place.
    """

    @staticmethod
    def forward(ctx, qkv3, n_heads, n_kv_heads, head_dim, position_ids, rope_base, softmax_scale):
        B, L, _ = qkv3.shape
        qkv = qkv3.view(B, L, n_heads + 2 * n_kv_heads, head_dim)
        ops.rope_(qkv, n_heads + n_kv_heads, position_ids, rope_base)
        ctx.mark_dirty(qkv3)
        ctx.set_materialize_grads(False)  # no zero tensor for the rotated projection when nothing consumes it
        a, b = n_heads, n_heads + n_kv_heads
        out, lse = ops.attn_fwd(qkv[:, :, :a], qkv[:, :, a:b], qkv[:, :, b:], causal=True, scale=softmax_scale)
        ctx.save_for_backward(qkv3, out, lse, position_ids)
        ctx.dims = (n_heads, n_kv_heads, head_dim, rope_base, softmax_scale)
        ctx.mark_non_differentiable(lse)
        return qkv3, out, lse

    @staticmethod
    def backward(ctx, _dqkv_unused, dout, _dlse):
        qkv3, out, lse, position_ids = ctx.saved_tensors
        n_heads, n_kv_heads, head_dim, rope_base, softmax_scale = ctx.dims
        B, L, _ = qkv3.shape
        qkv = qkv3.view(B, L, n_heads + 2 * n_kv_heads, head_dim)
        if dout is None:
            dout = torch.zeros_like(out)
        if dout.stride(3) != 1:
            dout = dout.contiguous()
        dqkv = torch.empty_like(qkv)
        a, b = n_heads, n_heads + n_kv_heads
        ops.attn_bwd(qkv[:, :, :a], qkv[:, :, a:b], qkv[:, :, b:], out, lse, dout, causal=True, scale=softmax_scale,
                     dq=dqkv[:, :, :a], dk=dqkv[:, :, a:b], dv=dqkv[:, :, b:])
        ops.rope_(dqkv, b, position_ids, rope_base, inverse=True)
        if _dqkv_unused is not None:  # a consumer of the rotated projection itself (the KV cache does not differentiate)
            dqkv = dqkv + _dqkv_unused.view_as(dqkv)
        return dqkv.view_as(qkv3), None, None, None, None, None, None


class LlamaFlashAttention2TPSP(nn.Module):
    """Head-sharded causal attention over the gathered sequence
    (decoder/odysseus.py:45-271).

    Args (as the reference):
        config, layer_idx: the Llama config and the index of the layer.
        keep_master_weight_for_test: keep the unsplit weight of each sharded linear.
        pack_weight: one packed QKV projection (default) or three separate ones.
        sequence_parallel: the packed projection gathers the sequence itself and does
            not save the gathered activation.
    """

    def __init__(self, config, layer_idx: Optional[int] = None, *, keep_master_weight_for_test=False,
                 pack_weight=True, sequence_parallel=True):
        super().__init__()
        self.config = config
        self.layer_idx = layer_idx
        self.attention_dropout = getattr(config, "attention_dropout", 0.0)
        self.hidden_size = config.hidden_size
        self.num_heads = config.num_attention_heads
        self.head_dim = getattr(config, "head_dim", None) or self.hidden_size // self.num_heads
        self.num_key_value_heads = getattr(config, "num_key_value_heads", None) or self.num_heads
        self.num_key_value_groups = self.num_heads // self.num_key_value_heads
        self.max_position_embeddings = getattr(config, "max_position_embeddings", None)
        self.rope_theta = _rope_theta(config)
        self.is_causal = True
        self.fuse_rope = True   # rotary embedding inside the QKV projection and the attention backward when possible

        self.model_parallel_size = get_model_parallel_world_size()
        self.local_rank = get_model_parallel_rank()
        self.n_local_heads = self.num_heads // self.model_parallel_size
        self.n_local_kv_heads = self.num_key_value_heads // self.model_parallel_size

        self.q_proj = self.k_proj = self.v_proj = None
        self.pack_weight = pack_weight
        self.sequence_parallel = sequence_parallel
        kw = dict(bias=False, gather_output=False, keep_master_weight_for_test=keep_master_weight_for_test)
        if pack_weight:
            cls = ColumnParallelLinearAG if sequence_parallel else ColumnParallelLinear
            self.qkv_proj = cls(self.hidden_size, (self.num_heads + 2 * self.num_key_value_heads) * self.head_dim, **kw)
        else:
            self.q_proj = ColumnParallelLinear(self.hidden_size, self.num_heads * self.head_dim, **kw)
            self.k_proj = ColumnParallelLinear(self.hidden_size, self.num_key_value_heads * self.head_dim, **kw)
            self.v_proj = ColumnParallelLinear(self.hidden_size, self.num_key_value_heads * self.head_dim, **kw)
        self.o_proj = RowParallelLinearRS(self.num_heads * self.head_dim, self.hidden_size, bias=False,
                                          input_is_parallel=True,
                                          keep_master_weight_for_test=keep_master_weight_for_test)
        # arity of the tuple forward() returns: 3 as the reference (attn_output, attn_weights,
        # past_key_value); the patcher lowers it to 2 for host decoder layers that unpack two values
        self.return_arity = 3

    def forward(self, hidden_states: torch.Tensor, attention_mask: Optional[torch.Tensor] = None,
                position_ids: Optional[torch.LongTensor] = None, past_key_value=None, output_attentions: bool = False,
                use_cache: bool = False, cache_position: Optional[torch.LongTensor] = None, **kwargs):
        if past_key_value is None:
            past_key_value = kwargs.get("past_key_values")
        if type(past_key_value).__name__ == "StaticCache":
            raise ValueError(
                "`static` cache implementation is not compatible with `attn_implementation==flash_attention_2` "
                "make sure to use `sdpa` in the mean time, and open an issue at "
                "https://github.com/huggingface/transformers")
        bsz, local_q_len, _ = hidden_states.size()
        assert bsz == 1, f"bsz: {bsz}"
        # the training path: no padding and nothing in the cache yet.  A padding mask or earlier cache content takes
        # the general path below, as decoder/odysseus.py:215-263 hands both on to the host's flash-attention call.
        cached = past_key_value is not None and past_key_value.get_seq_length(self.layer_idx) > 0
        dropout = self.attention_dropout if self.training else 0.0   # decoder/odysseus.py:228
        general = cached or attention_mask is not None or dropout != 0.0
        scale = 1.0 / math.sqrt(self.head_dim)
        nh, nkv, D = self.n_local_heads, self.n_local_kv_heads, self.head_dim

        norm = kwargs.get("input_norm")   # an extension: hidden_states come before this norm, see OdysseusDecoderLayer._folds_norms
        if norm is not None and not (general and self.pack_weight and self._can_fuse_rope(hidden_states)):
            hidden_states, norm = norm(hidden_states), None

        if self.pack_weight:
            q_len = local_q_len * get_model_parallel_world_size()
            if not self.sequence_parallel:
                hidden_states = allgather_bsz1(hidden_states)
            if general:
                if norm is not None:   # ... and the norm in its prologue
                    if position_ids is not None:
                        ops.check_position_ids(position_ids, bsz, q_len, hidden_states.device)
                    qkv = ops.norm_linear_rope(hidden_states.reshape(q_len, -1), norm.weight, norm.variance_epsilon, self.qkv_proj.weight,
                                               nh + nkv, D, position_ids, self.rope_theta).view(bsz, q_len, nh + 2 * nkv, D)
                elif self._can_fuse_rope(hidden_states):   # the rotation rides in the projection's epilogue
                    qkv = ops.run_function(ops.LinearRoPEFunc, hidden_states, self.qkv_proj.weight, nh + nkv, D, position_ids,
                                           self.rope_theta)
                else:
                    qkv = self.qkv_proj(hidden_states).view(bsz, q_len, nh + 2 * nkv, D)
                    qkv = ops.apply_rope_packed(qkv, nh + nkv, position_ids, self.rope_theta)
                attn_output = self._attend_general(qkv[:, :, :nh], qkv[:, :, nh:nh + nkv], qkv[:, :, nh + nkv:],
                                                   attention_mask, past_key_value, cache_position, scale, dropout)
            elif self._can_fuse_rope(hidden_states):
                # projection, rotary embedding and attention as one autograd node: the rotation rides in the
                # projection's epilogue, its backward in the epilogues of the attention backward
                qkv3, attn_output, _ = ops.run_function(ops.QKVRoPEAttnFunc, hidden_states, self.qkv_proj.weight, nh, nkv, D,
                                                                 position_ids, self.rope_theta, scale)
            else:
                qkv3, attn_output, _ = PackedRoPEAttnFunc.apply(self.qkv_proj(hidden_states), nh, nkv, D, position_ids,
                                                                self.rope_theta, scale)
            if past_key_value is not None and not general:
                qkv = qkv3.detach().view(bsz, q_len, nh + 2 * nkv, D)
                self._update_cache(past_key_value, qkv[:, :, nh:nh + nkv], qkv[:, :, nh + nkv:], q_len, cache_position)
        else:
            hidden_states = allgather_bsz1(hidden_states)
            bsz, q_len, _ = hidden_states.size()
            q = self.q_proj(hidden_states).view(bsz, q_len, nh, D)
            k = self.k_proj(hidden_states).view(bsz, q_len, nkv, D)
            v = self.v_proj(hidden_states).view(bsz, q_len, nkv, D)
            q = ops.apply_rope_packed(q, nh, position_ids, self.rope_theta)
            k = ops.apply_rope_packed(k, nkv, position_ids, self.rope_theta)
            if general:
                attn_output = self._attend_general(q, k, v, attention_mask, past_key_value, cache_position, scale, dropout)
            else:
                if past_key_value is not None:
                    self._update_cache(past_key_value, k.detach(), v.detach(), q_len, cache_position)
                attn_output = ops.flash_attn_func(q, k, v, 0.0, softmax_scale=scale, causal=True)

        attn_output = attn_output.reshape(bsz, q_len, nh * D)
        residual = kwargs.get("residual")
        if residual is not None and self._can_fuse_residual(residual, attn_output):
            # the caller's skip connection rides in the output projection's epilogue
            attn_output = ops.run_function(ops.LinearResidualFunc, attn_output, self.o_proj.weight, residual)
        else:
            attn_output = self.o_proj(attn_output)
            if residual is not None:
                attn_output = residual + attn_output
        if self.return_arity == 2:
            return attn_output, None
        return attn_output, None, past_key_value

    def _can_fuse_rope(self, hidden_states) -> bool:
        """The fused node stands for gather(x) W^T followed by the rotation, which is what the packed projection
        computes when the gather is the identity (one rank), there is no bias and autocast asks for no cast;
        the fused kernels exist for bfloat16 and head_dim 128."""
        return (self.fuse_rope and self.head_dim == 128 and get_model_parallel_world_size() == 1
                and not _has_hooks(self.qkv_proj)
                and self.qkv_proj.bias is None and hidden_states.dtype == torch.bfloat16
                and self.qkv_proj.weight.dtype == torch.bfloat16 and hidden_states.is_cuda
                and not torch.is_autocast_enabled("cuda"))

    def _can_fuse_residual(self, residual, attn_output) -> bool:
        """The epilogue add stands for reduce_scatter(x W^T) + residual, which is only the same thing when the
        reduce-scatter is the identity (one rank), there is no bias (it is added after the scatter) and
        autocast does not ask for a cast."""
        return (get_model_parallel_world_size() == 1 and self.o_proj.bias is None and self.o_proj.input_is_parallel
                and not _has_hooks(self.o_proj)
                and residual.dtype == attn_output.dtype == self.o_proj.weight.dtype
                and not torch.is_autocast_enabled("cuda"))

    def _update_cache(self, cache, k, v, q_len, cache_position):
        """Hands the rotated keys and the values of a prefill into an EMPTY cache to the caller's cache, as
        decoder/odysseus.py:215-220 does; the attention itself then needs nothing back from it."""
        k_all, _ = cache.update(k.transpose(1, 2), v.transpose(1, 2), self.layer_idx,
                                {"cache_position": cache_position})
        assert k_all.shape[-2] == q_len, "the cache was not empty"

    def _attend_general(self, q, k, v, attention_mask, cache, cache_position, scale, dropout=0.0):
        """Attention of the rotated q (1, Lq, nh, D) over k, v (1, Lq, nkv, D) appended to the cache's earlier
        content, with an optional padding mask (1, Lk) of 0 / 1 over all keys -- what decoder/odysseus.py:215-263
        reaches through the cache's update() and the host's flash-attention forward: queries sit at the END of
        the keys (query i sees keys up to i + Lk - Lq), masked-out tokens take no part on either side and their
        output rows are zero (the unpad / varlen / pad sequence of the host collapses to one gather and one
        scatter at batch size 1)."""
        if cache is not None:
            k_all, v_all = cache.update(k.transpose(1, 2), v.transpose(1, 2), self.layer_idx,
                                        {"cache_position": cache_position})
            k, v = k_all.transpose(1, 2), v_all.transpose(1, 2)
        Lq, Lk = q.shape[1], k.shape[1]
        if attention_mask is None:
            return ops.flash_attn_func(q, k, v, dropout, softmax_scale=scale, causal=True)
        if attention_mask.dim() != 2 or attention_mask.shape[0] != 1 or attention_mask.shape[1] != Lk:
            raise ValueError(f"attention_mask must be a (1, {Lk}) padding mask over the keys; got {tuple(attention_mask.shape)}")
        keep_k = attention_mask[0] != 0
        idx_k = keep_k.nonzero().squeeze(1)
        # queries are the last Lq key positions; a single decoding query is always kept (as the host's unpad does)
        idx_q = idx_k.new_zeros(1) if Lq == 1 else keep_k[Lk - Lq:].nonzero().squeeze(1)
        if idx_k.numel() == Lk and idx_q.numel() == Lq:
            return ops.flash_attn_func(q, k, v, dropout, softmax_scale=scale, causal=True)
        if idx_q.numel() == 0 or idx_k.numel() == 0:
            return q * 0
        o = ops.flash_attn_func(q.index_select(1, idx_q), k.index_select(1, idx_k), v.index_select(1, idx_k), dropout,
                                softmax_scale=scale, causal=True)
        return torch.zeros_like(q).index_copy(1, idx_q, o)


class LlamaMLPZeRO(nn.Module):
    """SwiGLU MLP on the local tokens with ZeRO-3 sharded weights
    (decoder/odysseus.py:274-295): gate = rows [0, i) and up = rows [i, 2i) of the
    full gate_up weight."""

    def __init__(self, config):
        super().__init__()
        self.config = config
        self.hidden_size = config.hidden_size
        self.intermediate_size = config.intermediate_size
        self.gate_up_proj = LinearZeRO3(self.hidden_size, self.intermediate_size * 2, bias=False)
        self.down_proj = LinearZeRO3(self.intermediate_size, self.hidden_size, bias=False)
        act = getattr(config, "hidden_act", "silu")
        if act != "silu":
            raise NotImplementedError(f"hidden_act={act!r}: only the SiLU gate of Llama is implemented")
        self.act_fn = torch.nn.functional.silu  # kept as an attribute for introspection; the fused kernel applies it
        # SwiGLU (and its backward) inside the products' epilogues; False keeps one kernel per step
        self.fuse_elementwise = True

    def forward(self, x, residual=None, input_norm=None):
        """`residual` (an extension: the reference's module takes x only) makes the result
        residual + mlp(x) with every elementwise step fused into the products' epilogues.  `input_norm`: x comes
        before this norm (OdysseusDecoderLayer._folds_norms)."""
        if getattr(self.config, "pretraining_tp", 1) > 1:
            raise NotImplementedError("pretraining_tp > 1 is not supported yet.")
        w1, w2 = self.gate_up_proj.weight, self.down_proj.weight
        fusable = (get_model_parallel_world_size() == 1 and self.gate_up_proj.bias is None and self.down_proj.bias is None
                   and x.dtype == w1.dtype == w2.dtype and (residual is None or residual.dtype == x.dtype)
                   and not _has_hooks(self.gate_up_proj, self.down_proj)
                   and not torch.is_autocast_enabled("cuda"))
        if input_norm is not None:
            if fusable and self.fuse_elementwise and residual is not None:
                h = ops.norm_linear_swiglu_h(x.reshape(-1, x.shape[-1]), input_norm.weight, input_norm.variance_epsilon, w1)
                return ops.linear_residual(h, w2, residual.reshape(-1, residual.shape[-1])).view(residual.shape)
            x = input_norm(x)
        if fusable and self.fuse_elementwise:
            return ops.run_function(ops.SwiGLUMLPResidualFunc, x, w1, w2, residual)
        y = self.down_proj(ops.swiglu(self.gate_up_proj(x)))
        return y if residual is None else residual + y


class LlamaRMSNorm(nn.Module):
    """RMSNorm with fp32 statistics (the input_layernorm / post_attention_layernorm the
    decoder layer calls, decoder/ring.py:67,84)."""

    def __init__(self, hidden_size, eps=1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.variance_epsilon = eps

    def forward(self, hidden_states):
        return ops.rmsnorm(hidden_states, self.weight, self.variance_epsilon)


class OdysseusDecoderLayer(nn.Module):
    """h = x + attn(rms(x)); y = h + mlp(rms(h)) (the wiring at decoder/ring.py:65-86).

    fused=True (default) runs the same arithmetic with the memory-bound steps folded into their
    neighbours: both residual adds in the epilogues of the output / down projections, SwiGLU and its
    backward in the epilogues of the gate_up product and of the down projection's input gradient, and
    the sum of the two gradients at each fork of the residual stream inside the RMSNorm backward.
    fused=False keeps one kernel per step, as the reference's layer does."""

    def __init__(self, config, layer_idx: int = 0, fused: bool = True):
        super().__init__()
        self.fused = fused
        self.hidden_size = config.hidden_size
        eps = getattr(config, "rms_norm_eps", 1e-6)
        self.self_attn = LlamaFlashAttention2TPSP(config, layer_idx)
        self.mlp = LlamaMLPZeRO(config)
        self.mlp.fuse_elementwise = fused
        self.self_attn.fuse_rope = fused
        self.input_layernorm = LlamaRMSNorm(config.hidden_size, eps)
        self.post_attention_layernorm = LlamaRMSNorm(config.hidden_size, eps)
        # set by model.gradient_checkpointing_enable() on a host's layers (the reference's --grad-checkpoint,
        # train.py:163-164): in training the layer keeps its input only and runs its forward again in backward
        self.gradient_checkpointing = False

    def forward(self, hidden_states, attention_mask=None, position_ids=None, **kwargs):
        if self.gradient_checkpointing and self.training and torch.is_grad_enabled():
            from torch.utils.checkpoint import checkpoint
            return checkpoint(self._forward, hidden_states, attention_mask, position_ids, use_reentrant=False, **kwargs)
        return self._forward(hidden_states, attention_mask, position_ids, **kwargs)

    def _forward(self, hidden_states, attention_mask=None, position_ids=None, **kwargs):
        # what a host model hands its decoder layers besides (a cache to fill during a prefill)
        cache = {k: kwargs[k] for k in ("past_key_value", "past_key_values", "cache_position") if kwargs.get(k) is not None}
        if self.fused and self._folds_norms(hidden_states):
            h = self.self_attn(hidden_states, attention_mask=attention_mask, position_ids=position_ids, residual=hidden_states,
                               input_norm=self.input_layernorm, **cache)[0]
            return self.mlp(h, residual=h, input_norm=self.post_attention_layernorm)
        if self.fused:
            n1, skip = ops.rmsnorm_fork(hidden_states, self.input_layernorm.weight, self.input_layernorm.variance_epsilon)
            h = self.self_attn(n1, attention_mask=attention_mask, position_ids=position_ids, residual=skip, **cache)[0]
            n2, skip = ops.rmsnorm_fork(h, self.post_attention_layernorm.weight,
                                        self.post_attention_layernorm.variance_epsilon)
            return self.mlp(n2, residual=skip)
        residual = hidden_states
        hidden_states = self.self_attn(self.input_layernorm(hidden_states), attention_mask=attention_mask,
                                       position_ids=position_ids, **cache)[0]
        hidden_states = residual + hidden_states
        residual = hidden_states
        hidden_states = self.mlp(self.post_attention_layernorm(hidden_states))
        return residual + hidden_states


    def _folds_norms(self, hidden_states) -> bool:
        """A decoding step, or a handful of tokens that nothing records: the modules get the rows before their norm and the norm, which
        then rides in the prologue of their first product.  Only where nobody else would see those rows instead of the normalised
        ones, or a keyword that he does not know: modules that run what this file defines, and nothing around it."""
        if (not hidden_states.is_cuda or hidden_states.dtype != torch.bfloat16 or hidden_states.dim() != 3
                or hidden_states.shape[0] * hidden_states.shape[1] > ops.NORM_LINEAR_MAX_ROWS or ops.watched()
                or _EVERY_MODULE._global_forward_hooks or _EVERY_MODULE._global_forward_pre_hooks):
            return False
        m = self._modules
        n1, n2 = m["input_layernorm"], m["post_attention_layernorm"]
        return (_runs_its_own_forward(m["self_attn"], LlamaFlashAttention2TPSP) and _runs_its_own_forward(m["mlp"], LlamaMLPZeRO)
                and _runs_its_own_forward(n1, LlamaRMSNorm) and _runs_its_own_forward(n2, LlamaRMSNorm)
                and n1.weight.dtype == n2.weight.dtype == torch.bfloat16)


_EVERY_MODULE = torch.nn.modules.module
_OWN_FORWARD = {cls: cls.forward for cls in (LlamaFlashAttention2TPSP, LlamaMLPZeRO, LlamaRMSNorm)}


def _runs_its_own_forward(m, cls) -> bool:
    """Whether calling `m` is `cls`'s forward of this file and nothing else of its own: no subclass, no forward put on the instance or
    the class, no compiled call, no hooks."""
    d = m.__dict__
    return (type(m) is cls and cls.forward is _OWN_FORWARD[cls] and "forward" not in d and d.get("_compiled_call_impl") is None
            and not d["_forward_hooks"] and not d["_forward_pre_hooks"])


def _has_hooks(*modules) -> bool:
    """A fused path reads a projection's weight and never calls the module: forward hooks (or pre-hooks) that
    someone registered on it would be skipped without notice, so their presence sends the call down the
    module-by-module path."""
    return any(m is not None and (m._forward_hooks or m._forward_pre_hooks) for m in modules)


def _host_layer_unpacks_two(layer) -> bool:
    """Recent transformers decoder layers pass `position_embeddings` and unpack
    `hidden_states, _ = self.self_attn(...)`; older ones unpack three values."""
    try:
        return "position_embeddings" in inspect.signature(layer.forward).parameters
    except (TypeError, ValueError):
        return False


def _host_layer_returns_tensor(layer) -> bool:
    """Whether the host's decoder layer returns the hidden states alone (its forward is annotated `-> torch.Tensor`)
    rather than a tuple that the model unpacks."""
    try:
        ann = inspect.signature(layer.forward).return_annotation
    except (TypeError, ValueError):
        return False
    return ann is torch.Tensor or ann in ("torch.Tensor", "Tensor")


def _host_builds_no_mask(model) -> None:
    """The modules apply the causal mask themselves and refuse an explicit one.  With the `eager`
    attention implementation transformers hands every layer a dense causal mask; declaring
    flash_attention_2 (what the reference's train.py:72,84 asks for) makes the host pass None
    unless the batch is padded."""
    cfg = getattr(model, "config", None)
    if cfg is not None and getattr(cfg, "_attn_implementation", None) not in (None, "flash_attention_2"):
        try:
            cfg._attn_implementation = "flash_attention_2"   # this model's config only; nothing process-wide
        except Exception as e:   # a host that validates the assignment: the mask check in forward() still guards
            warnings.warn(f"could not declare flash_attention_2 in the model's config ({e!r}); the host may hand the "
                          "modules a dense mask, which they refuse")


def apply_odysseus_attn_patch_llama(model, use_zero3_linear=True, fuse_layers=False):
    """Swaps every layer's attention (and, by default, MLP) for the Odysseus modules
    (decoder/odysseus.py:298-309).  As in the reference the new modules are freshly
    initialised: pretrained attention / MLP weights are not carried over.

    fuse_layers=True (not in the reference) swaps the whole decoder layer for OdysseusDecoderLayer instead, with
    the host layer's two norm weights carried over: same arithmetic, but the residual adds ride in the output /
    down projections' epilogues and the gradient sums at the forks inside the RMSNorm backward.  It needs a host
    whose decoder layers return the hidden states alone (transformers >= 4.54)."""
    _host_builds_no_mask(model)
    if fuse_layers:
        if not use_zero3_linear:
            raise ValueError("fuse_layers swaps the MLP as well: it needs use_zero3_linear=True")
        for i in range(model.config.num_hidden_layers):
            old = model.model.layers[i]
            if not _host_layer_returns_tensor(old):
                raise NotImplementedError("this host's decoder layers return tuples: use fuse_layers=False")
            new = OdysseusDecoderLayer(model.config, i, fused=True).to(model.dtype)
            new.input_layernorm.weight = old.input_layernorm.weight
            new.post_attention_layernorm.weight = old.post_attention_layernorm.weight
            new.input_layernorm.variance_epsilon = getattr(old.input_layernorm, "variance_epsilon", new.input_layernorm.variance_epsilon)
            new.post_attention_layernorm.variance_epsilon = getattr(old.post_attention_layernorm, "variance_epsilon",
                                                                    new.post_attention_layernorm.variance_epsilon)
            for attr in ("attention_type", "gradient_checkpointing"):
                if hasattr(old, attr):
                    setattr(new, attr, getattr(old, attr))
            new.gradient_checkpointing = bool(getattr(new, "gradient_checkpointing", False))
            model.model.layers[i] = new
        print("Applied Odysseus patch for LlamaDecoderLayer")
        return
    for i in range(model.config.num_hidden_layers):
        layer = model.model.layers[i]
        new_module = LlamaFlashAttention2TPSP(model.config, i).to(model.dtype)
        if _host_layer_unpacks_two(layer):
            new_module.return_arity = 2
        layer.self_attn = new_module
        if use_zero3_linear:
            layer.mlp = LlamaMLPZeRO(model.config).to(model.dtype)
    print("Applied Odysseus patch for LlamaFlashAttn")
