"""One decoder layer of izwi-core's Qwen3 model at one token, composed from the library's calls.

Mirror of `Qwen3Layer::forward` (qwen3/core.rs:1863-1881) with `Qwen3Attention::forward`'s
single-token path (core.rs:1446-1575: q/k/v projections, per-head q/k norm, rotary embedding, cache
append, grouped-query attention, output projection) and `Qwen3Mlp::forward` (core.rs:1786-1798),
f32 activations.  Every arithmetic step is one library call; torch only appends the new key /
value rows to the caches in the unfused form and owns the tensors.  Per layer: 5 kernel launches, 6 where
the attention is split over the cache (the two RMSNorms ride in the projection launches behind them; q/k norm, rotary and the cache
append ride in the attention launch) behind one library call, or 11 to 12 with the reference's separate hooks and two copies,
where the reference's eager path issues one per operator.
"""
from __future__ import annotations

import torch

from .capi import check, lib
from .decode_ops import (_ok, decode_attention_step, qk_norm_rope_append, try_fused_decode_gqa_attention_with_kv_len, try_fused_qk_rms_norm,
                         try_fused_rms_norm, try_fused_rope_pair_bshd)
from .qmatmul import QMatMul, Qwen3GateUpProjection, _stream_ptr, forward_group


class Qwen3DecodeLayer:
    def __init__(self, input_layernorm: torch.Tensor, post_attention_layernorm: torch.Tensor, q_proj: QMatMul,
                 k_proj: QMatMul, v_proj: QMatMul, qk_norm_weight: torch.Tensor, o_proj: QMatMul, gate_proj: QMatMul,
                 up_proj: QMatMul, down_proj: QMatMul, num_heads: int, num_kv_heads: int, head_dim: int,
                 rms_norm_eps: float = 1e-6, fuse_prep: bool = True, fuse_norm: bool = True, fuse_step: bool = True):
        self.w_in, self.w_post, self.qk_w = input_layernorm, post_attention_layernorm, qk_norm_weight
        self.qkv = (q_proj, k_proj, v_proj)
        self.o_proj, self.down_proj = o_proj, down_proj
        self.gate_up = Qwen3GateUpProjection.new_separate(gate_proj, up_proj)
        self.heads, self.kv_heads, self.d, self.eps = num_heads, num_kv_heads, head_dim, rms_norm_eps
        self.fuse_prep = fuse_prep  # q/k norm, rotary and cache append as one launch instead of four
        self.fuse_norm = fuse_norm  # the two RMSNorms inside the projection launches that follow them
        self.fuse_step = fuse_step  # q/k norm, rotary and cache append inside the attention launch

    def forward(self, x: torch.Tensor, cos_sin: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                pos: int) -> torch.Tensor:
        """x [1, hidden] f32; cos_sin [1, head_dim] for position `pos`; caches [1, kv_heads, capacity,
        head_dim] holding positions < pos.  Returns the layer's output [1, hidden]; the caches gain
        position `pos`."""
        h, kv, d = self.heads, self.kv_heads, self.d
        if self.fuse_norm and self.fuse_prep and self.fuse_step:
            out = self._forward_one_call(x, cos_sin, k_cache, v_cache, pos)
            if out is not None:
                return out
        if self.fuse_norm:  # input_layernorm inside the q|k|v launch
            q, k, v = forward_group(self.qkv, x, norm_weight=self.w_in, eps=self.eps)
        else:
            q, k, v = forward_group(self.qkv, try_fused_rms_norm(x, self.w_in, self.eps))
        if self.fuse_prep and self.fuse_step:
            attn = decode_attention_step(q, k, v, self.qk_w, cos_sin, k_cache, v_cache, pos, self.eps, d ** -0.5)
        else:
            if self.fuse_prep:
                q4 = qk_norm_rope_append(q, k, v, self.qk_w, cos_sin, k_cache, v_cache, pos, self.eps)
            else:  # the same steps as the reference's separate hooks
                q4, k4 = try_fused_qk_rms_norm(q.view(1, 1, h, d), k.view(1, 1, kv, d), self.qk_w, self.eps)
                q4, k4 = try_fused_rope_pair_bshd(q4, k4, cos_sin)
                k_cache[0, :, pos] = k4.view(kv, d)
                v_cache[0, :, pos] = v.view(kv, d)
            attn = try_fused_decode_gqa_attention_with_kv_len(q4.view(1, h, 1, d), k_cache, v_cache, h, kv, d, pos + 1,
                                                              d ** -0.5)
        x = self.o_proj.forward_fused(attn.view(1, h * d), residual=x)       # x + o_proj(attn)
        if self.fuse_norm:  # post_attention_layernorm inside the gate|up launch
            hidden = self.gate_up.forward_silu_mul(x, norm_weight=self.w_post, eps=self.eps)
        else:
            hidden = self.gate_up.forward_silu_mul(try_fused_rms_norm(x, self.w_post, self.eps))  # silu(gate) * up
        return self.down_proj.forward_fused(hidden, residual=x)              # x + down_proj(hidden)

    def _forward_one_call(self, x, cos_sin, k_cache, v_cache, pos):
        """The fused form's five calls as one library call (the same kernels, the same results): the calls' own
        preparation, allocations and foreign-function overhead took 40 us of host time per layer, more than the
        launches of a 0.6B layer run for (28 layers and the head: 1850 us a token as calls, 855 this way).
        None for arguments it does not cover: those go call by call."""
        gate_up = self.gate_up._parts
        if gate_up is None or not _ok(x, self.w_in, self.w_post, self.qk_w, cos_sin, k_cache, v_cache):
            return None
        q, k, v, o, down = (p.qtensor for p in (*self.qkv, self.o_proj, self.down_proj))
        gate, up = gate_up[0].qtensor, gate_up[1].qtensor
        h, kv, d, hidden, inter = self.heads, self.kv_heads, self.d, q._k, gate._n
        cache = k_cache.shape
        if (x.dtype is not torch.float32 or x.shape != (1, hidden) or self.w_in.numel() != hidden or self.w_post.numel() != hidden
                or self.qk_w.numel() != 2 * d or cos_sin.numel() != d or len(cache) != 4 or cache[0] != 1 or cache[1] != kv
                or cache[3] != d or v_cache.shape != cache):
            return None
        for w, n, cols in ((q, h * d, hidden), (k, kv * d, hidden), (v, kv * d, hidden), (o, hidden, h * d), (gate, inter, hidden),
                           (up, inter, hidden), (down, hidden, inter)):
            if w._n != n or w._k != cols or w._e != 1:
                return None
        floats = sum(-(-n // 128) * 128 for n in (h * d, kv * d, kv * d, h * d, hidden, inter))
        workspace, y = x.new_empty(floats), x.new_empty((1, hidden))
        check(lib().izwi_qmm_decode_layer_f32(q._h, k._h, v._h, o._h, gate._h, up._h, down._h, x.data_ptr(), self.w_in.data_ptr(),
                                              self.w_post.data_ptr(), self.qk_w.data_ptr(), cos_sin.data_ptr(), h, kv, d, self.eps,
                                              k_cache.data_ptr(), v_cache.data_ptr(), cache[2], pos, workspace.data_ptr(),
                                              4 * floats, y.data_ptr(), _stream_ptr(x)))
        return y
