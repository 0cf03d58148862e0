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

from .capi import ERR_INVALID, check, lib
from .decode_ops import (decode_attention_step, qk_norm_rope_append, try_fused_decode_gqa_attention_with_kv_len, try_fused_qk_rms_norm,
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
        if gate_up is None:
            return None
        # (written out: every attribute and call here is paid once per layer and token; weights that do not fit together and a position
        # outside the caches are refused by the library before it launches anything, and then go call by call like everything else)
        w_in, w_post, qk_w = self.w_in, self.w_post, self.qk_w
        device = x.get_device()
        for t in (x, w_in, w_post, qk_w, cos_sin, k_cache, v_cache):
            if t.dtype is not torch.float32 or t.get_device() != device or not t.is_contiguous():
                return None
        qkv, h, kv, d = self.qkv, self.heads, self.kv_heads, self.d
        q, gate = qkv[0].qtensor, gate_up[0].qtensor
        hidden, cache = q._k, k_cache.shape
        if (device < 0 or x.shape != (1, hidden) or w_in.numel() != hidden or w_post.numel() != hidden or qk_w.numel() != 2 * d
                or cos_sin.numel() != d or len(cache) != 4 or cache[0] != 1 or cache[1] != kv or cache[3] != d or v_cache.shape != cache):
            return None
        floats = 2 * (h * d + 127 & -128) + 2 * (kv * d + 127 & -128) + (hidden + 127 & -128) + (gate._n + 127 & -128)
        workspace, y = x.new_empty(floats), x.new_empty((1, hidden))
        rc = lib().izwi_qmm_decode_layer_f32(q._h, qkv[1].qtensor._h, qkv[2].qtensor._h, self.o_proj.qtensor._h, gate._h,
                                             gate_up[1].qtensor._h, self.down_proj.qtensor._h, x.data_ptr(), w_in.data_ptr(),
                                             w_post.data_ptr(), qk_w.data_ptr(), cos_sin.data_ptr(), h, kv, d, self.eps,
                                             k_cache.data_ptr(), v_cache.data_ptr(), cache[2], pos, workspace.data_ptr(),
                                             4 * floats, y.data_ptr(), _stream_ptr(x))
        if rc == ERR_INVALID:
            return None
        check(rc)
        return y
