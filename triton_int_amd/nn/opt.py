"""A W8A8 OPT-shaped decoder layer assembled from the int8 modules.

Not part of the reference tree: its modules are the building blocks ("For qkv_proj", "For fc1",
"For fc2 and out_proj", nn/linear.py:19,71,126) and the layer that chains them lives in the
caller (SmoothQuant-style Int8OPTDecoderLayer).  This module is that caller for benchmarks and
end-to-end tests: every heavy step is one of the package's HIP kernels, torch only reshapes.

    hidden fp32 [B,S,H]
      LayerNormQ -> int8                                    (layer_norm_fwd_fused_single_pass_q)
      q,k,v = 3 x W8A8B8O8Linear -> int8, one launch        (linear_group_a8_w8_b8_o8)
      scores = BMM_S8T_S8N_S8T(q, k) -> int8                (bmm_s8t_s8n_s8t)
      probs  = softmax_q(scores, causal) -> int8 [0,127]    (ti_softmax_q)
      ctx    = BMM_S8T_S8N_S8T(probs, v^T) -> int8, written head-merged through output strides
               (with `fused_attention`, the default for 128 or more query positions and for any number of them
               against up to 4096 keys, these three run as one kernel, ti_attention_i8, and scores / probabilities
               never reach memory)
      acc    = W8A8B32O32LinearWithoutScaling(ctx) -> int32 (linear_a8_w8_b32_o32)   out_proj
      resid, h8 = DQ_Add_LayerNorm_Q(hidden, acc)           (ti_dq_add_layernorm_q)
      f8     = W8A8BFP32OFP32_GeLu_Q(h8) -> int8            (GEMM + GELU-quant epilogue)   fc1
      out    = W8A8BFP32OFP32Linear(f8) + resid -> fp32                                  fc2
               (one library call, ti_linear_i8_residual_f32: the GEMM kernel adds the residual)
"""
from __future__ import annotations

import sys

import torch
from torch.nn.modules import module as _torch_module

from .. import _lib as L
from ..kernels.bmm import bmm_s8t_s8n_s8t
from ..kernels.fused import attention_i8, kv_append_i8, softmax_q, transpose_i8
from ..kernels.linear import linear_group_a8_w8_b8_o8, linear_qkv_decode_a8_w8_b8_o8
from . import fused as _fused, linear as _linear
from .fused import DQ_Add_LayerNorm_Q, LayerNormQ, W8A8BFP32OFP32_GeLu_Q
from .linear import W8A8B8O8Linear, W8A8B32O32LinearWithoutScaling, W8A8BFP32OFP32Linear


class W8A8OPTDecoderLayer(torch.nn.Module):
    def __init__(self, hidden=5120, heads=40, ffn=20480, causal=True):
        super().__init__()
        assert hidden % heads == 0
        self.hidden, self.heads, self.head_dim, self.ffn, self.causal = hidden, heads, hidden // heads, ffn, causal
        self.ln1 = LayerNormQ(hidden)
        self.q_proj = W8A8B8O8Linear(hidden, hidden)
        self.k_proj = W8A8B8O8Linear(hidden, hidden)
        self.v_proj = W8A8B8O8Linear(hidden, hidden)
        self.out_proj = W8A8B32O32LinearWithoutScaling(hidden, hidden)
        self.ln2 = DQ_Add_LayerNorm_Q(hidden)
        self.fc1 = W8A8BFP32OFP32_GeLu_Q(hidden, ffn)
        self.fc2 = W8A8BFP32OFP32Linear(ffn, hidden)
        # attention scales: int8 scores = q8(qk_alpha * q.k), probabilities = softmax(scores * score_scale),
        # int8 context = q8(pv_alpha * P.V)
        self.qk_alpha = 1e-3
        self.score_scale = 0.05
        self.pv_alpha = 1.0 / 127.0
        # one-kernel attention for blocks of queries of this size against any number of keys, for shorter ones
        # against up to 4096; the three-launch chain otherwise (too few workgroups for the block kernel)
        self.fused_attention = True
        self.fused_attention_min_queries = 128
        # fc2 and the residual add that follows it as one library call (a traced forward keeps them apart
        # so that the fc2 output can be inspected)
        self.fused_residual = True

    @torch.no_grad()
    def randomize(self, seed=0):
        """Random int8 weights and per-tensor scales drawn uniformly from [1e-3, 1e-2]."""
        g = torch.Generator(device="cpu").manual_seed(seed)

        def s():
            return float(torch.empty(1).uniform_(1e-3, 1e-2, generator=g))

        for lin in (self.q_proj, self.k_proj, self.v_proj, self.out_proj, self.fc1, self.fc2):
            lin.weight = torch.randint(-127, 128, tuple(lin.weight.shape), dtype=torch.int8, generator=g).to(lin.weight.device)
        for lin in (self.q_proj, self.k_proj, self.v_proj):
            lin.bias = torch.randint(-127, 128, (self.hidden,), dtype=torch.int8, generator=g).to(lin.bias.device)
            lin.a = torch.tensor(s() / 10, dtype=torch.float32, device=lin.a.device)
            lin.b = torch.tensor(s(), dtype=torch.float32, device=lin.b.device)
        self.out_proj.bias = torch.randint(-1000, 1000, (self.hidden,), dtype=torch.int32, generator=g).to(self.out_proj.bias.device)
        self.ln2.input_scale = s() / 100
        self.fc1.bias = torch.randn(self.ffn, generator=g).to(self.fc1.bias.device)
        self.fc1.a = torch.tensor(s() / 30, dtype=torch.float32, device=self.fc1.a.device)
        self.fc1.b = torch.tensor(20.0, dtype=torch.float32, device=self.fc1.b.device)
        self.fc2.bias = torch.randn(self.hidden, generator=g).to(self.fc2.bias.device)
        self.fc2.a = torch.tensor(s() / 100, dtype=torch.float32, device=self.fc2.a.device)
        for ln in (self.ln1, self.ln2):
            ln.weight = (torch.randn(self.hidden, generator=g) * 0.1 + 1.0).div(0.05).to(ln.weight.device)
            ln.bias = (torch.randn(self.hidden, generator=g) * 0.1).div(0.05).to(ln.bias.device)
        return self

    def _qkv_pack(self):
        """The three projections' weights, biases and scales stacked for the grouped launch.  Built
        on first use and whenever one of the modules' tensors was replaced or moved; the modules'
        weight / bias are then re-pointed at slices of the pack, so the weights exist once."""
        mods = (self.q_proj, self.k_proj, self.v_proj)
        key = tuple((m.weight.data_ptr(), m.bias.data_ptr(), m.a.data_ptr(), m.b.data_ptr()) for m in mods)
        if getattr(self, "_qkv_key", None) != key:
            H = self.hidden
            w = torch.cat([m.weight for m in mods], dim=0).contiguous()
            bias = torch.cat([m.bias for m in mods], dim=0).contiguous()
            a = torch.stack([m.a.reshape(()) for m in mods]).to(torch.float32).contiguous()
            b = torch.stack([m.b.reshape(()) for m in mods]).to(torch.float32).contiguous()
            for i, m in enumerate(mods):
                m.weight, m.bias = w[i * H:(i + 1) * H], bias[i * H:(i + 1) * H]
                m.a, m.b = a[i], b[i]
            self._qkv = (w, bias, a, b)
            self._qkv_key = tuple((m.weight.data_ptr(), m.bias.data_ptr(), m.a.data_ptr(), m.b.data_ptr()) for m in mods)
        return self._qkv

    def _heads(self, t, B, S):
        # [B,S,H] int8 -> [B*heads, S, D].  One batch: a strided view (the BMM takes row and batch
        # strides, each head's rows stay K-contiguous).  Several batches: a copy.
        if B == 1:
            return t.view(S, self.heads, self.head_dim).transpose(0, 1)
        return t.view(B, S, self.heads, self.head_dim).transpose(1, 2).reshape(B * self.heads, S, self.head_dim)

    def _append(self, k_new, v_new, k_all, vt_all):
        """k_new, v_new int8 [B,S,H] into the last S slots of K [B*heads,T,D] (unless None) and of V^T
        [B*heads,D,T]: one launch for head dimensions that are multiples of 16 and caches whose rows have
        unit stride and one pitch."""
        B, S, H = v_new.shape
        heads, D, T = self.heads, self.head_dim, vt_all.shape[2]
        vs = vt_all.stride()
        if D % 16 == 0 and (k_all is None or k_all.stride(2) == 1) and vs[2] == 1 and (vs[0] == D * vs[1] or B * heads == 1):
            if B * heads <= 32767 or B <= self._at_once():
                kv_append_i8(k_new.view(B * S, H), v_new.view(B * S, H), k_all, vt_all, seqs=B)
                return
            n = self._at_once()
            for b in range(0, B, n):
                hs = slice(b * heads, (b + n) * heads)
                self._append(k_new[b:b + n], v_new[b:b + n], None if k_all is None else k_all[hs], vt_all[hs])
            return
        if k_all is not None:
            k_all[:, T - S:, :] = self._heads(k_new, B, S)
        for b in range(B):
            transpose_i8(v_new[b], out=vt_all[b * heads:(b + 1) * heads].view(H, T)[:, T - S:])

    def _at_once(self):
        """Sequences of one launch: an attention takes up to 65535 heads, an append up to 32767 sequences."""
        return max(1, min(32767, 65535 // self.heads))

    @staticmethod
    def _kernel_takes(k_all, vt_all, T, D):
        """Whether the attention kernel takes caches that lie like this; the three-launch chain takes any."""
        kh, kr, kc = k_all.stride()
        vr, vc = vt_all.stride()[1:]
        return kc == 1 and kr >= D and (k_all.data_ptr() | kh | kr) % 16 == 0 and (vc == 1 or T == 1) and vr >= T

    def forward(self, hidden, kv_cache=None, _trace=None, _mark=None):
        """hidden fp32 [B,S,H].  kv_cache = (K int8 [B*heads, T, D], V^T int8 [B*heads, D, T]) holds the
        T-S earlier positions in its first T-S slots; the S new positions are written into the last S
        slots before attention (decode / chunked prefill).  Returns fp32 [B,S,H].  A dict passed as
        `_trace` receives every intermediate tensor (for stage-by-stage parity tests); a callable
        passed as `_mark` is called with a stage name after that stage's launches (for timing the
        stages in sequence with stream events).

        The ordinary call is one function of the extension module, which makes the launches below from the modules' buffers
        (csrc/host_layer.cpp); what it declines (hooks on a module, other module types, caches that need a copy)
        runs step by step."""
        if _trace is None and _mark is None and self.head_dim == 128 and self.fused_attention:
            out = L.layer_host.decoder_layer(self, hidden, kv_cache, _TYPES, _GLOBAL_HOOKS)
            if out is not None:
                return out
        return self._forward_steps(hidden, kv_cache, _trace, _mark)

    @torch.no_grad()
    def _forward_steps(self, hidden, kv_cache, _trace, _mark):
        mark = _mark if _mark is not None else (lambda name: None)
        B, S, H = hidden.shape
        h8 = self.ln1(hidden)
        mark("ln1_layernorm_q")
        w3, b3, a3, s3 = self._qkv_pack()
        qkv = None
        if kv_cache is not None and B * S <= 16:
            # decode: projections and KV-cache append in one launch
            qkv = linear_qkv_decode_a8_w8_b8_o8(h8.view(B * S, H), w3, b3, a3, s3, kv_cache[0], kv_cache[1], seqs=B)
        appended = qkv is not None
        if appended:
            qkv = qkv.view(B, S, 3 * H)
        else:
            qkv = linear_group_a8_w8_b8_o8(h8, w3, b3, a3, s3, 3)                   # [B,S,3H] int8
        heads, D = self.heads, self.head_dim
        v = qkv[..., 2 * H:]                                                       # [B,S,H] int8, row pitch 3H
        mark("qkv_3x_linear_o8")
        T = S if kv_cache is None else kv_cache[0].shape[1]
        # short blocks of queries against up to 4096 keys run the attention kernel too; a traced
        # forward keeps the three steps of blocks of 17 .. 127 apart so that they can be inspected
        short = T <= 4096 and (S <= 16 or _trace is None)
        fused = (self.fused_attention and (S >= self.fused_attention_min_queries or short) and D == 128 and self.score_scale > 0.0
                 and (kv_cache is None or self._kernel_takes(*kv_cache, T, D)))
        if kv_cache is None:
            # rows of V^T padded to a multiple of 16 bytes: the attention kernel reads them in 16-byte pieces
            vt_all = torch.empty((B * heads, D, (S + 15) // 16 * 16), dtype=torch.int8, device=hidden.device)[:, :, :S]
            k_all = None
        else:
            k_all, vt_all = kv_cache
        if not appended:
            # the new K rows and V^T columns go into the last S slots of the cache
            self._append(qkv[..., H:2 * H], v, k_all, vt_all)
        mark("kv_append_v_transpose")
        ctx = torch.empty((B, S, H), dtype=torch.int8, device=hidden.device)
        q = scores = probs = None
        if not fused or _trace is not None:
            q = self._heads(qkv[..., :H], B, S)
            if k_all is None:
                k_all = self._heads(qkv[..., H:2 * H], B, S)
        if fused:
            # every operand as [B, heads, rows, D] views: all sequences in one launch, as far as one launch goes
            by_head = lambda t: t.view(B, S, heads, D).transpose(1, 2)
            q4, k4 = by_head(qkv[..., :H]), by_head(qkv[..., H:2 * H]) if kv_cache is None else k_all.unflatten(0, (B, heads))
            vt4, out4, causal = vt_all.unflatten(0, (B, heads)), by_head(ctx), S if self.causal else 0
            n = B if B * heads <= 65535 else self._at_once()
            if n == B:
                attention_i8(q4, k4, vt4, self.qk_alpha, self.score_scale, self.pv_alpha, causal_q_len=causal, out=out4)
            else:
                for b in (slice(b, b + n) for b in range(0, B, n)):
                    attention_i8(q4[b], k4[b], vt4[b], self.qk_alpha, self.score_scale, self.pv_alpha, causal_q_len=causal, out=out4[b])
            mark("attention_i8_fused")
        else:
            scores = bmm_s8t_s8n_s8t(q, k_all, self.qk_alpha)                       # [B*heads, S, T] int8
            mark("qk_bmm_o8")
            probs = softmax_q(scores, self.score_scale, causal_q_len=S if self.causal else 0)
            mark("softmax_q")
            # P.V with the head merge folded into the output strides: head h of batch b writes columns
            # h*D .. h*D+D of row (b, s) of a [B,S,H] tensor
            for b in range(B):
                out_view = ctx[b].view(S, heads, D).transpose(0, 1)                # [heads, S, D] strided
                bmm_s8t_s8n_s8t(probs[b * heads:(b + 1) * heads], vt_all[b * heads:(b + 1) * heads],
                                self.pv_alpha, out=out_view)
            mark("pv_bmm_o8")
        acc = self.out_proj(ctx)                                                    # int32 [B,S,H]
        mark("out_proj_linear_o32")
        resid, h8b = self.ln2(hidden, acc)
        mark("ln2_dq_add_layernorm_q")
        f8 = self.fc1(h8b)
        mark("fc1_linear_gelu_q")
        if self.fused_residual and _trace is None:
            y = None
            out = self.fc2.forward_add(f8, resid)   # one launch: the GEMM kernel adds the residual as it stores
            mark("fc2_linear_f32_plus_residual")
        else:
            y = self.fc2(f8)
            mark("fc2_linear_f32")
            out = y + resid
            mark("residual_add")
        if _trace is not None:
            _trace.update(h8=h8, q=q, k_all=k_all, vt_all=vt_all, scores=scores, probs=probs, ctx=ctx, acc=acc,
                          resid=resid, h8b=h8b, f8=f8, fc2=y, out=out)
        return out


# What the extension module's function stands for: exactly these types, nothing hooked into any module, and the methods and launchers that
# the steps above look up as they are here
def _found(where, *names):
    tables = [vars(c) for c in where.__mro__] if isinstance(where, type) else [vars(where)]
    return tuple((where if isinstance(where, type) else vars(where), n, next(t[n] for t in tables if n in t)) for n in names)


_CALL = ("__call__", "_call_impl", "_compiled_call_impl", "__getattr__", "forward")
_UNCHANGED = (*_found(W8A8OPTDecoderLayer, "__getattr__", "_forward_steps", "_qkv_pack", "_heads", "_append", "_at_once", "_kernel_takes"),
              *_found(LayerNormQ, *_CALL), *_found(DQ_Add_LayerNorm_Q, *_CALL), *_found(W8A8B8O8Linear, "__getattr__"),
              *_found(W8A8B32O32LinearWithoutScaling, *_CALL, "_launch"), *_found(W8A8BFP32OFP32_GeLu_Q, *_CALL, "_launch"),
              *_found(W8A8BFP32OFP32Linear, "__getattr__", "forward_add"),
              *_found(sys.modules[__name__], "linear_qkv_decode_a8_w8_b8_o8", "linear_group_a8_w8_b8_o8", "kv_append_i8", "attention_i8"),
              *_found(_fused, "layer_norm_fwd_fused_single_pass_q", "dq_add_layernorm_q_cpp", "linear_a8_w8_bfp32_ofp32_GeLu_Q"),
              *_found(_linear, "linear_a8_w8_b32_o32", "linear_a8_w8_bfp32_ofp32_residual"))
_TYPES = (W8A8OPTDecoderLayer, LayerNormQ, W8A8B8O8Linear, W8A8B8O8Linear, W8A8B8O8Linear, W8A8B32O32LinearWithoutScaling, DQ_Add_LayerNorm_Q,
          W8A8BFP32OFP32_GeLu_Q, W8A8BFP32OFP32Linear, _UNCHANGED)
_GLOBAL_HOOKS = tuple(getattr(_torch_module, name) for name in ("_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks",
                                                                "_global_backward_pre_hooks"))
