"""W8A16 Llama-3 module tree (interface of src/model_quantized.py).

Same composition as src/model.py with W8A16Linear for the seven per-layer
projections; embedding, norms and lm_head stay in the activation dtype
(src/model_quantized.py:137-142).  ``build_random_quantized`` makes the seeded
random-init model of the W8A16 decode benchmark: bf16 master weights drawn on
the device, quantised with quantize_weight_symmetric_per_channel.

Single-token decode (query length 1, up to 16 rows) runs each block through
the fused decode-layer kernels (src/decode_layer.py): six launches per layer
with the same rounding points as the op-by-op composition.  Prefill-sized
inputs keep the composition but fuse its GEMMs: wq|wk|wv in one launch
(QuantizedAttention.qkv), silu(w1(x)) * w3(x) in one launch
(QuantizedFeedForward), and the block's residual adds in the wo / w2
epilogues; other shapes run op by op.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _hooks

from . import decode_layer, quant_linear
from .flash_decode import flash_decode
from .model import Attention, FeedForward, Llama3, TransformerBlock
from .quant_linear import W8A16Linear
from .quant_utils import quantize_weight_symmetric_per_channel


def _no_hooks(*modules) -> bool:
    """Whether a call of these modules is only their class's forward: no forward
    (pre-)hook, their own or a global one, and no forward set on the instance."""
    if _hooks._global_forward_hooks or _hooks._global_forward_pre_hooks:
        return False
    for m in modules:
        if m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__:
            return False
    return True


def _plain(*lins) -> bool:
    """Whether projections up to chat-prompt size may run on their weights in one launch:
    W8A16Linear modules whose call nothing observes or replaces.  (The decode step of
    the block and prefill-sized GEMMs take the weights without this look.)"""
    for m in lins:
        if type(m).forward is not W8A16Linear.forward:
            return False
    return _no_hooks(*lins)


class QuantizedFeedForward(FeedForward):
    def __init__(self, dim: int, hidden_dim: int, linear=W8A16Linear):
        super().__init__(dim, hidden_dim, linear)

    def forward(self, x, *, residual=None):
        """silu(w1(x)) * w3(x) in one launch (the same rounding points, neither
        projection written out): up to 16 rows in the decode projection
        kernels, prefill-sized inputs in the large GEMM when its tiles fill the
        GPU and in the small-M GEMM otherwise; other sizes, and below the large
        GEMM's sizes projections that are not ``_plain``, take the op chain of
        src/model.py:23."""
        x2 = x.reshape(-1, x.shape[-1])
        w1, w3 = _children(self, "w1", "w3")
        plain = _plain(w1, w3)
        if (plain and x2.shape[0] <= 16 and w1.weight.shape == w3.weight.shape
                and _rows_fusable(x2, w1, swiglu=True) and _rows_fusable(x2, w3)):
            torch.cuda.nvtx.range_push("FFN")
            h = decode_layer.linear_fused(x2, w1, lin_b=w3)
            out = self.down(h.view(*x.shape[:-1], w1.out_features), residual)
            torch.cuda.nvtx.range_pop()
            return out
        if quant_linear.swiglu_worth(x2.shape[0], x2.shape[1], w1.out_features, x.device):
            torch.cuda.nvtx.range_push("FFN")
            h = quant_linear.w8a16_gemm_swiglu(x2, w1.weight, w1.scales, w3.weight, w3.scales)
        elif plain and quant_linear.small_gemm_fuses(x2, mats := _pairs(w1, w3)):
            torch.cuda.nvtx.range_push("FFN")
            h = quant_linear.w8a16_small_gemm(x2, mats, swiglu=True)[0]
        else:
            return super().forward(x, residual=residual)
        out = self.down(h.view(*x.shape[:-1], w1.out_features), residual)
        torch.cuda.nvtx.range_pop()
        return out

    def down(self, h, residual=None):
        return _project_residual(*_children(self, "w2"), h, residual)


def _pairs(*lins):
    return [decode_layer.raw_weights(m) for m in lins]


def _children(module, *names):
    """Submodules by name, from the module's own table where they are in it."""
    own = module._modules
    return [own[n] if n in own else getattr(module, n) for n in names]


def _rows_fusable(x2, lin, *, swiglu=False) -> bool:
    """Whether the decode projection kernels take rows x2 [M <= 16, K] through `lin`
    (whose weight has the rows it names: outputs and residual are sized by them)."""
    M, K = x2.shape
    if not 1 <= M <= 16:
        return False
    pair = decode_layer.weights_of(lin)
    return (pair[0].size(0) == lin.out_features
            and decode_layer.supported(M, K, x2.dtype, pair, swiglu=swiglu)
            and decode_layer.aligned(x2))


def _project_residual(lin, h, residual):
    """lin(h) + residual with the add in the epilogue of the decode projection
    (up to 16 rows) or of the GEMM (the same roundings as the separate ops);
    otherwise the two ops."""
    if residual is None:
        return lin(h)
    h2 = h.reshape(-1, h.shape[-1])
    rows = h2.shape[0]
    # below GEMM_MIN_ROWS any projection and any residual that `residual + out` takes are
    # served: the fused forms when the residual has h's dtype and the output's shape,
    # else the two ops
    plain = (residual.dtype == h.dtype and residual.device == h.device and _plain(lin)
             and residual.shape == (*h.shape[:-1], lin.out_features))
    if plain and _rows_fusable(h2, lin):
        res2 = residual.reshape(-1, lin.out_features)
        if res2.stride(1) == 1:
            return decode_layer.linear_fused(h2, lin, residual=res2).view(residual.shape)
    gemm = quant_linear.gemm_supported(rows, h2.shape[1])
    pair = decode_layer.raw_weights(lin) if gemm or plain else None
    small = pair is not None and quant_linear.small_gemm_worth(h2, pair[0])
    if not (small or gemm):
        return residual + lin(h)
    res2 = residual.reshape(-1, lin.out_features)
    if small:
        if not gemm:
            res2 = res2.contiguous()
        y = quant_linear.w8a16_small_gemm(h2, [pair], residual=res2)[0]
        return y.view(*h.shape[:-1], lin.out_features)
    y = quant_linear.w8a16_gemm_residual(h2, *pair, res2)
    return y.view(*h.shape[:-1], lin.out_features)


class QuantizedAttention(Attention):
    def __init__(self, args, linear=W8A16Linear):
        super().__init__(args, linear)

    def out_proj(self, output, residual=None):
        return _project_residual(*_children(self, "wo"), output, residual)

    def qkv(self, x):
        """wq, wk and wv in one launch: of the large GEMM (bitwise the three
        separate GEMMs without a K split) when their tiles together fill the
        GPU, else of the small-M GEMM; sizes neither takes, and modules that are
        not ``_plain`` at the small-M GEMM's, run one W8A16Linear call each."""
        x2 = x.reshape(-1, x.shape[-1])
        mats = _children(self, "wq", "wk", "wv")
        if quant_linear.gemm_multi_worth(x2.shape[0], x2.shape[1],
                                         [m.out_features for m in mats], x.device):
            ys = quant_linear.w8a16_gemm_multi(x2, _pairs(*mats))
        elif _plain(*mats) and quant_linear.small_gemm_fuses(x2, pairs := _pairs(*mats)):
            ys = quant_linear.w8a16_small_gemm(x2, pairs)
        else:
            return super().qkv(x)
        return tuple(y.reshape(*x.shape[:-1], m.out_features) for y, m in zip(ys, mats))


class QuantizedTransformerBlock(TransformerBlock):
    #: run single-token decode through the fused decode-layer kernels
    fused_decode = True
    #: prefill-sized inputs: q|k|v in one GEMM launch, wo / w2 with the
    #: residual add in their epilogues, silu(w1) * w3 in one launch
    attention_cls = QuantizedAttention
    feed_forward_cls = QuantizedFeedForward

    def __init__(self, args, linear=W8A16Linear):
        super().__init__(args, W8A16Linear)

    def _fused_weights(self, x, rope_cos, rope_sin, kv_cache, layer_idx, positions,
                       rope_by_position, start_pos):
        """The block's weights (``decode_layer.weights_of`` pairs of wq, wk, wv, wo,
        w1, w3, w2), its two norms, and whether the QKV and the SwiGLU projection
        normalise their rows themselves, if the fused decode-layer kernels take this call, else None.  Rows
        that need a launch of their own for a norm are taken only at a position inside
        the cache and where no module's call is observed or replaced."""
        if not self.fused_decode or kv_cache is None or layer_idx is None or x.shape[1] != 1:
            return None
        if positions is not None and not rope_by_position:
            return None  # per-step sliced tables at a device position: op chain
        attn, ff = self.attention, self.feed_forward
        B, _, dim = x.shape
        dt, sup = x.dtype, decode_layer.supported
        if (B > kv_cache.max_batch_size or kv_cache.k.dtype != dt
                or rope_cos.dtype != dt or attn.head_dim % 16 != 0 or not x.is_contiguous()
                or not decode_layer.aligned(x.view(B, dim))):
            return None
        kv, rope = kv_cache.k.stride(), rope_cos.stride()
        if (rope[1] != 1 or rope != rope_sin.stride() or rope_sin.dtype != dt
                or rope_sin.size(0) != rope_cos.size(0)
                or kv[4] != 1 or kv != kv_cache.v.stride() or kv_cache.v.dtype != dt):
            return None  # the kernels take one set of strides for each pair
        lins = (*_children(attn, "wq", "wk", "wv", "wo"), *_children(ff, "w1", "w3", "w2"))
        norms = _children(self, "attention_norm", "ffn_norm")
        wq, wk, wv, wo, w1, w3, w2 = ws = tuple(map(decode_layer.weights_of, lins))
        n_q, n_kv = attn.n_heads * attn.head_dim, attn.n_kv_heads * attn.head_dim
        # (rows first: the kernels read as many as the heads and the residual have)
        ok = (wq[0].size(0) == n_q and wk[0].size(0) == wv[0].size(0) == n_kv
              and wo[0].size(0) == w2[0].size(0) == dim
              and sup(B, dim, dt, wq) and sup(B, dim, dt, wk) and sup(B, dim, dt, wv)
              and sup(B, n_q, dt, wo)
              and sup(B, dim, dt, w1, swiglu=True) and sup(B, dim, dt, w3)
              and sup(B, w1[0].size(0), dt, w2))
        if not ok:
            return None
        prologue = (decode_layer.norm_supported(B, dim, dt, norms[0].weight),
                    decode_layer.norm_supported(B, dim, dt, norms[1].weight))
        # past the prologue the op chain served (and at a position outside the cache
        # refused) these rows: it still does where a module's call is observed
        if not (prologue[0] and prologue[1]) and not (
                (positions is not None or 0 <= int(start_pos) < kv_cache.k.size(3))
                and _plain(*lins) and _no_hooks(attn, ff, *norms)):
            return None
        return ws, norms, prologue

    def forward(self, x, rope_cos, rope_sin, layer_idx=None, start_pos=0, kv_cache=None,
                use_cuda_graph=False, scatter_positions=None, decode_attn_mask=None, **ext):
        positions = scatter_positions if (use_cuda_graph and scatter_positions is not None) else None
        by_pos = bool(ext.get("rope_by_position", False))
        fused = self._fused_weights(x, rope_cos, rope_sin, kv_cache, layer_idx, positions,
                                    by_pos, start_pos)
        if fused is None:
            return super().forward(x, rope_cos, rope_sin, layer_idx=layer_idx, start_pos=start_pos,
                                   kv_cache=kv_cache, use_cuda_graph=use_cuda_graph,
                                   scatter_positions=scatter_positions,
                                   decode_attn_mask=decode_attn_mask, **ext)
        ws, (norm, ffn_norm), (qkv_norms, ffn_norms) = fused
        wo, w1, w3, w2 = ws[3:]
        B, _, dim = x.shape
        x2 = x.view(B, dim)
        if positions is not None:  # graph path: device position, full-table RoPE rows
            pos, row0 = positions, 0
            if pos.dtype != torch.int64 or pos.device != x.device:
                pos = pos.to(device=x.device, dtype=torch.int64)
        else:
            p = int(start_pos)
            table = getattr(kv_cache, "_slot_numbers", None)
            if (isinstance(table, torch.Tensor) and table.dtype == torch.int64 and table.dim() == 1
                    and 0 <= p < table.shape[0] and table.device == x.device):
                pos = table[p:p + 1]
            else:
                pos = torch.full((1,), p, dtype=torch.int64, device=x.device)
            row0 = 0 if by_pos else p
        h, nw = (x2, norm.weight) if qkv_norms else (norm(x2), None)
        q = decode_layer.qkv_rope_append(h, self.attention, nw, norm.eps, rope_cos, rope_sin,
                                         row0, pos, kv_cache, layer_idx, weights=ws[:3])
        ck, cv = kv_cache.k[layer_idx, :B], kv_cache.v[layer_idx, :B]
        if positions is None:
            ck, cv = ck[:, :, :int(start_pos) + 1], cv[:, :, :int(start_pos) + 1]
        o = flash_decode(q, ck, cv, mask=decode_attn_mask, seq_lens=ext.get("seq_lens"))
        h = decode_layer.linear_fused(o.view(B, -1), wo, residual=x2)
        n, nw = (h, ffn_norm.weight) if ffn_norms else (ffn_norm(h), None)
        g = decode_layer.linear_fused(n, w1, norm_weight=nw, eps=ffn_norm.eps, lin_b=w3)
        y = decode_layer.linear_fused(g, w2, residual=h)
        return y.view(B, 1, dim)


class Llama3Quantized(Llama3):
    block_cls = QuantizedTransformerBlock
    linear_cls = W8A16Linear


_QUANT_NAMES = ("attention.wq", "attention.wk", "attention.wv", "attention.wo",
                "feed_forward.w1", "feed_forward.w2", "feed_forward.w3")


@torch.no_grad()
def build_random_quantized(args, seed: int = 0, dtype=torch.bfloat16, device="cuda") -> Llama3Quantized:
    """Seeded random-init W8A16 model on `device`.

    Master weights: linears ~ U(-1/sqrt(in), 1/sqrt(in)) (nn.Linear's default
    range), embedding ~ N(0, 1), norms = 1, all in `dtype`; each per-layer
    linear is then quantised with the symmetric per-channel int8 recipe.
    """
    g = torch.Generator(device=device).manual_seed(seed)
    with torch.device("meta"):
        model = Llama3Quantized(args)
    model = model.to_empty(device=device)
    model.tok_embeddings.weight.data = torch.randn(
        model.tok_embeddings.weight.shape, generator=g, device=device, dtype=torch.float32).to(dtype)
    bound = 1.0 / (args.dim ** 0.5)
    model.output.weight.data = ((torch.rand(model.output.weight.shape, generator=g, device=device,
                                            dtype=torch.float32) * 2 - 1) * bound).to(dtype)
    for layer in model.layers:
        for name in _QUANT_NAMES:
            mod = layer.get_submodule(name)
            b = 1.0 / (mod.in_features ** 0.5)
            w = ((torch.rand((mod.out_features, mod.in_features), generator=g, device=device,
                             dtype=torch.float32) * 2 - 1) * b).to(dtype)
            q, s = quantize_weight_symmetric_per_channel(w)
            mod.weight.data = q
            mod.scales.data = s
        layer.attention_norm.weight.data = torch.ones(args.dim, device=device, dtype=dtype)
        layer.ffn_norm.weight.data = torch.ones(args.dim, device=device, dtype=dtype)
    model.norm.weight.data = torch.ones(args.dim, device=device, dtype=dtype)
    return model.eval()
