"""GPU parity of the fused W8A16 decode-layer kernels (mi_w8a16_linear_fused,
mi_w8a16_qkv_rope_append) against the CPU oracle's op-by-op composition
(rmsnorm -> w8a16 -> RoPE / residual / silu*mul) and against the engine's own
unfused GPU chain.  bf16 outputs within 2e-2 of the output scale (the W8A16
bar used for the unfused GEMV); the fused and unfused GPU chains differ only in
fp32 summation order, so they agree to a bf16 rounding step (1e-2 of scale).
"""
import pytest
import torch

from helpers import max_abs, randn
from oracle import quant as oq
from oracle import rope as orope

pytestmark = pytest.mark.gpu


def _linear(dev, K, N, dtype, seed):
    from src.quant_linear import W8A16Linear
    from src.quant_utils import quantize_weight_symmetric_per_channel
    w = randn((N, K), seed, torch.float32, dev, scale=K ** -0.5)
    q, s = quantize_weight_symmetric_per_channel(w.to(dtype))
    lin = W8A16Linear(K, N).to(dev)
    lin.weight.data = q
    lin.scales.data = s.to(dtype)
    return lin


def _close(a, b, tol):
    scale = float(b.float().abs().max()) + 1e-6
    assert max_abs(a, b) < tol * scale, (max_abs(a, b), scale)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(1, 512, 384), (3, 2048, 512), (8, 2048, 2048), (16, 1024, 256),
                                   (8, 8192, 2048), (12, 2048, 4096), (5, 3072, 600),
                                   (7, 1024, 100), (2, 4096, 36),
                                   # 9..16 rows: 8-row tiles up to 128 tiles of 16, then 16-row
                                   (9, 512, 7), (11, 2048, 100), (16, 1536, 2041), (13, 1024, 2048),
                                   (10, 4096, 2049), (9, 6144, 1020), (16, 8192, 2048)])
@pytest.mark.parametrize("norm", [False, True])
def test_linear_store_and_residual(dev, dtype, M, K, N, norm):
    if norm and (M * K * 2 > 64 * 1024 or (M > 8 and K > 2048)):
        pytest.skip("the RMSNorm prologue stages at most 64 KB of rows (K <= 2048 above 8 rows)")
    from src import decode_layer
    from src.rms_norm import rmsnorm_triton
    lin = _linear(dev, K, N, dtype, 1)
    x = randn((M, K), 2, dtype, dev)
    nw = (1.0 + 0.1 * randn((K,), 3, torch.float32)).to(dtype).to(dev) if norm else None
    res = randn((M, N), 4, dtype, dev)
    y = decode_layer.linear_fused(x, lin, norm_weight=nw, eps=1e-5)
    yr = decode_layer.linear_fused(x, lin, norm_weight=nw, eps=1e-5, residual=res)
    a = oq.rmsnorm(x, nw, 1e-5) if norm else x.cpu()
    ref = oq.w8a16(a, lin.weight, lin.scales)
    _close(y, ref, 2e-2)
    _close(yr, (res.cpu().float() + ref.float()).to(dtype), 2e-2)
    # the unfused GPU chain (RMSNorm kernel, GEMV kernel, torch add)
    from src.quant_linear import w8a16_gemv_launch
    un = w8a16_gemv_launch(rmsnorm_triton(x, nw, 1e-5) if norm else x, lin.weight, lin.scales)
    _close(y, un, 1e-2)
    _close(yr, res + un, 1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 5, 8])
def test_swiglu_with_norm(dev, dtype, M):
    from src import decode_layer
    from src.rms_norm import rmsnorm_triton
    K, N = 2048, 1024
    w1, w3 = _linear(dev, K, N, dtype, 5), _linear(dev, K, N, dtype, 6)
    x = randn((M, K), 7, dtype, dev, scale=3.0)
    nw = (1.0 + 0.1 * randn((K,), 8, torch.float32)).to(dtype).to(dev)
    y = decode_layer.linear_fused(x, w1, norm_weight=nw, eps=1e-5, lin_b=w3)
    a = oq.rmsnorm(x, nw, 1e-5)
    g = oq.w8a16(a, w1.weight, w1.scales).float()
    ref = ((g * torch.sigmoid(g)).to(dtype).float() * oq.w8a16(a, w3.weight, w3.scales).float()).to(dtype)
    _close(y, ref, 2e-2)
    xn = rmsnorm_triton(x, nw, 1e-5)
    _close(y, torch.nn.functional.silu(w1(xn)) * w3(xn), 1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [(9, 2048, 8192), (16, 2048, 8192), (11, 1024, 4250), (16, 512, 4100)])
def test_rows_gemv_norm_with_two_tiles(dev, dtype, M, K, N):
    """9..16 rows with the RMSNorm prologue and two tiles per block (more than 256
    tiles), an odd last tile among them: every epilogue."""
    from src import decode_layer
    from src.quant_linear import w8a16_gemv_launch
    from src.rms_norm import rmsnorm_triton
    w1, w3 = _linear(dev, K, N, dtype, 55), _linear(dev, K, N, dtype, 56)
    x, res = randn((M, K), 57, dtype, dev, scale=3.0), randn((M, N), 58, dtype, dev)
    nw = (1.0 + 0.1 * randn((K,), 59, torch.float32)).to(dtype).to(dev)
    a, xn = oq.rmsnorm(x, nw, 1e-5), rmsnorm_triton(x, nw, 1e-5)
    ref = oq.w8a16(a, w1.weight, w1.scales)
    un, un3 = (w8a16_gemv_launch(xn, w.weight, w.scales) for w in (w1, w3))
    y = decode_layer.linear_fused(x, w1, norm_weight=nw, eps=1e-5)
    _close(y, ref, 2e-2)
    _close(y, un, 1e-2)
    yr = decode_layer.linear_fused(x, w1, norm_weight=nw, eps=1e-5, residual=res)
    _close(yr, (res.cpu().float() + ref.float()).to(dtype), 2e-2)
    _close(yr, res + un, 1e-2)
    g = decode_layer.linear_fused(x, w1, norm_weight=nw, eps=1e-5, lin_b=w3)
    _close(g, torch.nn.functional.silu(ref.float()) * oq.w8a16(a, w3.weight, w3.scales).float(), 2e-2)
    _close(g, torch.nn.functional.silu(un) * un3, 1e-2)


class _Attn:
    def __init__(self, dev, dim, Hq, Hkv, D, dtype):
        self.n_heads, self.n_kv_heads, self.head_dim = Hq, Hkv, D
        self.wq = _linear(dev, dim, Hq * D, dtype, 11)
        self.wk = _linear(dev, dim, Hkv * D, dtype, 12)
        self.wv = _linear(dev, dim, Hkv * D, dtype, 13)


class _Cache:
    def __init__(self, dev, L, MB, Hkv, T, D, dtype):
        self.k = randn((L, MB, Hkv, T, D), 21, dtype, dev)
        self.v = randn((L, MB, Hkv, T, D), 22, dtype, dev)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,Hq,Hkv,D", [(8, 32, 8, 64), (3, 24, 8, 128), (1, 4, 1, 64), (16, 8, 2, 32)])
@pytest.mark.parametrize("by_position", [True, False])
def test_qkv_rope_append(dev, dtype, M, Hq, Hkv, D, by_position):
    from src import decode_layer
    from src.rope import DeviceRopeTable, apply_rotary
    dim, T, L, layer, p = 512, 128, 2, 1, 77
    attn = _Attn(dev, dim, Hq, Hkv, D, dtype)
    cache = _Cache(dev, L, M + 1, Hkv, T, D, dtype)
    k0, v0 = cache.k.clone(), cache.v.clone()
    x = randn((M, dim), 31, dtype, dev)
    nw = (1.0 + 0.1 * randn((dim,), 32, torch.float32)).to(dtype).to(dev)
    fc = orope.freqs_cis(D, T, 500000.0)
    table = DeviceRopeTable(fc, dtype, dev)
    cos, sin = (table.cos, table.sin) if by_position else table.rows(p, 1)
    row0 = 0 if by_position else p
    pos = torch.full((1,), p, dtype=torch.int64, device=dev)
    q = decode_layer.qkv_rope_append(x, attn, nw, 1e-5, cos, sin, row0, pos, cache, layer)
    # oracle: rmsnorm -> projections (rounded) -> rotate-half at row p
    a = oq.rmsnorm(x, nw, 1e-5)
    oc, os_ = orope.cos_sin(fc[p:p + 1], dtype)
    rq = orope.rotate(oq.w8a16(a, attn.wq.weight, attn.wq.scales).view(M, Hq, 1, D), oc, os_)
    rk = orope.rotate(oq.w8a16(a, attn.wk.weight, attn.wk.scales).view(M, Hkv, 1, D), oc, os_)
    rv = oq.w8a16(a, attn.wv.weight, attn.wv.scales).view(M, Hkv, D)
    assert q.shape == (M, Hq, 1, D)
    _close(q, rq, 2e-2)
    _close(cache.k[layer, :M, :, p], rk[:, :, 0], 2e-2)
    _close(cache.v[layer, :M, :, p], rv, 2e-2)
    # every other slot (other positions, rows >= M, other layers) is untouched
    mask = torch.ones_like(cache.k, dtype=torch.bool)
    mask[layer, :M, :, p] = False
    assert torch.equal(cache.k[mask], k0[mask]) and torch.equal(cache.v[mask], v0[mask])
    # unfused GPU chain: GEMV kernel then the RoPE kernel on the same rounded values
    from src.rms_norm import rmsnorm_triton
    xn = rmsnorm_triton(x, nw, 1e-5)
    uq = apply_rotary(attn.wq(xn).view(M, 1, Hq, D).transpose(1, 2), *table.rows(p, 1))
    _close(q, uq, 1e-2)


@pytest.mark.parametrize("M", [9, 13, 16])
@pytest.mark.parametrize("K,N", [(512, 16), (1536, 4112), (2048, 250), (3072, 4100), (4096, 4112),
                                 (6144, 40), (8192, 4112)])
def test_rows_gemv_widths_and_tile_edges(dev, M, K, N):
    """9..16 rows: every wave split of K, one and two tiles per block (N past
    16 x 256 rows), a last tile and a last pair that are not full; the sums run
    over the same products as the unfused kernel in another order."""
    from src import decode_layer
    from src.quant_linear import w8a16_gemv_launch
    dtype = torch.bfloat16
    lin = _linear(dev, K, N, dtype, 51)
    x, res = randn((M, K), 52, dtype, dev), randn((M, N), 53, dtype, dev)
    y = decode_layer.linear_fused(x, lin)
    un = w8a16_gemv_launch(x, lin.weight, lin.scales)
    _close(y, oq.w8a16(x, lin.weight, lin.scales), 2e-2)
    _close(y, un, 1e-2)
    _close(decode_layer.linear_fused(x, lin, residual=res), res + un, 1e-2)
    if K <= 4096:
        lin3 = _linear(dev, K, N, dtype, 54)
        g = decode_layer.linear_fused(x, lin, lin_b=lin3)
        _close(g, torch.nn.functional.silu(un) * w8a16_gemv_launch(x, lin3.weight, lin3.scales), 1e-2)


@pytest.mark.parametrize("M,dim,Hq,Hkv,D", [(16, 3072, 24, 8, 128), (9, 2048, 32, 8, 64),
                                            (11, 1024, 3, 1, 48)])
def test_block_of_9_to_16_rows_matches_op_chain(dev, M, dim, Hq, Hkv, D, monkeypatch):
    """The fused block at batches above 8 (RMSNorm as its own launch where the
    prologue does not take the size) against its op-by-op form."""
    from src import model_quantized
    from src.config import ModelArgs
    from src.kv_cache import KVCache
    from src.model_quantized import QuantizedTransformerBlock, build_random_quantized
    if dim != Hq * D:      # heads that do not fill dim: not a model shape, keep the QKV kernel only
        from src import decode_layer
        from src.rope import DeviceRopeTable, apply_rotary
        attn = _Attn(dev, dim, Hq, Hkv, D, torch.bfloat16)
        cache = _Cache(dev, 1, M, Hkv, 32, D, torch.bfloat16)
        t = DeviceRopeTable(orope.freqs_cis(D, 32, 500000.0), torch.bfloat16, dev)
        x = randn((M, dim), 61, torch.bfloat16, dev)
        pos = torch.full((1,), 5, dtype=torch.int64, device=dev)
        q = decode_layer.qkv_rope_append(x, attn, None, 0.0, t.cos, t.sin, 0, pos, cache, 0)
        rot = lambda l, h: apply_rotary(l(x).view(M, 1, h, D).transpose(1, 2), *t.rows(5, 1))  # noqa: E731
        _close(q, rot(attn.wq, Hq), 1e-2)
        _close(cache.k[0, :, :, 5], rot(attn.wk, Hkv)[:, :, 0], 1e-2)
        _close(cache.v[0, :, :, 5], attn.wv(x).view(M, Hkv, D), 1e-2)
        return
    args = ModelArgs(dim=dim, n_layers=1, n_heads=Hq, n_kv_heads=Hkv, vocab_size=64, hidden_dim=4096,
                     max_batch_size=M, max_seq_len=64, device=str(dev))
    block = build_random_quantized(args, seed=3, device=str(dev)).layers[0]
    kv = [KVCache(args, dtype=torch.bfloat16) for _ in range(2)]
    kv[0].k.normal_(generator=torch.Generator(device=dev).manual_seed(1))
    kv[0].v.normal_(generator=torch.Generator(device=dev).manual_seed(2))
    kv[1].k.copy_(kv[0].k)
    kv[1].v.copy_(kv[0].v)
    x = randn((M, 1, dim), 62, torch.bfloat16, dev)
    cos, sin = orope.cos_sin(orope.freqs_cis(D, 64, 500000.0)[40:41], torch.bfloat16)
    ys = []
    with torch.no_grad():
        for c, fused in zip(kv, (True, False)):
            monkeypatch.setattr(QuantizedTransformerBlock, "fused_decode", fused)
            if not fused:      # nor the feed-forward's and the residual's fused forms
                monkeypatch.setattr(model_quantized, "_plain", lambda *lins: False)
            ys.append(block(x, cos.to(dev), sin.to(dev), layer_idx=0, start_pos=40, kv_cache=c))
    _close(ys[0], ys[1], 1e-2)
    _close(kv[0].k, kv[1].k, 1e-2)
    _close(kv[0].v, kv[1].v, 1e-2)


@pytest.mark.parametrize("M", [3, 11])
def test_feed_forward_with_strided_scales(dev, M):
    """Scales that are a column of a wider tensor (every second element): the
    fused projections read N consecutive scales, so such a layer is not theirs."""
    from src import decode_layer
    from src.model_quantized import QuantizedFeedForward
    from src.quant_linear import W8A16Linear
    ff = QuantizedFeedForward(512, 1024, W8A16Linear).to(dev)
    for i, name in enumerate(("w1", "w2", "w3")):
        lin = getattr(ff, name)
        setattr(ff, name, _linear(dev, lin.in_features, lin.out_features, torch.bfloat16, 70 + i))
    x = randn((M, 512), 73, torch.bfloat16, dev)
    with torch.no_grad():
        want = ff(x, residual=x)
        for lin in (ff.w1, ff.w2, ff.w3):
            wide = torch.full((lin.out_features, 2), 7.0, device=dev, dtype=torch.bfloat16)
            wide[:, :1] = lin.scales
            lin.scales.data = wide[:, :1]
            assert not decode_layer.supported(M, lin.in_features, torch.bfloat16, lin)
        _close(ff(x, residual=x), want, 1e-2)


def test_feed_forward_rows_2gb_apart(dev):
    """Rows of x (the last position of long sequences, say) or weights that span 2 GB
    and more: past the fused projections' 32-bit offsets, so not theirs, but served."""
    from src import decode_layer
    from src.model_quantized import QuantizedFeedForward
    from src.quant_linear import W8A16Linear
    M, K, row = 9, 512, 1 << 27                       # (M - 1) * row * 2 bytes = 2 GiB
    ff = QuantizedFeedForward(K, 1024, W8A16Linear).to(dev)
    for i, name in enumerate(("w1", "w2", "w3")):
        lin = getattr(ff, name)
        setattr(ff, name, _linear(dev, lin.in_features, lin.out_features, torch.bfloat16, 80 + i))
    near = randn((M, K), 83, torch.bfloat16, dev)
    far = torch.empty((M - 1) * row + K, device=dev, dtype=torch.bfloat16).as_strided((M, K), (row, 1))
    far.copy_(near)
    assert decode_layer.aligned(near) and decode_layer.aligned(far[:-1]) and not decode_layer.aligned(far)
    with torch.no_grad():
        _close(ff(far, residual=far), ff(near, residual=near), 1e-2)
    scales = torch.ones((1 << 20), device=dev, dtype=torch.bfloat16)
    weight = torch.empty((1 << 20, 2048), device=dev, dtype=torch.int8)
    assert not decode_layer.supported(M, 2048, torch.bfloat16, (weight, scales))
    assert decode_layer.supported(M, 2048, torch.bfloat16, (weight[:-1], scales[:-1]))


def _watched_block(dev, dim, M, S):
    """A quantized block, its rope rows, a cache and x [M, S, dim]."""
    from src.config import ModelArgs
    from src.kv_cache import KVCache
    from src.model_quantized import build_random_quantized
    from src.rope import DeviceRopeTable
    args = ModelArgs(dim=dim, n_layers=1, n_heads=dim // 128, n_kv_heads=2, vocab_size=64,
                     hidden_dim=1024, max_batch_size=M, max_seq_len=64, device=str(dev))
    block = build_random_quantized(args, seed=3, device=str(dev)).layers[0]
    rope = DeviceRopeTable(orope.freqs_cis(128, 64, 500000.0), torch.bfloat16, dev).rows(0, S)
    x = randn((M, S, dim), 90, torch.bfloat16, dev)
    return block, rope, KVCache(args, dtype=torch.bfloat16), x


# chat prompts and feed-forwards of up to 16 rows, decode past the RMSNorm prologue
@pytest.mark.parametrize("dim,M,S", [(1024, 2, 4), (1024, 1, 24), (1024, 3, 40), (3072, 9, 1)])
def test_hooks_of_the_projections_fire(dev, dim, M, S):
    """Every projection and norm of a block called at these sizes is called as a
    module where a hook watches it; hooked and plain calls agree.  (From 33 rows wo
    and w2 add the residual in the GEMM, hook or not.)"""
    block, rope, kv, x = _watched_block(dev, dim, M, S)
    names = ("attention.wq", "attention.wk", "attention.wv", "attention.wo", "feed_forward.w1",
             "feed_forward.w2", "feed_forward.w3", "attention_norm", "ffn_norm")
    if M * S >= 33:
        names = tuple(n for n in names if not n.endswith(("wo", "w2")))
    with torch.no_grad():
        want = block(x, *rope, layer_idx=0, start_pos=0, kv_cache=kv)
        fired = []
        handles = [block.get_submodule(n).register_forward_hook(lambda m, i, o, n=n: fired.append(n))
                   for n in names]
        got = block(x, *rope, layer_idx=0, start_pos=0, kv_cache=kv)
        for h in handles:
            h.remove()
        assert sorted(fired) == sorted(names)
        _close(got, want, 1e-2)
        again = block(x, *rope, layer_idx=0, start_pos=0, kv_cache=kv)
        assert torch.equal(again, want) and len(fired) == len(names)


@pytest.mark.parametrize("rows", [3, 12, 24])
def test_replaced_projections_are_called(dev, rows):
    """A projection swapped for another module (one without int8 weights), or with its
    forward replaced on the instance, is called: its weights are not read around it."""
    block, _, _, _ = _watched_block(dev, 1024, 1, 1)
    ff, attn = block.feed_forward, block.attention
    x = randn((rows, 1024), 91, torch.bfloat16, dev)

    class Dense(torch.nn.Module):            # no weight, scales or out_features of its own
        def __init__(self, lin):
            super().__init__()
            self.dense = (lin.weight.float() * lin.scales.float()).to(torch.bfloat16)

        def forward(self, x):
            return x @ self.dense.t()

    with torch.no_grad():
        want = ff(x, residual=x), attn.out_proj(x, x)
        for name in ("w1", "w2", "w3"):
            lin = getattr(ff, name)
            lin.forward = Dense(lin).forward
        attn.wo = Dense(attn.wo)
        ff.w2 = Dense(ff.w2)
        got = ff(x, residual=x), attn.out_proj(x, x)
        for a, b in zip(got, want):
            _close(a, b, 2e-2)
        ff.w1.forward = lambda x: torch.zeros((rows, 1024), device=dev, dtype=x.dtype)
        assert torch.equal(ff(x, residual=x), x)         # silu(0) * w3(x) = 0


# rows of the RMSNorm prologue and past it
@pytest.mark.parametrize("dim,M", [(1024, 3), (3072, 9)])
def test_decode_tables_and_caches_of_other_layouts(dev, dim, M):
    """RoPE tables that are every second column of a wider one, a cache whose V has
    other strides than its K, and a position tensor on the host: the same step."""
    block, (cos, sin), kv, x = _watched_block(dev, dim, M, 1)
    other = _watched_block(dev, dim, M, 1)[2]
    other.v = torch.zeros([other.v.shape[i] for i in (0, 1, 3, 2, 4)], device=dev,
                          dtype=torch.bfloat16).transpose(2, 3)
    wide = [torch.full((1, 128), 9.0, device=dev, dtype=torch.bfloat16) for _ in range(2)]
    for w, t in zip(wide, (cos, sin)):
        w[:, ::2] = t
    full = [t.repeat(64, 1) for t in (cos, sin)]
    with torch.no_grad():
        want = block(x, cos, sin, layer_idx=0, start_pos=7, kv_cache=kv)
        kv.reset()
        got = block(x, wide[0][:, ::2], wide[1][:, ::2], layer_idx=0, start_pos=7, kv_cache=kv)
        _close(got, want, 1e-2)
        _close(block(x, cos, sin, layer_idx=0, start_pos=7, kv_cache=other), want, 1e-2)
        _close(other.k, kv.k, 1e-2)
        _close(other.v, kv.v, 1e-2)
        kv.reset()
        lens = torch.full((M,), 8, dtype=torch.int64, device=dev)
        got = block(x, *full, layer_idx=0, kv_cache=kv, use_cuda_graph=True, rope_by_position=True,
                    scatter_positions=torch.tensor([7]), seq_lens=lens)
        _close(got, want, 1e-2)


def test_decode_past_the_cache_is_refused_past_the_prologue(dev):
    """9 rows of 3072: a host position outside the cache raises, as the op chain does."""
    block, rope, kv, x = _watched_block(dev, 3072, 9, 1)
    with torch.no_grad(), pytest.raises(ValueError, match="capacity"):
        block(x, *rope, layer_idx=0, start_pos=64, kv_cache=kv)
    assert not kv.k.any() and not kv.v.any()


def test_decode_weights_of_other_heads_are_refused(dev):
    """Projections with fewer rows than the heads, or than the residual: refused, not read past."""
    for name, rows in (("wk", 128), ("wo", 512)):
        block, rope, kv, x = _watched_block(dev, 1024, 3, 1)
        lin = getattr(block.attention, name)
        lin.weight.data, lin.scales.data = lin.weight[:rows].clone(), lin.scales[:rows].clone()
        lin.out_features = rows
        with torch.no_grad(), pytest.raises((RuntimeError, ValueError)):
            block(x, *rope, layer_idx=0, start_pos=7, kv_cache=kv)


def test_feed_forward_weights_of_other_sizes_are_refused(dev):
    """A w2 or w1 / w3 with other rows than the module names: refused, and the residual
    is not read by the weight's rows."""
    for names, rows in ((("w2",), 2048), (("w1", "w3"), 512)):
        block, _, _, _ = _watched_block(dev, 1024, 1, 1)
        ff = block.feed_forward
        for name in names:
            lin = getattr(ff, name)
            lin.weight.data = lin.weight.repeat(2, 1)[:rows].clone()
            lin.scales.data = lin.scales.repeat(2, 1)[:rows].clone()
        x = randn((3, 1024), 92, torch.bfloat16, dev)
        with torch.no_grad(), pytest.raises((RuntimeError, ValueError)):
            ff(x, residual=x)


def test_unsupported_shapes_are_rejected(dev):
    """K outside the built set, M > 16: the C side refuses (nothing launched)
    and the model-level predicate routes such calls to the op chain."""
    from src import decode_layer
    lin = _linear(dev, 256, 64, torch.bfloat16, 9)
    x = randn((4, 256), 10, torch.bfloat16, dev)
    assert not decode_layer.supported(4, 256, torch.bfloat16, lin)
    with pytest.raises(NotImplementedError):
        decode_layer.linear_fused(x, lin)
    lin2 = _linear(dev, 512, 64, torch.bfloat16, 9)
    assert not decode_layer.supported(17, 512, torch.bfloat16, lin2)
    # two weight streams (SwiGLU) are built for K <= 4096 only
    lin3 = _linear(dev, 8192, 64, torch.bfloat16, 9)
    x3 = randn((4, 8192), 10, torch.bfloat16, dev)
    assert decode_layer.supported(4, 8192, torch.bfloat16, lin3)
    assert not decode_layer.supported(4, 8192, torch.bfloat16, lin3, swiglu=True)
    with pytest.raises(NotImplementedError):
        decode_layer.linear_fused(x3, lin3, lin_b=lin3)


# (32, 8): 384 tiles, more than the CUs of an MI355X, so the blocks own two tiles each
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (32, 8)])
def test_qkv_position_outside_cache_writes_nothing(dev, Hq, Hkv):
    from src import decode_layer
    from src.rope import DeviceRopeTable
    dtype, M, D, dim, T = torch.bfloat16, 4, 64, 512, 64
    attn = _Attn(dev, dim, Hq, Hkv, D, dtype)
    cache = _Cache(dev, 1, M, Hkv, T, D, dtype)
    k0, v0 = cache.k.clone(), cache.v.clone()
    table = DeviceRopeTable(orope.freqs_cis(D, T, 500000.0), dtype, dev)
    x = randn((M, dim), 41, dtype, dev)
    for p in (T, T + 5):
        pos = torch.full((1,), p, dtype=torch.int64, device=dev)
        q = decode_layer.qkv_rope_append(x, attn, None, 0.0, table.cos, table.sin, 0, pos, cache, 0)
        torch.cuda.synchronize()
        assert torch.isfinite(q.float()).all()
    assert torch.equal(cache.k, k0) and torch.equal(cache.v, v0)


def test_decode_at_a_host_position_trusts_no_attribute_of_the_cache(dev):
    """A cache that keeps something of its own under the name ``positions`` (or no
    table of slot numbers): the fused block still writes slot start_pos."""
    from src.config import ModelArgs
    from src.kv_cache import KVCache
    from src.model_quantized import build_random_quantized
    args = ModelArgs(dim=512, n_layers=1, n_heads=8, n_kv_heads=2, vocab_size=1000, hidden_dim=1024,
                     max_batch_size=2, max_seq_len=32, device=str(dev))
    model = build_random_quantized(args, seed=3, device=str(dev))
    toks = torch.randint(0, args.vocab_size, (2, 1), generator=torch.Generator().manual_seed(6)).to(dev)
    seen = []
    for change in (None, "positions", "no table", "int32 table"):
        kv = KVCache(args, dtype=torch.bfloat16)
        if change == "positions":       # the next free slot of each sequence, say
            kv.positions = torch.zeros(32, dtype=torch.int64, device=dev)
        elif change == "no table":
            del kv._slot_numbers
        elif change == "int32 table":
            kv._slot_numbers = kv._slot_numbers.int()
        with torch.no_grad():
            logits = model(toks, start_pos=5, kv_cache=kv)
        assert kv.k[:, :, :, 5].any() and not kv.k[:, :, :, :5].any() and not kv.k[:, :, :, 6:].any()
        seen.append((logits, kv.k, kv.v))
    for other in seen[1:]:
        assert all(torch.equal(a, b) for a, b in zip(seen[0], other))


def test_fused_decode_step_matches_unfused(dev, monkeypatch):
    """The quantized block's fused single-token path against the op-by-op
    composition of the same model (eager, three decode steps)."""
    from src import model_quantized
    from src.config import ModelArgs
    from src.kv_cache import KVCache
    from src.model_quantized import QuantizedTransformerBlock, build_random_quantized
    args = ModelArgs(dim=512, n_layers=2, n_heads=8, n_kv_heads=2, vocab_size=1000, hidden_dim=1024,
                     max_batch_size=4, max_seq_len=128, device=str(dev))
    model = build_random_quantized(args, seed=3, device=str(dev))
    kv_a, kv_b = KVCache(args, dtype=torch.bfloat16), KVCache(args, dtype=torch.bfloat16)
    toks = torch.randint(0, args.vocab_size, (4, 20), generator=torch.Generator().manual_seed(5)).to(dev)
    with torch.no_grad():
        model(toks, start_pos=0, kv_cache=kv_a)
        kv_b.k.copy_(kv_a.k)
        kv_b.v.copy_(kv_a.v)
        for step in range(3):
            tok = toks[:, step:step + 1]
            la = model(tok, start_pos=20 + step, kv_cache=kv_a)
            with monkeypatch.context() as m:
                m.setattr(QuantizedTransformerBlock, "fused_decode", False)
                m.setattr(model_quantized, "_plain", lambda *lins: False)   # the sub-blocks' fused forms
                lb = model(tok, start_pos=20 + step, kv_cache=kv_b)
            _close(la, lb, 1e-2)
            _close(kv_a.k, kv_b.k, 1e-2)
            _close(kv_a.v, kv_b.v, 1e-2)
