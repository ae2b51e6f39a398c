"""GPU parity of the ops around the FC GEMMs: LayerNorm-affine (and its fused next-GEMM
operand), fp16-K/V flash attention, the fp32 GEMM of the tied head, and the graph glue.

Bars:
  * LN-affine vs the oracle (the reference CPU executor's double statistics): every element
    within 2 fp32 ulps of max|y|, and nearly all bit-exact; the fused int8-dot operand equals
    the activation quantizer applied to the kernel's own y, bit for bit.
  * Flash attention vs the oracle attention on fp16-rounded q/k/v: max|o - o_ref| <= 2e-5 *
    max|o_ref| (fp32 softmax; only summation order and the online rescaling differ).
  * fp32 GEMM vs the oracle's sequential fp32 GEMM: <= 1e-5 * max|y|.
  * get_rows / add / strided copy: exact.
"""
import numpy as np
import pytest

import edge_maskgit_amd as ema
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ema.Context(0)
    yield c
    c.close()


def _rel(y, ref):
    return float(np.abs(y - ref).max() / max(np.abs(ref).max(), 1e-30))


# ---- LayerNorm-affine ------------------------------------------------------------------
@pytest.mark.parametrize("rows,D", [(1, 256), (5, 768), (1025, 768), (33, 2048)])
def test_layernorm_vs_oracle(ctx, rows, D):
    print(f"layernorm rows={rows} D={D}", flush=True)
    rng = np.random.default_rng(rows + D)
    x = (rng.standard_normal((rows, D)) * 3 + 0.5).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    b = (0.1 * rng.standard_normal(D)).astype(np.float32)
    ref = oracle.layernorm_affine(x, g, b, 1e-12)
    dX, dG, dB, dY = ctx.upload(x), ctx.upload(g), ctx.upload(b), ctx.alloc(x.nbytes)
    ctx.layernorm_affine(dX, dG, dB, rows, D, 1e-12, dY)
    y = ctx.download(dY, x.shape, np.float32)
    for t in (dX, dG, dB, dY):
        ctx.free(t)
    ulp = np.spacing(np.abs(ref).max())
    assert np.abs(y - ref).max() <= 2 * ulp
    frac = float(np.mean(y.view(np.uint32) == ref.view(np.uint32)))
    print(f"  bit-exact fraction {frac:.5f}")
    assert frac >= 0.99


def test_layernorm_emit_int8_operand(ctx):
    rows, D = 257, 768
    print("layernorm emit int8", flush=True)
    rng = np.random.default_rng(7)
    x = rng.standard_normal((rows, D)).astype(np.float32)
    x[3] = 0.0                                   # constant row: y = beta
    g = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    b = (0.1 * rng.standard_normal(D)).astype(np.float32)
    b[:32] = 0.0
    dX, dG, dB, dY = ctx.upload(x), ctx.upload(g), ctx.upload(b), ctx.alloc(x.nbytes)
    dC, dD, dS = ctx.alloc(rows * D * 2), ctx.alloc(rows * D // 32 * 4), ctx.alloc(rows * D // 32 * 4)
    ctx.layernorm_affine(dX, dG, dB, rows, D, 1e-12, dY, ema.EMIT_INT8, dC, dD, dS)
    y = ctx.download(dY, x.shape, np.float32)
    codes = ctx.download(dC, (rows, D), np.float16)
    dx = ctx.download(dD, (rows, D // 32), np.float32)
    sx = ctx.download(dS, (rows, D // 32), np.int32)
    # the same y without the operand
    ctx.layernorm_affine(dX, dG, dB, rows, D, 1e-12, dY)
    y0 = ctx.download(dY, x.shape, np.float32)
    for t in (dX, dG, dB, dY, dC, dD, dS):
        ctx.free(t)
    assert np.array_equal(y.view(np.uint32), y0.view(np.uint32))
    qx, dx_r, sx_r = oracle.quantize_act_q8(y)
    assert np.array_equal(codes.astype(np.int32), qx.astype(np.int32))
    assert np.array_equal(dx.view(np.uint32), dx_r.view(np.uint32))
    assert np.array_equal(sx, sx_r)


def test_layernorm_emit_deq_operand(ctx):
    rows, D = 65, 768
    print("layernorm emit deq-f16", flush=True)
    rng = np.random.default_rng(8)
    x = rng.standard_normal((rows, D)).astype(np.float32)
    g = np.ones(D, np.float32)
    b = np.zeros(D, np.float32)
    dX, dG, dB, dY = ctx.upload(x), ctx.upload(g), ctx.upload(b), ctx.alloc(x.nbytes)
    dC, dD, dS = ctx.alloc(rows * D * 2), ctx.alloc(rows * D // 32 * 4), ctx.alloc(rows * D // 32 * 4)
    ctx.layernorm_affine(dX, dG, dB, rows, D, 1e-12, dY, ema.EMIT_DEQ_F16, dC, dD, dS)
    y = ctx.download(dY, x.shape, np.float32)
    h = ctx.download(dC, (rows, D), np.float16)
    dx = ctx.download(dD, (rows, D // 32), np.float32)
    ux = ctx.download(dS, (rows, D // 32), np.float32)
    # the block scales and sums are optional: the fp16 operand alone, bit-identical
    dC2, dY2 = ctx.alloc(rows * D * 2), ctx.alloc(x.nbytes)
    ctx.layernorm_affine(dX, dG, dB, rows, D, 1e-12, dY2, ema.EMIT_DEQ_F16, dC2, None, None)
    y2 = ctx.download(dY2, x.shape, np.float32)
    h2 = ctx.download(dC2, (rows, D), np.float16)
    for t in (dX, dG, dB, dY, dC, dD, dS, dC2, dY2):
        ctx.free(t)
    assert np.array_equal(h2.view(np.uint16), h.view(np.uint16))
    assert np.array_equal(y2.view(np.uint32), y.view(np.uint32))
    assert np.array_equal(h, y.astype(np.float16))
    assert np.all(dx == 1.0)
    blk = h.astype(np.float64).reshape(rows, D // 32, 32).sum(-1)
    assert np.abs(ux - blk).max() <= 1e-5 * max(np.abs(blk).max(), 1.0)


# ---- flash attention -------------------------------------------------------------------
def _qkv(rng, D, S, H, B):
    shape = (B * S, H * D)                       # the FC outputs [S*B][H*D] (batch-major rows)
    return [rng.standard_normal(shape).astype(np.float32) for _ in range(3)]


# S <= 272 runs the whole-head kernel (K/V of a head resident in LDS), longer sequences the
# chunked online-softmax kernel
@pytest.mark.parametrize("D,S,H,B", [(48, 1, 2, 1), (48, 16, 2, 1), (48, 17, 2, 1), (48, 64, 3, 2), (48, 65, 2, 1),
                                     (48, 257, 16, 2), (64, 130, 4, 1), (16, 40, 1, 1), (32, 300, 2, 1),
                                     (48, 512, 2, 1), (64, 512, 1, 1), (48, 513, 2, 1), (48, 1025, 1, 1)])
def test_flash_attn_vs_oracle(ctx, D, S, H, B):
    print(f"flash_attn D={D} S={S} H={H} B={B}", flush=True)
    rng = np.random.default_rng(D * S + H + B)
    q, k, v = _qkv(rng, D, S, H, B)
    st = (1, H * D, D, H * D * S)
    scale = 1.0 / np.sqrt(D)
    ref = oracle.attention(q, k, v, st, D, S, H, B, scale, True)
    dq, dk, dv = ctx.upload(q), ctx.upload(k), ctx.upload(v)
    do = ctx.alloc(D * S * H * B * 4)
    ctx.flash_attn_f16kv(dq, dk, dv, st, D, S, H, B, scale, do)
    o = ctx.download(do, (D * S * H * B,), np.float32)
    # merged-head output written directly ({D,S,H,B} -> [S*B][H*D])
    ctx.flash_attn_f16kv(dq, dk, dv, st, D, S, H, B, scale, do, o_strides=(1, H * D, D, H * D * S))
    om = ctx.download(do, (D * S * H * B,), np.float32)
    for t in (dq, dk, dv, do):
        ctx.free(t)
    err = _rel(o, ref)
    print(f"  rel err {err:.2e}")
    assert err <= 2e-5
    assert np.array_equal(om, oracle.merge_heads(o, D, S, H, B))


@pytest.mark.parametrize("D,S,H", [(48, 257, 16), (64, 130, 4), (48, 40, 1)])
def test_flash_attn_split_queries_bit_identical(ctx, D, S, H):
    """with few heads the whole-head kernel spreads a head's query tiles over several
    workgroups; one image alone (split) and the same image repeated 16 times in a batch (at
    H = 16 unsplit) give the same bits"""
    rng = np.random.default_rng(D + S + H)
    q, k, v = _qkv(rng, D, S, H, 1)
    outs = []
    for B in (1, 16):
        qb, kb, vb = (np.ascontiguousarray(np.tile(a, (B, 1))) for a in (q, k, v))
        st = (1, H * D, D, H * D * S)
        dq, dk, dv = ctx.upload(qb), ctx.upload(kb), ctx.upload(vb)
        do = ctx.alloc(D * S * H * B * 4)
        ctx.flash_attn_f16kv(dq, dk, dv, st, D, S, H, B, 1.0 / np.sqrt(D), do)
        outs.append(ctx.download(do, (B, D * S * H), np.float32))
        for t in (dq, dk, dv, do):
            ctx.free(t)
    for b in range(16):
        assert np.array_equal(outs[1][b], outs[0][0])


@pytest.mark.parametrize("S", [257, 600])
def test_flash_attn_o16_is_rounded_output(ctx, S):
    """The fp16-output variant stores exactly the fp32 attention output rounded to fp16."""
    D, H, B = 48, 4, 2
    print(f"flash_attn_o16 S={S}", flush=True)
    rng = np.random.default_rng(S)
    q, k, v = _qkv(rng, D, S, H, B)
    st, ost = (1, H * D, D, H * D * S), (1, H * D, D, H * D * S)
    dq, dk, dv = ctx.upload(q), ctx.upload(k), ctx.upload(v)
    do, dh = ctx.alloc(D * S * H * B * 4), ctx.alloc(D * S * H * B * 2)
    ctx.flash_attn_f16kv(dq, dk, dv, st, D, S, H, B, 0.144, do, o_strides=ost)
    ctx.flash_attn_f16kv_o16(dq, dk, dv, st, D, S, H, B, 0.144, dh, o_strides=ost)
    o = ctx.download(do, (D * S * H * B,), np.float32)
    h = ctx.download(dh, (D * S * H * B,), np.float16)
    for t in (dq, dk, dv, do, dh):
        ctx.free(t)
    assert np.array_equal(h.view(np.uint16), o.astype(np.float16).view(np.uint16))


# The long kernel (S > 272) at the edges of its blocks and chunks: a whole number of 64-key chunks
# and one key past it; a last block of one query (split over the keys), of exactly one wave's
# queries and one more; the 64-query form with two key groups (an odd and an even number of
# chunks) and, from 200 (D = 64: 120) 128-query blocks, the 128-query form; padded rows (q/k/v
# strides 4 elements past the heads); fp16 output; outputs whose rows are not 16-byte aligned.
@pytest.mark.parametrize("D,S,H,B,pad,opad", [
    (48, 273, 3, 1, 0, 0), (48, 576, 2, 1, 0, 0), (48, 577, 2, 1, 4, 0), (48, 592, 2, 2, 0, 0), (48, 593, 2, 1, 0, 1),
    (16, 300, 2, 1, 4, 0), (32, 385, 3, 2, 0, 2), (64, 641, 2, 1, 0, 0), (64, 384, 40, 1, 0, 0), (64, 1025, 14, 1, 4, 1),
    (48, 385, 50, 1, 0, 0), (48, 400, 25, 2, 4, 0), (48, 417, 50, 1, 0, 3), (32, 2049, 12, 1, 0, 0), (16, 513, 40, 1, 0, 0)])
def test_flash_attn_long(ctx, D, S, H, B, pad, opad):
    """against float64 on the fp16-rounded operands: |o - ref| <= 2e-5 max|ref|, the bar of the
    other attention kernels (fp32 sums over S / 64 chunks: about 1e-6)"""
    print(f"flash_attn_long D={D} S={S} H={H} B={B} pad={pad} opad={opad}", flush=True)
    rng = np.random.default_rng(11 * D + S + H)
    E = H * D
    R, RO = 3 * E + pad, E + opad
    wide = rng.standard_normal((B, S, R)).astype(np.float32)
    # scores that grow along the keys move the softmax reference many times
    wide[:, :, E:2 * E] *= np.linspace(0.2, 4.0, S)[None, :, None]
    h = wide[:, :, :3 * E].astype(np.float16).astype(np.float64).reshape(B, S, 3, H, D)
    scale = D ** -0.5
    ref = np.empty((B, S, H, D))
    for b in range(B):
        for i in range(H):
            s = h[b, :, 0, i] @ h[b, :, 1, i].T * scale
            p = np.exp(s - s.max(-1, keepdims=True))
            ref[b, :, i] = p @ h[b, :, 2, i] / p.sum(-1, keepdims=True)
    ref = ref.reshape(B * S, E)
    dw, do, dh = ctx.upload(wide), ctx.alloc(B * S * RO * 4), ctx.alloc(B * S * RO * 2)
    st, ost = (1, R, D, R * S), (1, RO, D, RO * S)
    ctx.flash_attn_f16kv(dw.ptr, dw.ptr + 4 * E, dw.ptr + 8 * E, st, D, S, H, B, scale, do, o_strides=ost)
    ctx.flash_attn_f16kv_o16(dw.ptr, dw.ptr + 4 * E, dw.ptr + 8 * E, st, D, S, H, B, scale, dh, o_strides=ost)
    o = ctx.download(do, (B * S, RO), np.float32)[:, :E]
    o16 = ctx.download(dh, (B * S, RO), np.float16)[:, :E]
    for t in (dw, do, dh):
        ctx.free(t)
    err = _rel(o, ref)
    print(f"  rel err {err:.2e}")
    assert err <= 2e-5
    assert np.array_equal(o16.view(np.uint16), o.astype(np.float16).view(np.uint16))


def test_flash_attn_long_weights_are_rounded_to_nearest(ctx):
    """the softmax weights enter P . V as two fp16 parts rounded to nearest. One key in 32 has a lower
    score s (another for every query) and value 1, the others value 0, so the output follows the
    weight of s alone. RMS of its relative error over 8 heads of queries, with exp2, scale and division
    in fp32: measured 1.43e-7 and 1.15e-7; with truncated parts 1.62e-7 and 1.35e-7"""
    rms = []
    for D, S in ((16, 1024), (48, 640)):
        H, E = 8, 8 * D
        rng = np.random.default_rng(3)
        x = np.zeros((S, 3, H, D), np.float32)
        x[:, 0, :, 0] = -rng.uniform(0.5, 7, (S, H)).astype(np.float16)
        x[::32, 1:, :, 0] = 1.0
        d, do = ctx.upload(x), ctx.alloc(S * E * 4)
        ctx.flash_attn_f16kv(d.ptr, d.ptr + 4 * E, d.ptr + 8 * E, (1, 3 * E, D, 3 * E * S), D, S, H, 1, 1.0, do,
                             o_strides=(1, E, D, E * S))
        o = ctx.download(do, (S, H, D), np.float32)[:, :, 0].astype(np.float64)
        for t in (d, do):
            ctx.free(t)
        p = np.exp(x[:, 0, :, 0].astype(np.float64)) * (S // 32)
        ref = p / (p + S - S // 32)
        rms.append(float(np.sqrt((((o - ref) / ref) ** 2).mean())))
    print("  rms", rms)
    assert rms[0] <= 1.53e-7 and rms[1] <= 1.25e-7


# one image's call takes two key groups side by side, a batch of them one after the other (from 200
# 128-query blocks in the call, 120 at D = 64), an image with as many blocks of its own one group
@pytest.mark.parametrize("D,S,H,B", [(48, 273, 16, 6), (48, 400, 16, 4), (48, 577, 16, 3), (48, 592, 10, 5), (48, 600, 16, 3),
                                     (32, 385, 16, 4), (16, 321, 16, 5), (64, 513, 16, 3), (64, 450, 16, 2), (64, 528, 8, 4),
                                     (48, 1025, 8, 4), (48, 1025, 25, 2)])
def test_flash_attn_long_batch_invariant(ctx, D, S, H, B):
    """an image's output is the same bits alone and in a batch, for fp32 and fp16 outputs and inputs"""
    print(f"flash_attn_long batch D={D} S={S} H={H} B={B}", flush=True)
    rng = np.random.default_rng(D + S + B)
    E = H * D
    x = rng.standard_normal((B, S, 3, E)).astype(np.float32)
    x[:, :, 1] *= np.linspace(0.2, 4.0, S)[None, :, None]       # the softmax reference moves
    st, ost = (1, 3 * E, D, 3 * E * S), (1, E, D, E * S)
    d, d16 = ctx.upload(x), ctx.upload(x.astype(np.float16))
    do, dh, one = ctx.alloc(B * S * E * 4), ctx.alloc(B * S * E * 2), ctx.alloc(S * E * 4)

    def attn(fn, base, elem, n, out, **kw):
        fn(base, base + elem * E, base + 2 * elem * E, st, D, S, H, n, D ** -0.5, *out, **kw)

    attn(ctx.flash_attn_f16kv, d.ptr, 4, B, (do,), o_strides=ost)
    attn(ctx.flash_attn_f16kv_o16, d.ptr, 4, B, (dh,), o_strides=ost)
    o, o16 = ctx.download(do, (B, S, E), np.float32), ctx.download(dh, (B, S, E), np.float16)
    if S <= 512:
        attn(ctx.flash_attn_f16in, d16.ptr, 2, B, (do, None, ost))
        assert np.array_equal(ctx.download(do, (B, S, E), np.float32).view(np.uint32), o.view(np.uint32))
    assert np.array_equal(o16.view(np.uint16), o.astype(np.float16).view(np.uint16))
    for b in (0, B - 1):
        attn(ctx.flash_attn_f16kv, d.ptr + 12 * E * S * b, 4, 1, (one,), o_strides=ost)
        assert np.array_equal(ctx.download(one, (S, E), np.float32).view(np.uint32), o[b].view(np.uint32))
    for t in (d, d16, do, dh, one):
        ctx.free(t)
    # both forms against float64, on one head
    h = x[B - 1].astype(np.float16).astype(np.float64).reshape(S, 3, H, D)[:, :, H - 1]
    sc = h[:, 0] @ h[:, 1].T * D ** -0.5
    p = np.exp(sc - sc.max(-1, keepdims=True))
    assert _rel(o[B - 1].reshape(S, H, D)[:, H - 1], p @ h[:, 2] / p.sum(-1, keepdims=True)) <= 2e-5


# S % 64 = 1, 17, 33, 0 keys in the last chunk, an odd and an even number of chunks for the two key
# groups, and the 128-query form (50 heads); heads interleaved in rows and image after image, so that
# the row after an image's last is the next image's first.
@pytest.mark.parametrize("D,S,H", [(48, 577, 2), (48, 593, 2), (32, 353, 2), (64, 640, 2), (16, 273, 3), (48, 417, 50),
                                   (64, 385, 50)])
def test_flash_attn_long_reads_no_row_past_the_image(ctx, D, S, H):
    """an image's output is the same bits whether the next image's q/k/v are numbers or NaN"""
    print(f"flash_attn_long past the image D={D} S={S} H={H}", flush=True)
    rng = np.random.default_rng(D + S)
    E = H * D
    x = rng.standard_normal((2, S, 3 * E)).astype(np.float32)
    do = ctx.alloc(2 * S * E * 4)
    outs = []
    for fill in (None, np.nan, np.inf):
        if fill is not None:
            x[1] = fill
        d = ctx.upload(x)
        ctx.flash_attn_f16kv(d.ptr, d.ptr + 4 * E, d.ptr + 8 * E, (1, 3 * E, D, 3 * E * S), D, S, H, 2, D ** -0.5, do,
                             o_strides=(1, E, D, E * S))
        outs.append(ctx.download(do, (2, S, E), np.float32))
        ctx.free(d)
    ctx.free(do)
    assert np.isfinite(outs[0]).all()
    for o in outs[1:]:
        assert np.array_equal(o[0].view(np.uint32), outs[0][0].view(np.uint32))
        assert np.isnan(o[1]).all()


@pytest.mark.parametrize("D,S,H", [(48, 577, 2), (48, 417, 50), (32, 353, 2), (64, 640, 2)])
def test_flash_attn_long_not_finite(ctx, D, S, H):
    """NaN and infinities (also fp32 values past fp16's largest) in q, k and v of one head: a score of
    -inf is a weight of zero, one of +inf or NaN makes the query's row NaN, a value that is not
    finite spoils its feature; everything else is what the finite softmax gives"""
    print(f"flash_attn_long not finite D={D} S={S} H={H}", flush=True)
    rng = np.random.default_rng(S)
    E = H * D
    x = rng.standard_normal((S, 3, H, D)).astype(np.float32)
    x[5, 0, 0, 3] = np.nan                        # a query
    x[7, 0, 0, 2] = np.inf
    x[100, 1, 0, 1] = -np.inf                     # a key: scores of either infinity, by the query's sign
    x[S - 1, 1, 1, 0] = 7e4                       # fp16: inf, in the last chunk
    x[70, 2, 0, 4], x[S - 2, 2, 0, 6] = np.nan, np.inf
    d, do = ctx.upload(x), ctx.alloc(S * E * 4)
    ctx.flash_attn_f16kv(d.ptr, d.ptr + 4 * E, d.ptr + 8 * E, (1, 3 * E, D, 3 * E * S), D, S, H, 1, D ** -0.5, do,
                         o_strides=(1, E, D, E * S))
    o = ctx.download(do, (S, H, D), np.float32)
    for t in (d, do):
        ctx.free(t)
    with np.errstate(invalid="ignore", over="ignore"):
        h = x.astype(np.float16).astype(np.float64)
        for i in range(min(H, 3)):
            sc = (h[:, 0, i, None, :] * h[None, :, 1, i, :]).sum(-1) * D ** -0.5
            p = np.exp(sc - sc.max(-1, keepdims=True))
            p /= p.sum(-1, keepdims=True)
            bad = ~np.isfinite(h[:, 2, i]).all(0)                     # features with a value that is not finite
            ref = p @ np.where(np.isfinite(h[:, 2, i]), h[:, 2, i], 0.0)
            rows = np.isfinite(p).all(-1)
            assert i or (0 < rows.sum() < S and bad.sum() == 2)
            assert np.isnan(o[~rows, i]).all()
            assert not np.isfinite(o[:, i][:, bad]).any()
            got, want = o[rows, i][:, ~bad], ref[rows][:, ~bad]
            assert np.isfinite(got).all() and np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


# rows closer together than a head: the whole-head kernel up to 512 keys (its 17-, 24- and 32-tile
# forms), the kernel for any strides beyond
@pytest.mark.parametrize("D,S,R", [(48, 270, 16), (48, 300, 20), (16, 384, 8), (64, 385, 32), (32, 512, 4), (48, 500, 44), (48, 600, 16),
                                   (32, 320, 0)])
def test_flash_attn_overlapping_rows(ctx, D, S, R):
    """key t's features start R elements after key t - 1's (R = 0: one key for all): against float64 on
    the fp16-rounded operands (bar of the other attention tests), fp16 inputs equal bit for bit"""
    H, B = 2, 2
    print(f"flash_attn overlapping rows D={D} S={S} R={R}", flush=True)
    rng = np.random.default_rng(D + S + R)
    P = -(-(S * R + D) // 8) * 8                  # elements between heads
    x = rng.standard_normal((3, B, H, P)).astype(np.float32)
    h = np.lib.stride_tricks.sliding_window_view(x.astype(np.float16).astype(np.float64), D, axis=-1)
    q, k, v = h[..., np.arange(S) * R, :]         # [B][H][S][D]
    sc = q @ k.swapaxes(-1, -2) * D ** -0.5
    p = np.exp(sc - sc.max(-1, keepdims=True))
    ref = (p @ v / p.sum(-1, keepdims=True)).transpose(0, 2, 1, 3).reshape(B * S, H * D)
    st, ost = (1, R, P, H * P), (1, H * D, D, H * D * S)
    d, do = ctx.upload(x), ctx.alloc(B * S * H * D * 4)
    n = B * H * P
    ctx.flash_attn_f16kv(d.ptr, d.ptr + 4 * n, d.ptr + 8 * n, st, D, S, H, B, D ** -0.5, do, o_strides=ost)
    o = ctx.download(do, (B * S, H * D), np.float32)
    assert _rel(o, ref) <= 2e-5
    if S <= 512:
        d16 = ctx.upload(x.astype(np.float16))
        ctx.flash_attn_f16in(d16.ptr, d16.ptr + 2 * n, d16.ptr + 4 * n, st, D, S, H, B, D ** -0.5, do, None, ost)
        assert np.array_equal(ctx.download(do, (B * S, H * D), np.float32).view(np.uint32), o.view(np.uint32))
        ctx.free(d16)
    for t in (d, do):
        ctx.free(t)


def test_flash_attn_long_strides(ctx):
    """The same attention through strides the long kernel does not take (features two elements
    apart: the kernel for any strides) and through ones it takes: both within 2e-5 max|ref| of
    each other."""
    D, S, H, B = 48, 600, 3, 2
    E = H * D
    rng = np.random.default_rng(5)
    x = rng.standard_normal((3, B * S, E)).astype(np.float32)
    two = np.zeros((3, B * S, 2 * E), np.float32)
    two[:, :, ::2] = x
    outs = []
    for a, m in ((x, 1), (two, 2)):
        d = [ctx.upload(a[i]) for i in range(3)]
        do = ctx.alloc(B * S * E * 4)
        st = (m, m * E, m * D, m * E * S)
        ctx.flash_attn_f16kv(d[0], d[1], d[2], st, D, S, H, B, 0.144, do, o_strides=(1, E, D, E * S))
        outs.append(ctx.download(do, (B * S, E), np.float32))
        for t in d + [do]:
            ctx.free(t)
    assert _rel(outs[0], outs[1]) <= 2e-5


@pytest.mark.parametrize("D,S,H,B,pad", [(48, 257, 16, 2, 0), (48, 1, 2, 1, 0), (64, 130, 4, 1, 0), (32, 512, 2, 1, 0),
                                         (48, 257, 4, 2, 4), (16, 33, 1, 3, 4), (64, 512, 2, 1, 12),
                                         (48, 273, 3, 1, 4), (48, 385, 50, 1, 0), (16, 300, 1, 1, 12)])
def test_flash_attn_f16in_equals_rounded_inputs(ctx, D, S, H, B, pad):
    """The fp16-input variant on q/k/v rounded to fp16 gives the same bits as the fp32-input
    attention (which rounds its inputs to fp16 on load), for both output types, with q/k/v
    read through the strides of one wide [S*B][3*H*D + pad] buffer (the fused QKV output; a
    pad of 4 or 12 halves leaves fp16 rows 8-byte but not 16-byte aligned)."""
    print(f"flash_attn_f16in D={D} S={S} H={H} B={B} pad={pad}", flush=True)
    rng = np.random.default_rng(7 * D + S)
    E = H * D
    R = 3 * E + pad
    wide = rng.standard_normal((B * S, R)).astype(np.float16)
    st = (1, R, D, R * S)
    ost = (1, E, D, E * S)
    d32 = ctx.upload(wide.astype(np.float32))
    d16 = ctx.upload(wide)
    n = D * S * H * B
    o_ref, o_32, o_16 = ctx.alloc(n * 4), ctx.alloc(n * 4), ctx.alloc(n * 2)
    ctx.flash_attn_f16kv(d32.ptr, d32.ptr + 4 * E, d32.ptr + 8 * E, st, D, S, H, B, 0.144, o_ref, o_strides=ost)
    ctx.flash_attn_f16in(d16.ptr, d16.ptr + 2 * E, d16.ptr + 4 * E, st, D, S, H, B, 0.144, o=o_32, o_strides=ost)
    ctx.flash_attn_f16in(d16.ptr, d16.ptr + 2 * E, d16.ptr + 4 * E, st, D, S, H, B, 0.144, o16=o_16, o_strides=ost)
    ref = ctx.download(o_ref, (n,), np.float32)
    a = ctx.download(o_32, (n,), np.float32)
    h = ctx.download(o_16, (n,), np.float16)
    for t in (d32, d16, o_ref, o_32, o_16):
        ctx.free(t)
    assert np.array_equal(a.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(h.view(np.uint16), ref.astype(np.float16).view(np.uint16))


def test_flash_attn_f16in_rejects_long_sequences(ctx):
    buf = ctx.alloc(1 << 20)
    with pytest.raises(ema.MghError):
        ctx.flash_attn_f16in(buf, buf, buf, (1, 48, 48, 48 * 600), 48, 600, 1, 1, 0.1, o=buf)
    with pytest.raises(ema.MghError):
        ctx.flash_attn_f16in(buf, buf, buf, (1, 48, 48, 48 * 4), 48, 4, 1, 1, 0.1, o=buf, o16=buf)
    ctx.free(buf)


def test_flash_attn_large_scores(ctx):
    """Peaked softmax (large logits): the running max rescaling must stay exact."""
    D, S, H, B = 48, 257, 2, 1
    print("flash_attn peaked", flush=True)
    rng = np.random.default_rng(3)
    q, k, v = _qkv(rng, D, S, H, B)
    q *= 6.0
    st = (1, H * D, D, H * D * S)
    ref = oracle.attention(q, k, v, st, D, S, H, B, 1.0 / np.sqrt(D), True)
    dq, dk, dv, do = ctx.upload(q), ctx.upload(k), ctx.upload(v), ctx.alloc(D * S * H * B * 4)
    ctx.flash_attn_f16kv(dq, dk, dv, st, D, S, H, B, 1.0 / np.sqrt(D), do)
    o = ctx.download(do, (D * S * H * B,), np.float32)
    for t in (dq, dk, dv, do):
        ctx.free(t)
    assert np.isfinite(o).all()
    assert _rel(o, ref) <= 2e-5


# ---- fp32 GEMM -------------------------------------------------------------------------
@pytest.mark.parametrize("M,N,K,act,res", [(1, 2025, 768, 0, False), (257, 2025, 768, 0, False),
                                           (70, 100, 64, 1, True), (130, 768, 3072, 2, True)])
def test_gemm_f32_vs_oracle(ctx, M, N, K, act, res):
    print(f"gemm_f32 M={M} N={N} K={K} act={act} resid={res}", flush=True)
    rng = np.random.default_rng(M + N + K)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    x = rng.standard_normal((M, K)).astype(np.float32)
    bias = (rng.standard_normal(N) * 0.1).astype(np.float32)
    resid = rng.standard_normal((M, N)).astype(np.float32) if res else None
    ref = oracle.gemm_f32(w, x, bias=bias, act=act, resid=resid)
    dW, dX, dB, dY = ctx.upload(w), ctx.upload(x), ctx.upload(bias), ctx.alloc(M * N * 4)
    dR = ctx.upload(resid) if res else None
    ctx.gemm_f32(dW, N, K, dX, M, dB, act, dR, dY)
    y = ctx.download(dY, (M, N), np.float32)
    for t in (dW, dX, dB, dY, dR):
        if t is not None:
            ctx.free(t)
    err = _rel(y, ref)
    print(f"  rel err {err:.2e}")
    assert err <= 1e-5


# Edges of the 64 x 64 tiles and of the 32-deep K steps, with up to one workgroup per CU (two LDS
# buffers) and more (one buffer); operands over 12 decades, so that all three parts of a value and the
# small products count.
@pytest.mark.parametrize("M,N,K,act,res", [(1, 1, 32, 0, False), (63, 65, 64, 0, True), (64, 64, 96, 1, False),
                                           (65, 63, 128, 2, True), (1088, 1024, 32, 0, False), (1089, 961, 96, 0, True),
                                           (1100, 1000, 160, 1, False)])
def test_gemm_f32_vs_float64(ctx, M, N, K, act, res):
    """each output within 2e-6 of sum_k |w x| + |bias| + |resid|, a few fp32 roundings of the running
    sum (2^-24 each, at most six per 32 values of k: below 3e-7 sqrt(6 K / 32))"""
    print(f"gemm_f32 float64 M={M} N={N} K={K} act={act} resid={res}", flush=True)
    rng = np.random.default_rng(M + 3 * N + K)

    def wide(*shape):
        return (rng.standard_normal(shape) * 10.0 ** rng.uniform(-6, 6, shape)).astype(np.float32)

    w, x = wide(N, K), wide(M, K)
    bias, resid = wide(N), wide(M, N) if res else None
    dW, dX, dB, dY = ctx.upload(w), ctx.upload(x), ctx.upload(bias), ctx.alloc(M * N * 4)
    dR = ctx.upload(resid) if res else None
    ctx.gemm_f32(dW, N, K, dX, M, dB, act, dR, dY)
    y = ctx.download(dY, (M, N), np.float32)
    for t in (dW, dX, dB, dY, dR):
        if t is not None:
            ctx.free(t)
    w, x, bias = w.astype(np.float64), x.astype(np.float64), bias.astype(np.float64)
    ref, mag = x @ w.T + bias, np.abs(x) @ np.abs(w).T + np.abs(bias)
    from scipy.special import erf
    with np.errstate(over="ignore"):
        ref = 0.5 * ref * (1 + erf(ref / np.sqrt(2))) if act == 1 else ref / (1 + np.exp(-ref)) if act == 2 else ref
    if res:
        ref, mag = ref + resid, mag + np.abs(resid)
    err = float((np.abs(y - ref) / mag).max())
    print(f"  err / sum of magnitudes {err:.2e}")
    assert err <= 2e-6


# exponents of x and w (ranges of powers of two): the smallest normal and subnormal numbers against
# large ones (products and sums of ordinary size), and values past the range that the parts are scaled for
@pytest.mark.parametrize("M", [65, 1089])
@pytest.mark.parametrize("ex,ew", [((-126, -100), (90, 110)), ((-149, -120), (100, 111)), ((90, 110), (-126, -100)),
                                   ((112, 126), (-126, -90)), ((-100, -64), (-40, -20)), ((40, 60), (30, 50))])
def test_gemm_f32_whole_range(ctx, M, ex, ew):
    """each output within 2e-6 of sum_k |w x| (as test_gemm_f32_vs_float64) or of the smallest normal
    number, over fp32's whole exponent range"""
    N, K = 1000, 64
    print(f"gemm_f32 range M={M} x 2^{ex} w 2^{ew}", flush=True)
    rng = np.random.default_rng(1000 + M + ex[0] + ew[0])

    def wide(lo, hi, *shape):
        v = rng.uniform(1, 2, shape) * rng.choice([-1.0, 1.0], shape)
        return np.ldexp(v, rng.integers(lo, hi + 1, shape)).astype(np.float32)

    x, w = wide(*ex, M, K), wide(*ew, N, K)
    dW, dX, dY = ctx.upload(w), ctx.upload(x), ctx.alloc(M * N * 4)
    ctx.gemm_f32(dW, N, K, dX, M, None, 0, None, dY)
    y = ctx.download(dY, (M, N), np.float32).astype(np.float64)
    for t in (dW, dX, dY):
        ctx.free(t)
    x, w = x.astype(np.float64), w.astype(np.float64)
    ref, mag = x @ w.T, np.abs(x) @ np.abs(w).T
    assert mag.max() < 2.0 ** 127
    err = float((np.abs(y - ref) / (mag + 2.0 ** -126)).max())
    print(f"  err / sum of magnitudes {err:.2e}")
    assert err <= 2e-6


@pytest.mark.parametrize("v", [1 + 2.0 ** -8, 1 + 2.0 ** -8 + 2.0 ** -16, 1.0 - 2.0 ** -9])
def test_gemm_f32_equal_operands(ctx, v):
    """equal operands, where the products left out (at most 2^-24 of a product each) add up with one
    sign: that and the running sum's roundings (2^-24 of it, six per 32 k, K = 128) in the worst case"""
    M, N, K = 70, 100, 128
    dW, dX, dY = ctx.upload(np.full((N, K), v, np.float32)), ctx.upload(np.full((M, K), v, np.float32)), ctx.alloc(M * N * 4)
    ctx.gemm_f32(dW, N, K, dX, M, None, 0, None, dY)
    y = ctx.download(dY, (M, N), np.float32).astype(np.float64)
    for t in (dW, dX, dY):
        ctx.free(t)
    ref = K * float(np.float32(v)) ** 2
    err = float(np.abs(y - ref).max() / ref)
    print(f"  relative error {err:.2e}")
    assert err <= 2.0 ** -24 * (1 + 6 * K / 32)


@pytest.mark.parametrize("M", [70, 1100])
def test_gemm_f32_not_finite(ctx, M):
    """infinities, NaN and values next to the largest float give what fp32 products and sums give"""
    N, K = 1000, 64
    print(f"gemm_f32 not finite M={M}", flush=True)
    rng = np.random.default_rng(M)
    w, x = (rng.standard_normal(s).astype(np.float32) for s in ((N, K), (M, K)))
    x[3, 5], x[66, 9], x[M - 1, 0] = np.inf, np.nan, -np.inf
    x[7] = 0
    x[7, 2] = np.finfo(np.float32).max
    w[11, 2], w[12, 5], w[13, 3], w[14] = 1.0, 0.0, np.inf, 0.0
    dW, dX, dY = ctx.upload(w), ctx.upload(x), ctx.alloc(M * N * 4)
    ctx.gemm_f32(dW, N, K, dX, M, None, 0, None, dY)
    y = ctx.download(dY, (M, N), np.float32)
    for t in (dW, dX, dY):
        ctx.free(t)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (x.astype(np.float64)[:, None, :] * w.astype(np.float64)[None]).sum(-1) if M < 100 else \
            np.stack([(x[m].astype(np.float64) * w.astype(np.float64)).sum(-1) for m in range(M)])
        ref = ref.astype(np.float32)
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    assert np.array_equal(np.isinf(y), np.isinf(ref)) and np.array_equal(np.sign(y[np.isinf(y)]), np.sign(ref[np.isinf(ref)]))
    ok = np.isfinite(ref)
    assert np.abs(y[ok] / np.maximum(np.abs(ref[ok]), 1.0) - ref[ok] / np.maximum(np.abs(ref[ok]), 1.0)).max() <= 2e-5


@pytest.mark.parametrize("M", [70, 1100])
@pytest.mark.parametrize("act", [0, 2])
def test_gemm_f32_not_finite_epilogue(ctx, M, act):
    """sums that are redone get bias, activation and residual once, also where the residual is y
    itself (read and written once per element): equal bit for bit to a residual of its own"""
    N, K = 1000, 64
    print(f"gemm_f32 not finite, epilogue M={M} act={act}", flush=True)
    rng = np.random.default_rng(M + act)
    w, x = (rng.standard_normal(s).astype(np.float32) for s in ((N, K), (M, K)))
    bias, resid = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    big = np.finfo(np.float32).max                # its first bf16 part is an infinity
    x[3, 5], x[M - 1, 0] = np.inf, np.nan
    x[7] = 0
    x[7, 2] = big
    w[:, 2] *= 0.25
    w[11, 2] = 1.0
    dW, dX, dB, dR = ctx.upload(w), ctx.upload(x), ctx.upload(bias), ctx.upload(resid)
    dY = ctx.alloc(M * N * 4)
    ctx.gemm_f32(dW, N, K, dX, M, dB, act, dR, dY)
    ctx.gemm_f32(dW, N, K, dX, M, dB, act, dR, dR)
    y, inplace = ctx.download(dY, (M, N), np.float32), ctx.download(dR, (M, N), np.float32)
    for t in (dW, dX, dB, dR, dY):
        ctx.free(t)
    assert np.array_equal(y.view(np.uint32), inplace.view(np.uint32))
    with np.errstate(invalid="ignore", over="ignore"):
        s = np.stack([(x[m].astype(np.float64) * w.astype(np.float64)).sum(-1) for m in range(M)]) + bias
        s = s.astype(np.float32).astype(np.float64)
        ref = ((s if act == 0 else s / (1 + np.exp(-s))) + resid).astype(np.float32)
    assert np.array_equal(np.isnan(y), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(y[inf], ref[inf])
    ok = np.isfinite(ref)
    assert ok[7].sum() > N // 2                   # finite sums of the largest value among them
    # as test_gemm_f32_not_finite: a few fp32 roundings of sums of K terms
    assert (np.abs(y[ok].astype(np.float64) - ref[ok]) / np.maximum(np.abs(ref[ok]).astype(np.float64), 1.0)).max() <= 2e-5


def test_gemm_f32_not_finite_cost(ctx):
    """rows of NaN cost at most ten times finite ones (measured: three and a half; summed one output
    after the other 160 times)"""
    M, N, K = 4112, 2025, 768
    rng = np.random.default_rng(1)
    dW, dY = ctx.upload(rng.standard_normal((N, K)).astype(np.float32)), ctx.alloc(M * N * 4)
    ms = []
    for fill, reps in ((1.0, 20), (np.nan, 2)):
        dX = ctx.upload(np.full((M, K), fill, np.float32))
        for timed in (False, True):
            ctx.sync()
            ctx.timer_start()
            for _ in range(reps):
                ctx.gemm_f32(dW, N, K, dX, M, None, 0, None, dY)
            t = ctx.timer_stop() / reps
        ms.append(t)
        ctx.free(dX)
    y = ctx.download(dY, (M, N), np.float32)
    for b in (dW, dY):
        ctx.free(b)
    print(f"  finite {ms[0] * 1e3:.0f} us, NaN {ms[1] * 1e3:.0f} us")
    assert np.isnan(y).all() and ms[1] <= 10 * ms[0]


# ---- glue ------------------------------------------------------------------------------
def test_get_rows_add_copy(ctx):
    print("glue ops", flush=True)
    rng = np.random.default_rng(11)
    R, E = 2025, 768
    table = rng.standard_normal((R, E)).astype(np.float32)
    ids = rng.integers(-R, R, 3 * 257).astype(np.int32)
    dT, dI, dO = ctx.upload(table), ctx.upload(ids), ctx.alloc(ids.size * E * 4)
    ctx.get_rows(dT, E, R, dI, ids.size, dO)
    got = ctx.download(dO, (ids.size, E), np.float32)
    assert np.array_equal(got, oracle.get_rows(table, ids))
    pos = rng.standard_normal((257, E)).astype(np.float32)
    dP, dS = ctx.upload(pos), ctx.alloc(ids.size * E * 4)
    ctx.add(dO, dP, pos.size, dS, ids.size * E)
    s = ctx.download(dS, (3, 257, E), np.float32)
    assert np.array_equal(s, got.reshape(3, 257, E) + pos[None])
    # head merge: {D,S,H,B} contiguous -> permute(0,2,1,3) -> [S*B][H*D]
    D, S, H, B = 48, 257, 16, 2
    a = rng.standard_normal(D * S * H * B).astype(np.float32)
    dA, dM = ctx.upload(a), ctx.alloc(a.nbytes)
    ctx.copy_strided(dA, (D, H, S, B), (1, D * S, D, D * S * H), dM)
    m = ctx.download(dM, (a.size,), np.float32)
    assert np.array_equal(m, oracle.merge_heads(a, D, S, H, B))
    for t in (dT, dI, dO, dP, dS, dA, dM):
        ctx.free(t)
