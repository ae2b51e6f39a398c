"""Performance cases of the MI355X MaskGIT backend: what a program that uses it runs, through its
Python entry points (`edge_maskgit_amd.Context` over include/mgh.h and
`edge_maskgit_amd.runtime.TransformerRuntime` over include/mgr.h).

Model sizes are the production ones (hidden 768, 16 heads of 48, MLP 3072, vocabulary 2025, 24
layers; VQGAN decoder 16 x 16 tokens -> 256 x 256, 128 filters, multipliers 1, 1, 2, 2, 4); token
rows are those of 256-, 1024- and 4096-token images (257, 1025 and 4097 with the class token) and
of batches of 257-token images.

Kinds:
  layer    one post-norm transformer layer as the runtime runs it: fused QKV FC (fp16 out),
           attention, out-projection + LayerNorm, up-projection + GELU, down-projection +
           LayerNorm
  fc4      the four FC nodes of a layer, each on fp32 activations (the graph API's MulMat node)
  attn     attention on the fp32 output of the fused QKV FC, heads merged
  head     the tied fp32 output head (F32 MulMat)
  conv     a convolution of the VQGAN decoder, fp32
  conv_i8  the same on the int8 path
  forward  a whole 24-layer forward: token ids in, logits back on the host
  decode   a whole VQGAN decode: token grids in, images back on the host

Every operand a program holds before the call (weights in the backend's layout, activations,
output buffers) is made in prepare(); run() only makes the calls.
"""
import math
import os
import tempfile

import numpy as np
import torch

import edge_maskgit_amd as ema
from edge_maskgit_amd.gguf import write_gguf
from edge_maskgit_amd.runtime import TransformerRuntime

E, FFN, HEADS, VOCAB, CODES, LAYERS = 768, 3072, 16, 2025, 1024, 24
EPS = 1e-12
VQ_EMBED, VQ_FILTERS, VQ_MULT, VQ_BLOCKS, VQ_TOKENS, VQ_GROUPS = 256, 128, (1, 1, 2, 2, 4), 2, 256, 32
QUANT = {"q8_0": ema.WTYPE_Q8_0, "q4_k": ema.WTYPE_Q4_K}
# (N, K, activation, residual) of a layer's FCs: fused QKV, out, up, down
FC4 = ((3 * E, E, 0, False), (E, E, 0, True), (FFN, E, 1, False), (E, FFN, 0, True))


def listed():
    return [
        # one image (256 tokens + class): the smallest layer call, launches and latency count
        dict(name="layer_b1", kind="layer", batch=1, form="f16", quant="q8_0"),
        # a batch of 16 images, the throughput case
        dict(name="layer_b16", kind="layer", batch=16, form="f16", quant="q8_0"),
        # the FC nodes of a 1024-token image on the stored Q8_0 bytes
        dict(name="fc4_q8_m1025", kind="fc4", rows=1025, form="bytes", quant="q8_0"),
        # the FC nodes of a 4096-token image on Q4_K, the smallest model file
        dict(name="fc4_q4k_m4097", kind="fc4", rows=4097, form="bytes", quant="q4_k"),
        # the int8-dot algorithm (per-32 activation codes) on a 1024-token image
        dict(name="fc4_int8_m1025", kind="fc4", rows=1025, form="int8", quant="q8_0"),
        # attention over a 1024-token and a 4096-token image
        dict(name="attn_s1025", kind="attn", batch=1, seq=1025, heads=16, dim=48),
        dict(name="attn_s4097", kind="attn", batch=1, seq=4097, heads=16, dim=48),
        # logits of 16 images
        dict(name="head_m4112", kind="head", rows=4112, n=VOCAB, k=E),
        # the decoder's full-resolution 3 x 3 convolution with a res-block's residual, one image
        dict(name="conv_256", kind="conv", side=256, ic=128, oc=128, ksz=3, batch=1, resid=True),
        # the decoder's middle level on the int8 path, 8 images (one decode group)
        dict(name="conv_i8_64", kind="conv_i8", side=64, ic=256, oc=256, ksz=3, batch=8, resid=True),
        # one step of a single image's generation
        dict(name="forward_b1", kind="forward", batch=1, algo=2),
        # two generated grids to images
        dict(name="decode_b2", kind="decode", batch=2, algo=2),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "fc4", "fc4", "fc4", "attn", "attn", "head", "conv", "conv", "conv_i8",
                       "forward", "decode"])
    if kind == "layer":
        return dict(kind=kind, batch=_log_int(rng, 1, 16), form=rng.choice(["f16", "bytes"]),
                    quant=rng.choice(["q8_0", "q4_k"]))
    if kind == "fc4":
        return dict(kind=kind, rows=_log_int(rng, 200, 4097), form=rng.choice(["f16", "bytes", "bytes", "int8"]),
                    quant=rng.choice(["q8_0", "q4_k"]))
    if kind == "attn":
        seq = _log_int(rng, 257, 4097)
        most = max(1, min(4, 4097 * 4097 // (seq * seq)))
        return dict(kind=kind, batch=rng.randint(1, most), seq=seq, heads=rng.choice([8, 12, 16]),
                    dim=rng.choice([32, 48, 48, 64]) if seq < 3500 else 48)
    if kind == "head":
        return dict(kind=kind, rows=_log_int(rng, 257, 4112), n=rng.choice([VOCAB, VOCAB, CODES, 1000, 2001]),
                    k=rng.choice([512, E, E]))
    if kind in ("conv", "conv_i8"):
        top = 256 * 256 * 128 * 128 * 9 if kind == "conv" else 8 * 64 * 64 * 256 * 256 * 9
        side = rng.choice([16, 20, 32, 48, 50, 64, 96, 128, 200, 256])
        chan = [c for c in (64, 128, 256, 512) if side * side * c * c * 9 <= top]
        ic, oc = rng.choice(chan), rng.choice(chan)
        ksz = rng.choice([3, 3, 3, 1])
        batch = rng.randint(1, max(1, min(8, top // (side * side * ic * oc * 9))))
        return dict(kind=kind, side=side, ic=ic, oc=oc, ksz=ksz, batch=batch, resid=rng.choice([True, False]))
    if kind == "forward":
        return dict(kind=kind, batch=rng.randint(1, 6), algo=rng.choice([2, 2, 3]))
    return dict(kind="decode", batch=rng.choice([1, 2]), algo=2)


# ---- inputs -------------------------------------------------------------------------------

_CTX = None


def _ctx():
    """the program's one kernel context"""
    global _CTX
    if _CTX is None:
        _CTX = ema.Context(0)
    return _CTX


def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape, scale=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device=g.device, dtype=torch.float32) * scale + mean


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _quantize(quant, w):
    """ggml blocks [N][row bytes] of w [N][K]: Q8_0 (fp16 d = amax / 127, int8 codes) or Q4_K
    (min / max sub-blocks of 32 with 6-bit scales and mins over fp16 d, dmin)"""
    n, k = w.shape
    if quant == "q8_0":
        b = w.view(n, k // 32, 32)
        d = b.abs().amax(-1, keepdim=True) / 127
        q = (b / d).round().clamp(-127, 127).to(torch.int8)
        return torch.cat([_bytes(d.half()).view(n, k // 32, 2), _bytes(q)], -1).view(n, -1)
    x = w.view(-1, 8, 32)
    mn = x.amin(-1).clamp(max=0)
    sc = (x.amax(-1) - mn) / 15
    d, dm = sc.amax(-1, keepdim=True) / 63, (-mn).amax(-1, keepdim=True) / 63
    scq, mq = (sc / d).round().clamp(1, 63), (-mn / dm).round().clamp(0, 63)
    q = ((x + (dm * mq)[..., None]) / (d * scq)[..., None]).round().clamp(0, 15).to(torch.uint8)
    scq, mq = scq.to(torch.uint8), mq.to(torch.uint8)
    out = [_bytes(d.half()), _bytes(dm.half()), (scq[:, :4] & 63) | ((scq[:, 4:] >> 4) << 6),
           (mq[:, :4] & 63) | ((mq[:, 4:] >> 4) << 6), (scq[:, 4:] & 15) | ((mq[:, 4:] & 15) << 4)]
    out += [q[:, 2 * i] | (q[:, 2 * i + 1] << 4) for i in range(4)]
    return torch.cat(out, -1).view(n, -1)


def _dequantize(quant, blocks, n, k):
    """the blocks' values as the formats define them, float64 [N][K]"""
    if quant == "q8_0":
        b = blocks.view(n, k // 32, 34)
        d = b[..., :2].contiguous().view(torch.float16).double()
        return (d * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    b = blocks.reshape(-1, 144)
    d, dm = (b[:, i:i + 2].contiguous().view(torch.float16).double() for i in (0, 2))
    s, m, h = b[:, 4:8].int(), b[:, 8:12].int(), b[:, 12:16].int()
    sc = torch.cat([s & 63, (h & 15) | ((s >> 6) << 4)], -1)
    mn = torch.cat([m & 63, (h >> 4) | ((m >> 6) << 4)], -1)
    qs = b[:, 16:].view(-1, 4, 32).int()
    q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32)
    return ((d * sc)[..., None] * q - (dm * mn)[..., None]).reshape(n, k)


def _pack(form, quant, blocks, n, k):
    """the weight in the layout of `form`, as a program lays it out once at load"""
    c, wt = _ctx(), QUANT[quant]
    size, fn = {"f16": (ema.packed_weight_bytes_f16(n, k), c.pack_weights_f16),
                "bytes": (ema.packed_weight_bytes_dq(wt, n, k), c.pack_weights_dq),
                "int8": (ema.packed_weight_bytes(wt, n, k), c.pack_weights)}[form]
    out = torch.empty(size, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    fn(wt, blocks.data_ptr(), n, k, out.data_ptr())
    c.sync()
    return out


def _dev(*shape, dtype=torch.float32):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


def _prepare_layer(case, seed):
    g = _gen(seed)
    m = case["batch"] * 257
    s = {"case": case, "m": m, "x": _randn(g, m, E)}
    s["x16"] = s["x"].half()
    for i, (n, k, _, _) in enumerate(FC4):
        blocks = _quantize(case["quant"], _randn(g, n, k, scale=0.02))
        s["w%d" % i] = _pack(case["form"], case["quant"], blocks, n, k)
        s["b%d" % i] = _randn(g, n, scale=0.01)
        s["blocks%d" % i] = blocks.cpu()
    for i in (1, 3):
        s["gamma%d" % i], s["beta%d" % i] = _randn(g, E, scale=0.02, mean=1.0), _randn(g, E, scale=0.01)
        s["ln%d" % i], s["ln16%d" % i] = _dev(m, E), _dev(m, E, dtype=torch.float16)
    s["qkv"], s["att"], s["up"] = (_dev(m, n, dtype=torch.float16) for n in (3 * E, E, FFN))
    return s


def _prepare_fc4(case, seed):
    g = _gen(seed)
    m = case["rows"]
    s = {"case": case, "m": m}
    for i, (n, k, _, resid) in enumerate(FC4):
        blocks = _quantize(case["quant"], _randn(g, n, k, scale=0.02))
        s["w%d" % i] = _pack(case["form"], case["quant"], blocks, n, k)
        s["blocks%d" % i] = blocks.cpu()
        s["b%d" % i] = _randn(g, n, scale=0.01)
        x = _randn(g, m, k)
        # the down-projection reads GELU outputs
        s["x%d" % i] = torch.nn.functional.gelu(x) if k == FFN else x
        s["r%d" % i] = _randn(g, m, n) if resid else None
        s["y%d" % i] = _dev(m, n)
    return s


def _prepare_attn(case, seed):
    g = _gen(seed)
    b, sq, w = case["batch"], case["seq"], case["heads"] * case["dim"]
    return {"case": case, "qkv": _randn(g, b * sq, 3 * w), "o": _dev(b * sq, w)}


def _prepare_head(case, seed):
    g = _gen(seed)
    m, n, k = case["rows"], case["n"], case["k"]
    return {"case": case, "w": _randn(g, n, k, scale=0.02), "x": _randn(g, m, k), "b": _randn(g, n, scale=0.01),
            "y": _dev(m, n)}


def _prepare_conv(case, seed):
    g, c = _gen(seed), _ctx()
    side, ic, oc, ksz, nb = (case[k] for k in ("side", "ic", "oc", "ksz", "batch"))
    x = _randn(g, nb, ic, side, side)
    s = {"case": case, "x": torch.nn.functional.silu(x), "w": _randn(g, oc, ic, ksz, ksz, scale=(ic * ksz * ksz) ** -0.5),
         "b": _randn(g, oc, scale=0.05), "r": _randn(g, nb, oc, side, side) if case["resid"] else None,
         "y": _dev(nb, oc, side, side)}
    if case["kind"] == "conv":
        s["pk"] = torch.empty(c.conv2d_packed_bytes(ksz, ksz, ic, oc), dtype=torch.uint8, device="cuda")
        pack = c.conv2d_pack_weights
    else:
        s["pk"] = torch.empty(c.conv2d_i8_weight_bytes(ksz, ksz, ic, oc), dtype=torch.uint8, device="cuda")
        pack = c.conv2d_i8_pack_weights
    torch.cuda.synchronize()
    pack(s["w"].data_ptr(), ksz, ksz, ic, oc, s["pk"].data_ptr())
    c.sync()
    return s


# The models of the whole calls: one file and one runtime per algorithm for the program's life.
_MODEL = {}


def _model_tensors(kind):
    """metadata, [(name, shape, ggml type, bytes)] and the values (float tensors, blocks of the FC
    weights) of a random-init model of the given kind"""
    g = _gen(5 if kind == "forward" else 11)
    tensors, values = [], {}

    def f32(name, t):
        values[name] = t.cpu()
        tensors.append((name, tuple(t.shape), 0, values[name].numpy().tobytes()))

    def fc(name, n, k):
        blocks = _quantize("q8_0", _randn(g, n, k, scale=0.02)).cpu()
        values[name + ".weight"] = blocks
        tensors.append((name + ".weight", (n, k), ema.WTYPE_Q8_0, blocks.numpy().tobytes()))
        f32(name + ".bias", _randn(g, n, scale=0.01))

    def norm(name, n, scale=0.02, bias=0.01):
        f32(name + ".weight", _randn(g, n, scale=scale, mean=1.0))
        f32(name + ".bias", _randn(g, n, scale=bias))

    def conv(name, oc, ic, k, bias):
        f32(name + ".weight", _randn(g, oc, ic, k, k, scale=(ic * k * k) ** -0.5))
        if bias:
            f32(name + ".bias", _randn(g, oc, scale=0.05))

    meta = [("general.architecture", "str", "maskgit"), ("general.alignment", "u32", 32),
            ("maskgit.n_tokens", "u32", VQ_TOKENS), ("maskgit.vqgan.codebook_size", "u32", CODES)]
    if kind == "forward":
        f32("token_embd.weight", _randn(g, VOCAB, E, scale=0.02))
        f32("pos_embd.weight", _randn(g, VQ_TOKENS + 1, E, scale=0.02))
        norm("token_embd_norm", E)
        for i in range(LAYERS):
            p = "blk.%d." % i
            for name, n, k in (("attn_q", E, E), ("attn_k", E, E), ("attn_v", E, E), ("attn_o", E, E),
                               ("ffn_up", FFN, E), ("ffn_down", E, FFN)):
                fc(p + name, n, k)
            norm(p + "attn_norm", E)
            norm(p + "ffn_norm", E)
        fc("output_proj", E, E)
        norm("output_norm", E)
        f32("output.bias", _randn(g, VOCAB, scale=0.01))
        meta += [("maskgit.n_layer", "u32", LAYERS), ("maskgit.n_head", "u32", HEADS), ("maskgit.n_embd", "u32", E),
                 ("maskgit.n_ffn", "u32", FFN), ("maskgit.head_dim", "u32", E // HEADS),
                 ("maskgit.vocab_size", "u32", VOCAB), ("maskgit.n_positions", "u32", VQ_TOKENS + 1),
                 ("maskgit.mask_token_id", "i32", VOCAB - 1), ("maskgit.layernorm_eps", "f32", EPS),
                 ("maskgit.sampling.choice_temperature", "f32", 4.5)]
    else:
        f32("vqgan.quantizer.codebook.weight", _randn(g, CODES, VQ_EMBED))
        for name, spec in _decoder():
            if spec[0] == "conv":
                conv(name, *spec[1:])
            elif spec[0] == "norm":
                norm(name, spec[1], 0.1, 0.1)
        meta += [("maskgit.resolution", "u32", 256), ("maskgit.vqgan.embedding_dim", "u32", VQ_EMBED),
                 ("maskgit.vqgan.filters", "u32", VQ_FILTERS), ("maskgit.vqgan.num_res_blocks", "u32", VQ_BLOCKS),
                 ("maskgit.vqgan.group_norm_groups", "u32", VQ_GROUPS),
                 ("maskgit.vqgan.channel_multipliers", "i32_array", list(VQ_MULT))]
    return meta, tensors, values


def _decoder():
    """the decoder's layers in order: (name, ("conv", oc, ic, ksz, bias)), (name, ("norm", c)), and the
    markers ("block", ...) / ("up",) that exact() follows"""
    d, out = "vqgan.decoder.", []
    width = VQ_FILTERS * VQ_MULT[-1]

    def block(p, ci, co):
        out.append((p, ("block", ci, co)))
        out.append((p + "norm0", ("norm", ci)))
        out.append((p + "conv0", ("conv", co, ci, 3, False)))
        out.append((p + "norm1", ("norm", co)))
        out.append((p + "conv1", ("conv", co, co, 3, False)))
        if ci != co:
            out.append((p + "conv_res", ("conv", co, co, 1, False)))

    out.append((d + "conv_in", ("conv", width, VQ_EMBED, 3, True)))
    for b in range(VQ_BLOCKS):
        block(d + "res_blocks.0.%d." % b, width, width)
    for i in range(len(VQ_MULT) - 1, -1, -1):
        j, co = len(VQ_MULT) - i, VQ_FILTERS * VQ_MULT[i]
        for b in range(VQ_BLOCKS):
            block(d + "res_blocks.%d.%d." % (j, b), width, co)
            width = co
        if i > 0:
            out.append(("up", ("up",)))
            out.append((d + "res_blocks.%d.%d" % (j, VQ_BLOCKS + 1), ("conv", width, width, 3, True)))
    out.append((d + "norm_out", ("norm", width)))
    out.append((d + "conv_out", ("conv", 3, width, 3, True)))
    return out


def _values(kind):
    if kind not in _MODEL:
        _MODEL[kind] = _model_tensors(kind)
    return _MODEL[kind]


def _runtime(kind, algo):
    if (kind, algo) not in _MODEL:
        meta, tensors, _ = _values(kind)
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "model.gguf")
            write_gguf(path, meta, tensors)
            rt = TransformerRuntime(path, algo=algo)
            if kind == "forward":       # the first call lays the weights out
                rt.forward(np.full((1, VQ_TOKENS + 1), VOCAB - 1, np.int32), readback=False)
            else:
                rt.decode_images(np.zeros((1, VQ_TOKENS), np.int32), readback=False)
        _MODEL[(kind, algo)] = rt
    return _MODEL[(kind, algo)]


def _prepare_forward(case, seed):
    g = _gen(seed, "cpu")
    b = case["batch"]
    t = torch.randint(0, CODES, (b, VQ_TOKENS + 1), generator=g)
    t[:, 0] = CODES + torch.randint(0, 1000, (b,), generator=g)            # class token
    hide = torch.rand(b, VQ_TOKENS, generator=g) < 0.5                     # half the image still masked
    t[:, 1:][hide] = VOCAB - 1
    return {"case": case, "rt": _runtime("forward", case["algo"]), "tokens": t.to(torch.int32).numpy()}


def _prepare_decode(case, seed):
    g = _gen(seed, "cpu")
    grid = torch.randint(0, CODES, (case["batch"], VQ_TOKENS), generator=g)
    return {"case": case, "rt": _runtime("decode", case["algo"]), "grids": grid.to(torch.int32).numpy()}


def prepare(case, seed):
    state = {"layer": _prepare_layer, "fc4": _prepare_fc4, "attn": _prepare_attn, "head": _prepare_head,
             "conv": _prepare_conv, "conv_i8": _prepare_conv, "forward": _prepare_forward,
             "decode": _prepare_decode}[case["kind"]](case, seed)
    # device addresses, as a program that binds the C ABI holds them
    state["ptr"] = {k: v.data_ptr() for k, v in state.items() if torch.is_tensor(v) and v.is_cuda}
    torch.cuda.synchronize()
    return state


# ---- one pass -----------------------------------------------------------------------------


def _run_layer(s):
    c, p, m, case = _ctx(), s["ptr"], s["m"], s["case"]
    seq, d = 257, E // HEADS
    qkv, st, ost = p["qkv"], (1, 3 * E, d, seq * 3 * E), (1, E, d, seq * E)
    if case["form"] == "f16":
        y16, ln = c.gemm_h16_y16, c.gemm_h16_ln
    else:
        wt = QUANT[case["quant"]]

        def y16(*a):
            c.gemm_dq_y16(wt, *a)

        def ln(*a):
            c.gemm_dq_ln(wt, *a)
    y16(p["w0"], 3 * E, E, p["x16"], m, p["b0"], 0, None, qkv)
    c.flash_attn_f16in(qkv, qkv + 2 * E, qkv + 4 * E, st, d, seq, HEADS, case["batch"], d ** -0.5, None, p["att"], ost)
    ln(p["w1"], E, E, p["att"], m, p["b1"], 0, p["x"], None, p["gamma1"], p["beta1"], EPS, p["ln1"],
       ema.EMIT_DEQ_F16, p["ln161"])
    y16(p["w2"], FFN, E, p["ln161"], m, p["b2"], ema.ACT_GELU, None, p["up"])
    ln(p["w3"], E, FFN, p["up"], m, p["b3"], 0, p["ln1"], None, p["gamma3"], p["beta3"], EPS, p["ln3"],
       ema.EMIT_DEQ_F16, p["ln163"])
    return {"x": s["ln3"], "x16": s["ln163"]}


def _run_fc4(s):
    c, p, m, case = _ctx(), s["ptr"], s["m"], s["case"]
    wt = QUANT[case["quant"]]
    for i, (n, k, act, resid) in enumerate(FC4):
        w, x, b, r, y = p["w%d" % i], p["x%d" % i], p["b%d" % i], p["r%d" % i] if resid else None, p["y%d" % i]
        if case["form"] == "f16":
            c.gemm_h16_f32in(w, n, k, x, m, b, act, r, y)
        elif case["form"] == "bytes":
            c.gemm_dq_f32in(wt, w, n, k, x, m, b, act, r, y)
        else:
            c.gemm_q_packed_f32in(ema.ALGO_INT8, wt, w, n, k, x, m, b, act, r, y)
    return [s["y%d" % i] for i in range(4)]


def _run_attn(s):
    case, q = s["case"], s["ptr"]["qkv"]
    h, d, seq = case["heads"], case["dim"], case["seq"]
    w = h * d
    _ctx().flash_attn_f16kv(q, q + 4 * w, q + 8 * w, (1, 3 * w, d, seq * 3 * w), d, seq, h, case["batch"], d ** -0.5,
                            s["ptr"]["o"], (1, w, d, seq * w))
    return s["o"]


def _run_head(s):
    case, p = s["case"], s["ptr"]
    _ctx().gemm_f32(p["w"], case["n"], case["k"], p["x"], case["rows"], p["b"], 0, None, p["y"])
    return s["y"]


def _run_conv(s):
    case, p = s["case"], s["ptr"]
    side, ic, oc, ksz, nb = (case[k] for k in ("side", "ic", "oc", "ksz", "batch"))
    if case["kind"] == "conv":
        _ctx().conv2d_ex(p["x"], side, side, ic, nb, p["w"], p["pk"], ksz, ksz, oc, 1, ksz // 2, p["b"], p.get("r"),
                         p["y"])
    else:
        _ctx().conv2d_i8(p["x"], side, side, ic, nb, p["pk"], ksz, ksz, oc, 1, ksz // 2, p["b"], p.get("r"), p["y"])
    return s["y"]


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return _run_layer(state)
    if kind == "fc4":
        return _run_fc4(state)
    if kind == "attn":
        return _run_attn(state)
    if kind == "head":
        return _run_head(state)
    if kind in ("conv", "conv_i8"):
        return _run_conv(state)
    if kind == "forward":
        return state["rt"].forward(state["tokens"])
    return state["rt"].decode_images(state["grids"])


# ---- what a pass cannot do without ----------------------------------------------------------


def _row_bytes(quant, k):
    return k // 32 * 34 if quant == "q8_0" else k // 256 * 144


def _conv_flops(side, ic, oc, ksz, batch):
    return 2 * side * side * ic * oc * ksz * ksz * batch


def work(case):
    kind = case["kind"]
    if kind == "layer":
        m = case["batch"] * 257
        w = sum(n * (_row_bytes(case["quant"], k) if case["form"] == "bytes" else 2 * k) for n, k, _, _ in FC4)
        return {"bytes": w + m * E * (4 + 2) * 2,
                "flops": 2 * m * sum(n * k for n, k, _, _ in FC4) + 4 * m * 257 * E}
    if kind == "fc4":
        m, total = case["rows"], 0
        for n, k, _, resid in FC4:
            total += n * (2 * k if case["form"] == "f16" else _row_bytes(case["quant"], k)) + 4 * n
            total += 4 * m * (k + n + (n if resid else 0))
        return {"bytes": total, "flops": 2 * m * sum(n * k for n, k, _, _ in FC4)}
    if kind == "attn":
        r, w = case["batch"] * case["seq"], case["heads"] * case["dim"]
        return {"bytes": 16 * r * w, "flops": 4 * r * case["seq"] * w}
    if kind == "head":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + n * k + n + m * n), "flops": 2 * m * n * k}
    if kind in ("conv", "conv_i8"):
        side, ic, oc, ksz, nb = (case[k] for k in ("side", "ic", "oc", "ksz", "batch"))
        out = nb * side * side * oc
        w = oc * ic * ksz * ksz * (4 if kind == "conv" else 1.125)
        return {"bytes": 4 * (nb * side * side * ic + out * (2 if case["resid"] else 1)) + w,
                "flops": _conv_flops(side, ic, oc, ksz, nb)}
    if kind == "forward":
        m = case["batch"] * 257
        fcs = LAYERS * sum(n * k for n, k, _, _ in FC4) + E * E
        return {"bytes": fcs * (2 if case["algo"] == 2 else 1.0625) + 4 * VOCAB * E + 4 * m * VOCAB,
                "flops": 2 * m * (fcs + VOCAB * E) + LAYERS * 4 * m * 257 * E}
    side, flops, weights = 16, 0, 0
    for _, spec in _decoder():
        if spec[0] == "up":
            side *= 2
        elif spec[0] == "conv":
            _, oc, ic, ksz, _ = spec
            flops += _conv_flops(side, ic, oc, ksz, case["batch"])
            weights += oc * ic * ksz * ksz
    return {"bytes": weights * 4 + case["batch"] * 3 * 256 * 256 * 4, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    # one product on fixed operands (fp16 or int8 operands and their scales are part of the
    # definition): only the order of fp32 sums is free. Measured against 64 bits: up to 7e-7
    # (4097-key attention), 5e-7 (head), 3e-7 (conv), 2e-7 (FC)
    if kind == "fc4" and case["form"] == "int8" and case["quant"] == "q4_k":
        # the Q4_K min term is summed from 16-bit halves (hi + lo): 2.5e-4 from 64 bits, max 4e-4
        return {"rel": 1e-3, "max": 2e-3}
    if kind in ("fc4", "attn", "head", "conv", "conv_i8"):
        return {"rel": 4e-6, "max": 1e-4}
    # fp16 between the calls: a sum that lands on a rounding boundary moves a value by 2^-11.
    # Measured between tile plans (other K splits): layer 1e-4, max 1e-3; forward 6.6e-4, max 3.8e-3
    if kind == "layer":
        return {"rel": 4e-4, "max": 4e-3}
    if kind == "forward":
        return {"rel": 2.6e-3, "max": 1.5e-2}
    # fp32 throughout, 39 convolutions deep: 2.4e-6 from 64 bits, max 1.3e-5
    return {"rel": 1e-5, "max": 6e-5}


# ---- the same in 64 bits ----------------------------------------------------------------------


def _h(t):
    """rounded to fp16, where the path's definition says so"""
    return t.half().double()


def _gelu64(t):
    return 0.5 * t * (1 + torch.erf(t * 0.5 ** 0.5))


def _ln64(t, gamma, beta):
    d = t - t.mean(-1, keepdim=True)
    return d / (d.square().mean(-1, keepdim=True) + EPS).sqrt() * gamma.double() + beta.double()


def _attn64(q, k, v, scale):
    """q, k, v [B][H][S][D], head by head"""
    o = torch.empty_like(q)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            o[b, h] = torch.softmax(q[b, h] @ k[b, h].t().contiguous() * scale, -1) @ v[b, h]
    return o


def _split_heads(t, batch, seq, heads, dim):
    return [x.reshape(batch, seq, heads, dim).transpose(1, 2).contiguous() for x in t.split(heads * dim, -1)]


def _merge_heads(o):
    return o.transpose(1, 2).reshape(-1, o.shape[1] * o.shape[3]).contiguous()


def _layer64(x, w, b, g1, be1, g3, be3, batch):
    """the dequantize-fused layer: operands rounded to fp16, everything else in 64 bits"""
    qkv = _h(_h(x) @ w[0].t() + b[0])
    o = _merge_heads(_attn64(*_split_heads(qkv, batch, 257, HEADS, E // HEADS), (E // HEADS) ** -0.5))
    y = _ln64(_h(o) @ w[1].t() + b[1] + x, g1, be1)
    up = _h(_gelu64(_h(y) @ w[2].t() + b[2]))
    return _ln64(up @ w[3].t() + b[3] + y, g3, be3)


def _codes64(x):
    """per-32 int8 activation codes times their fp32 scale (amax / 127, halves away from zero)"""
    b = x.float().reshape(*x.shape[:-1], -1, 32)
    d = (b.abs().amax(-1, keepdim=True).double() / 127).float()
    i = torch.where(d > 0, (1 / d.double()).float(), torch.zeros_like(d))
    y = (b * i).double()
    return (torch.sign(y) * torch.floor(y.abs() + 0.5) * d.double()).reshape(x.shape)


def _conv64(x, w, codes=False):
    """x [N][C][H][W], w [OC][IC][K][K], padding K // 2"""
    n, c, h, wd = x.shape
    oc, k = w.shape[0], w.shape[2]
    out = torch.empty(n, oc, h, wd, dtype=torch.float64, device=x.device)
    for i in range(n):
        if codes:
            cols = torch.nn.functional.unfold(x[i:i + 1].float(), k, padding=k // 2)[0].t().contiguous()
            out[i] = (_codes64(w.float().reshape(oc, -1)) @ _codes64(cols).t().contiguous()).view(oc, h, wd)
            continue
        p = torch.nn.functional.pad(x[i].double(), [k // 2] * 4)
        acc = torch.zeros(oc, h * wd, dtype=torch.float64, device=x.device)
        for a in range(k):
            for b in range(k):
                acc += w[:, :, a, b].double().contiguous() @ p[:, a:a + h, b:b + wd].reshape(c, -1)
        out[i] = acc.view(oc, h, wd)
    return out


def _gn_silu64(x, gamma, beta):
    n, c = x.shape[:2]
    g = x.view(n, VQ_GROUPS, -1)
    d = g - g.mean(-1, keepdim=True)
    y = (d / (d.square().mean(-1, keepdim=True) + 1e-5).sqrt()).view_as(x)
    return torch.nn.functional.silu(y * gamma.double().view(1, c, 1, 1) + beta.double().view(1, c, 1, 1))


def _decode64(grids, values):
    v = {k: t.cuda() for k, t in values.items()}
    x = v["vqgan.quantizer.codebook.weight"].double()[torch.from_numpy(grids).long().cuda()]
    x = x.view(-1, 16, 16, VQ_EMBED).permute(0, 3, 1, 2).contiguous()
    steps, i = _decoder(), 0

    def conv(t, name):
        y = _conv64(t, v[name + ".weight"])
        b = v.get(name + ".bias")
        return y if b is None else y + b.double().view(1, -1, 1, 1)

    def norm(t, name):
        return _gn_silu64(t, v[name + ".weight"], v[name + ".bias"])

    while i < len(steps):
        name, spec = steps[i]
        if spec[0] == "block":
            h = conv(norm(x, name + "norm0"), name + "conv0")
            h = conv(norm(h, name + "norm1"), name + "conv1")
            # a block that changes the width convolves its own output for the shortcut
            x = h + (x if spec[1] == spec[2] else conv(h, name + "conv_res"))
            i += 4 + (spec[1] != spec[2])
        elif spec[0] == "up":
            x = x.repeat_interleave(2, 2).repeat_interleave(2, 3)
        elif spec[0] == "norm":
            x = norm(x, name)
        else:
            x = conv(x, name)
        i += 1
    return x


def _forward64(tokens, values):
    v = {k: t.cuda() for k, t in values.items()}
    batch, seq = tokens.shape

    def w(name):
        n = v[name + ".bias"].numel()
        return _h(_dequantize("q8_0", v[name + ".weight"], n, v[name + ".weight"].shape[1] // 34 * 32))

    def b(name):
        return v[name + ".bias"].double()

    ids = torch.from_numpy(tokens).long().cuda().view(-1)
    x = v["token_embd.weight"].double()[ids] + v["pos_embd.weight"].double()[:seq].repeat(batch, 1)
    x = _ln64(x, v["token_embd_norm.weight"], v["token_embd_norm.bias"])
    for i in range(LAYERS):
        p = "blk.%d." % i
        qkv = [p + "attn_q", p + "attn_k", p + "attn_v"]
        ws = [torch.cat([w(n) for n in qkv])] + [w(p + n) for n in ("attn_o", "ffn_up", "ffn_down")]
        bs = [torch.cat([b(n) for n in qkv])] + [b(p + n) for n in ("attn_o", "ffn_up", "ffn_down")]
        norms = [v[p + n + e] for n in ("attn_norm", "ffn_norm") for e in (".weight", ".bias")]
        x = _layer64(x, ws, bs, *norms, batch)
    h = _gelu64(_h(x) @ w("output_proj").t() + b("output_proj"))
    h = _ln64(h, v["output_norm.weight"], v["output_norm.bias"])
    return (h @ v["token_embd.weight"].double().t() + v["output.bias"].double()).view(batch, seq, VOCAB)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "decode"):
        s = prepare(case, seed)
        values = _values(kind)[2]
        return _forward64(s["tokens"], values) if kind == "forward" else _decode64(s["grids"], values)
    s = prepare(case, seed)
    if kind == "layer":
        w = [_h(_dequantize(case["quant"], s["blocks%d" % i].cuda(), n, k)) for i, (n, k, _, _) in enumerate(FC4)]
        x = _layer64(s["x"].double(), w, [s["b%d" % i].double() for i in range(4)], s["gamma1"], s["beta1"], s["gamma3"],
                     s["beta3"], case["batch"])
        return {"x": x, "x16": x}
    if kind == "fc4":
        out = []
        for i, (n, k, act, resid) in enumerate(FC4):
            w = _dequantize(case["quant"], s["blocks%d" % i].cuda(), n, k)
            x = s["x%d" % i]
            y = (_codes64(x) @ w.t() if case["form"] == "int8" else _h(x) @ _h(w).t()) + s["b%d" % i].double()
            y = _gelu64(y) if act == 1 else y
            out.append(y + s["r%d" % i].double() if resid else y)
        return out
    if kind == "attn":
        q, k, v = _split_heads(_h(s["qkv"]), case["batch"], case["seq"], case["heads"], case["dim"])
        return _merge_heads(_attn64(q, k, v, case["dim"] ** -0.5))
    if kind == "head":
        return s["x"].double() @ s["w"].double().t() + s["b"].double()
    y = _conv64(s["x"], s["w"], kind == "conv_i8") + s["b"].double().view(1, -1, 1, 1)
    return y + s["r"].double() if case["resid"] else y
