"""Performance cases of the W4A4 real-quant path: what a program that serves a
quantized Llama-style model calls, each through a public entry point.

Kinds of case, and what each stands for in use:

  qlinear            one down_proj / q_proj as a model runs it: the online
                     Hadamard rotation with its sign, the per-token quantizer
                     and the int4 linear, from one token (decode) to a prompt
                     (prefill), symmetric or asymmetric activations
  mlp                a gate/up + SwiGLU + down block (70B widths)
  moe                a sparse feed-forward block (8 experts, top 2), a decode
                     batch or a prompt
  decode_attention   one query token per request over the paged int4 cache,
                     requests of different lengths
  decode_layer       one whole decoder layer of a decode step, replayed as the
                     HIP graph that a serving loop captures
  prefill_attention  causal attention of a prompt over fp16 q/k/v
  prefill_layer      a decoder layer's first update: a prompt through
                     projections, cache fill, attention and MLP

Sizes are those of the benchmark's configurations and of the tests (hidden
4096 / 8192, FFN 14336 / 28672 / 11008 / 13824, 32/8 and 64/8 heads), with
token counts over the whole range, odd ones among them.  Weights are on a
real int4 grid: N(0, 0.02) rounded to about 1.75 steps of deviation.
Activations before a rotation are N(0, 1) with a few outlier channels, the
hidden states of a rotated model plain N(0, 1).
"""
import json
import math
import pathlib

import torch

from signrot_amd import _CUDA
from signrot_amd.nn import (AsymQuantizer, HadamardQuantizer, Linear4bit, OnlineHadamard,
                            Quantizer, SignRotMoEBlock)
from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
from signrot_amd.transformers.decode_layer import W4A4LlamaDecodeLayer, rope_cos_sin

DEV = "cuda"
D = 128                       # head dim
W_STD, W_STEPS = 0.02, 1.75   # weight deviation, and in int4 steps
LAYER = dict(hidden=4096, heads=32, kv_heads=8, ffn=14336)   # 8B widths
PAGE = 256


def listed():
    return [
        # one decode token through a down_proj: the smallest call, launches count
        dict(name="qlinear_m1", kind="qlinear", m=1, k=14336, n=4096, asym=False),
        # a small decode batch through a projection with a power-of-two rotation
        dict(name="qlinear_m16_pow2", kind="qlinear", m=16, k=4096, n=4096, asym=False),
        # a short, odd prompt through the down_proj of an FFN of 11008 = 172 x 64
        dict(name="qlinear_m137_ffn11008", kind="qlinear", m=137, k=11008, n=4096, asym=False),
        # a prompt of 2048 tokens through the same layer of an FFN of 14336
        dict(name="qlinear_m2048", kind="qlinear", m=2048, k=14336, n=4096, asym=False),
        # asymmetric activations (uint4 codes and zero points), an odd prompt
        dict(name="qlinear_asym_m1000", kind="qlinear", m=1000, k=14336, n=4096, asym=True),
        # the feed-forward block at 70B widths, a prompt of 512 tokens
        dict(name="mlp_m512", kind="mlp", m=512, hidden=8192, ffn=28672),
        # sparse feed-forward: a prompt, and a decode batch that reaches every expert
        dict(name="moe_t512", kind="moe", m=512, asym=False),
        dict(name="moe_t24", kind="moe", m=24, asym=False),
        # decode attention alone: 8 requests of uneven lengths, 64 / 8 heads
        dict(name="decode_attention_b8", kind="decode_attention", batch=8, length=7000, heads=64,
             kv_heads=8),
        # a decoder layer of a decode step: 32 requests with 4096 cached tokens
        dict(name="decode_layer_b32", kind="decode_layer", batch=32, length=4096),
        # attention of a 2048-token prompt, 64 / 8 heads
        dict(name="prefill_attention_t2048", kind="prefill_attention", batch=1, length=2048,
             heads=64, kv_heads=8, padded=False),
        # a decoder layer's first update: a prompt of 2048 tokens
        dict(name="prefill_layer_t2048", kind="prefill_layer", batch=1, length=2048),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["qlinear", "qlinear", "qlinear", "mlp", "moe", "decode_attention",
                       "decode_layer", "prefill_attention", "prefill_layer"])
    if kind == "qlinear":
        k, n, top = rng.choice([(4096, 4096, 2048), (14336, 4096, 2048), (11008, 4096, 2048),
                                (13824, 5120, 2048), (28672, 8192, 768)])
        return dict(kind=kind, m=_log_int(rng, 1, top), k=k, n=n, asym=rng.random() < 0.35)
    if kind == "mlp":
        hidden, ffn, top = rng.choice([(4096, 14336, 1024), (8192, 28672, 512)])
        return dict(kind=kind, m=_log_int(rng, 1, top), hidden=hidden, ffn=ffn)
    if kind == "moe":
        return dict(kind=kind, m=_log_int(rng, 4, 512), asym=rng.random() < 0.25)
    if kind == "decode_attention":
        heads, kv_heads = rng.choice([(32, 8), (64, 8), (32, 32)])
        length = _log_int(rng, 200, 8192)
        return dict(kind=kind, batch=_log_int(rng, 1, max(1, min(48, 120000 // length))),
                    length=length, heads=heads, kv_heads=kv_heads)
    if kind == "decode_layer":
        return dict(kind=kind, batch=_log_int(rng, 1, 32), length=_log_int(rng, 256, 4096))
    if kind == "prefill_attention":
        heads, kv_heads = rng.choice([(32, 8), (64, 8)])
        return dict(kind=kind, batch=rng.choice([1, 1, 2]), length=_log_int(rng, 200, 3000),
                    heads=heads, kv_heads=kv_heads, padded=rng.random() < 0.4)
    return dict(kind=kind, batch=1, length=_log_int(rng, 100, 2000))


# ----------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _codes(g, rows, cols):
    """int4 codes u8 [rows, cols / 2] of weights N(0, W_STD)."""
    c = (torch.randn(rows, cols, device=DEV, generator=g) * W_STEPS).round_().clamp_(-8, 7)
    c = c.to(torch.int8).view(torch.uint8) & 15
    return c[:, 0::2] | (c[:, 1::2] << 4)


def _weight(g, rows, cols, std=W_STD):
    s = (torch.rand(rows, device=DEV, generator=g) * 0.4 + 0.8) * (std / W_STEPS)
    return _codes(g, rows, cols), s.half()


def _acts(g, rows, cols, outliers=8, mag=50.0):
    x = torch.randn(rows, cols, device=DEV, generator=g)
    if outliers:
        ch = torch.randperm(cols, device=DEV, generator=g)[:outliers]
        sg = torch.randint(0, 2, (outliers,), device=DEV, generator=g) * 2 - 1
        x[:, ch] *= sg * mag
    return x.half()


def _sign(g, *shape):
    return (torch.randint(0, 2, shape, device=DEV, generator=g) * 2 - 1).to(torch.int8)


def _inputs(case, seed):
    """The tensors of a case, from the seed alone: shared by prepare() and
    exact()."""
    g, kind = _gen(seed), case["kind"]
    if kind == "qlinear":
        m, k, n = case["m"], case["k"], case["n"]
        x = _acts(g, m, k)
        if case["asym"]:
            x = x + 0.5
        return dict(x=x, sign=_sign(g, k), w=_weight(g, n, k))
    if kind == "mlp":
        h, f = case["hidden"], case["ffn"]
        return dict(x=_acts(g, case["m"], h, outliers=0), sign=_sign(g, f), gu=_weight(g, 2 * f, h),
                    down=_weight(g, h, f))
    if kind == "moe":
        e, h, f = 8, 4096, 14336
        t = dict(x=_acts(g, case["m"], h, outliers=0).view(1, case["m"], h),
                 gate=(torch.randn(e, h, device=DEV, generator=g) / math.sqrt(h)).half(),
                 sign=_sign(g, e, f))
        for name, rows, cols in (("gate_w", f, h), ("up_w", f, h), ("down_w", h, f)):
            ws = [_weight(g, rows, cols) for _ in range(e)]
            t[name] = (torch.stack([w for w, _ in ws]), torch.stack([s for _, s in ws]))
        return t
    if kind == "decode_attention":
        b, length, hk = case["batch"], case["length"], case["kv_heads"]
        lens = torch.randint(max(1, length // 2), length + 1, (b,), device=DEV, generator=g)
        lens[0] = length
        pages = (lens + PAGE - 1) // PAGE
        total = int(pages.sum())
        indptr = torch.zeros(b + 1, dtype=torch.int32, device=DEV)
        indptr[1:] = torch.cumsum(pages, 0)
        data, param = _kv_pool(g, total, hk)
        return dict(q=torch.randn(b, case["heads"], D, device=DEV, generator=g).half(),
                    kv_data=data, kv_param=param, kv_indptr=indptr,
                    kv_indices=torch.randperm(total, device=DEV, generator=g).int(),
                    last_page_offset=((lens - 1) % PAGE + 1).int(), lens=lens)
    if kind == "prefill_attention":
        b, t = case["batch"], case["length"]
        q = torch.randn(b, t, case["heads"], D, device=DEV, generator=g).half()
        k = torch.randn(b, t, case["kv_heads"], D, device=DEV, generator=g).half()
        v = torch.randn(b, t, case["kv_heads"], D, device=DEV, generator=g).half()
        mask = None
        if case["padded"]:   # left padding, as a batch of prompts has it
            pad = torch.randint(0, t // 4 + 1, (b, 1), device=DEV, generator=g)
            mask = (torch.arange(t, device=DEV)[None, :] >= pad).int()
        return dict(q=q, k=k, v=v, mask=mask)
    # decoder layers
    h, f = LAYER["hidden"], LAYER["ffn"]
    # the projections that write to the residual stream are initialised smaller
    # by sqrt(2 x 32 layers), and the stream itself has grown over some layers
    t = dict(qkv=_weight(g, (LAYER["heads"] + 2 * LAYER["kv_heads"]) * D, h),
             o=_weight(g, h, h, W_STD / 8), gu=_weight(g, 2 * f, h),
             down=_weight(g, h, f, W_STD / 8), sign=_sign(g, f))
    b, length = case["batch"], case["length"]
    tokens = 1 if kind == "decode_layer" else length
    t["h"] = (4 * torch.randn(b, tokens, h, device=DEV, generator=g)).half()
    if kind == "decode_layer":
        t["pages"], t["scales"] = _kv_pool(g, b * (-(-(length + 1) // PAGE)), LAYER["kv_heads"])
    return t


def _kv_pool(g, pages, kv_heads):
    """A random int4 context: codes, and per token [scale, zero]."""
    data = torch.randint(0, 256, (pages, 1, 2, kv_heads, PAGE, D // 2), dtype=torch.uint8,
                         device=DEV, generator=g)
    param = torch.empty(pages, 1, 2, kv_heads, PAGE, 2, dtype=torch.float16, device=DEV)
    param[..., 0].uniform_(0.2, 0.4, generator=g)       # 15 steps over about +-2.3
    param[..., 1] = param[..., 0] * 7.5
    return data, param


# ---------------------------------------------------------------- prepare

def _rotation(k, sign, quantizer):
    had = OnlineHadamard(k, had_adj=True).to(DEV)
    had.had_adj_sign.copy_(sign)
    return HadamardQuantizer(had, quantizer)


def _linear(w):
    codes, scales = w
    lin = Linear4bit(codes.shape[1] * 2, codes.shape[0])
    lin.weight, lin.weight_scales = codes, scales.view(-1, 1)
    return lin


def _layer(t):
    layer = W4A4LlamaDecodeLayer(LAYER["hidden"], LAYER["heads"], LAYER["kv_heads"], D,
                                 LAYER["ffn"]).to(DEV)
    for name in ("qkv", "o", "gu", "down"):
        codes, scales = t[name]
        setattr(layer, f"w_{name}", codes)
        setattr(layer, f"s_{name}", scales)
    layer.down_sign.copy_(t["sign"])
    return layer


def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "qlinear":
        quantizer = AsymQuantizer() if case["asym"] else Quantizer()
        mod = torch.nn.Sequential(_rotation(case["k"], t["sign"], quantizer), _linear(t["w"]))
        return dict(kind=kind, x=t["x"], mod=mod)
    if kind == "mlp":
        gu, s_gu = _CUDA.interleave_gate_up(*t["gu"], case["ffn"])
        return dict(kind=kind, x=t["x"], quant=Quantizer(), gu=gu, s_gu=s_gu,
                    down=torch.nn.Sequential(_rotation(case["ffn"], t["sign"], Quantizer()),
                                             _linear(t["down"])))
    if kind == "moe":
        gate = torch.nn.Linear(t["gate"].shape[1], t["gate"].shape[0], bias=False,
                               dtype=torch.float16, device=DEV).requires_grad_(False)
        gate.weight.copy_(t["gate"])
        blk = SignRotMoEBlock(gate, top_k=2, norm_topk_prob=True,
                              w_gate=t["gate_w"][0], s_gate=t["gate_w"][1],
                              w_up=t["up_w"][0], s_up=t["up_w"][1],
                              w_down=t["down_w"][0], s_down=t["down_w"][1],
                              sign_down=t["sign"], asym=case["asym"]).eval()
        return dict(kind=kind, x=t["x"], blk=blk)
    if kind == "decode_attention":
        b, hq, hk = case["batch"], case["heads"], case["kv_heads"]
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        chunks = MultiLayerPagedKVCache4Bit.decode_chunks(b, hk, case["length"], cus)
        tmp = torch.empty(b, hq, chunks, D + 4, device=DEV) if chunks > 1 else None
        t.pop("lens")
        return dict(kind=kind, o=torch.empty_like(t["q"]), tmp=tmp, chunks=chunks, **t)
    if kind == "prefill_attention":
        return dict(kind=kind, **t)
    layer, b, length = _layer(t), case["batch"], case["length"]
    cache = MultiLayerPagedKVCache4Bit(b, PAGE, length + 1, DEV, 1, LAYER["kv_heads"], D,
                                       group_size=LAYER["heads"] // LAYER["kv_heads"])
    if kind == "prefill_layer":
        cache.pages.zero_()
        cache.scales.zero_()
        cos, sin = rope_cos_sin(range(length), D, layer.rope_theta, DEV)
        return dict(kind=kind, layer=layer, cache=cache, cos=cos, sin=sin, h=t["h"])
    cache.pages.copy_(t["pages"])
    cache.scales.copy_(t["scales"])
    cache.mark_prefilled(length)
    cos, sin = rope_cos_sin([length], D, layer.rope_theta, DEV)
    # the graph protocol: index buffers refreshed outside, frozen inside
    cache.refresh_specs(length + 1)
    cache.freeze_specs(True)

    def step():
        cache.length = length
        return layer(t["h"], cache, cos, sin)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return dict(kind=kind, layer=layer, cache=cache, graph=graph, out=out, keep=(t["h"], cos, sin))


# -------------------------------------------------------------------- run

@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "qlinear":
        return s["mod"](s["x"])
    if kind == "mlp":
        xq = s["quant"](s["x"])
        a = _CUDA.w4a4_linear_swiglu(xq.quantized_x, xq.scales_x.view(-1), s["gu"], s["s_gu"])
        return s["down"](a)
    if kind == "moe":
        out, logits = s["blk"](s["x"])
        return dict(out=out, logits=logits)
    if kind == "decode_attention":
        _CUDA.batch_decode_i4(s["o"], s["q"], s["kv_data"], s["kv_param"], s["kv_indptr"],
                              s["kv_indices"], s["last_page_offset"], 0, s["tmp"], s["chunks"])
        return s["o"]
    if kind == "prefill_attention":
        return _CUDA.prefill_attention(s["q"], s["k"], s["v"], s["mask"])
    if kind == "prefill_layer":
        s["cache"].reset()
        out = s["layer"].prefill(s["h"], s["cache"], s["cos"], s["sin"])
        return dict(out=out, pages=s["cache"].pages, scales=s["cache"].scales)
    s["graph"].replay()
    return dict(out=s["out"], pages=s["cache"].pages, scales=s["cache"].scales)


# ------------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    if kind == "qlinear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=2 * m * k + n * k // 2 + 2 * n + k + 2 * m * n, flops=2 * m * n * k)
    if kind == "mlp":
        m, h, f = case["m"], case["hidden"], case["ffn"]
        return dict(bytes=3 * f * h // 2 + 4 * m * h + 4 * f + 2 * h + f, flops=6 * m * h * f)
    if kind == "moe":
        m, h, f = case["m"], 4096, 14336
        experts = min(8, 2 * m)
        return dict(bytes=experts * 3 * f * h // 2 + 4 * m * h, flops=2 * 6 * m * h * f)
    if kind == "decode_attention":
        tokens = case["batch"] * 0.75 * case["length"]
        return dict(bytes=int(tokens * case["kv_heads"] * 2 * (D // 2 + 4))
                    + 4 * case["batch"] * case["heads"] * D,
                    flops=int(4 * tokens * case["heads"] * D))
    if kind == "prefill_attention":
        b, t = case["batch"], case["length"]
        return dict(bytes=2 * b * t * D * (2 * case["heads"] + 2 * case["kv_heads"]),
                    flops=2 * b * case["heads"] * D * t * (t + 1))
    h, f, hq, hk = (LAYER[n] for n in ("hidden", "ffn", "heads", "kv_heads"))
    wts = (hq + 2 * hk) * D * h + h * h + 3 * f * h
    b, t = case["batch"], case["length"]
    rows = b if kind == "decode_layer" else b * t
    kv = b * t * hk * 2 * (D // 2 + 4)
    att = 4 * b * hq * D * t if kind == "decode_layer" else 2 * b * hq * D * t * (t + 1)
    return dict(bytes=wts // 2 + kv + 4 * rows * h, flops=2 * rows * wts + att)


def tolerance(case):
    """Codes are rounded to 4 bits after fp16 rotations and norms: another
    correct order of those sums moves a value over a rounding edge in a few
    cases of a thousand, by a whole step each, which shows as about one per
    cent of a linear's output against 64 bits.  Attention over fp16 inputs
    has no such edges."""
    kind = case["kind"]
    if kind in ("decode_attention", "prefill_attention"):
        return {"rel": 3e-3, "max": 0.03}
    return {"rel": 0.03, "max": 0.5, "differ": 0.01}


# ------------------------------------------------------------------ exact
# 64 bits between the points where the path's own definition rounds to fp16:
# the tensors that pass from one step to the next, scales, and the quotients
# that become codes.

def _f16(x):
    return x.half().double()


def _had(k):
    path = pathlib.Path("signrot_amd/functional/had_tables.json").resolve()
    rows = json.loads(path.read_text())[str(k)]
    bits = torch.tensor([[(int(r, 16) >> j) & 1 for j in range(k)] for r in rows],
                        dtype=torch.float64, device=DEV)
    return bits * 2 - 1


def _fwht(x):
    shape, n, s = x.shape, x.shape[-1], 1
    while s < n:
        x = x.view(-1, n // (2 * s), 2, s)
        x = torch.stack((x[:, :, 0] + x[:, :, 1], x[:, :, 0] - x[:, :, 1]), 2)
        s *= 2
    return x.reshape(shape)


def _rotate(x, k_factor):
    n = x.shape[-1]
    y = x.double().view(-1, k_factor, n // k_factor)
    y = _fwht(y)
    if k_factor > 1:
        y = _had(k_factor) @ y
    return _f16(y.reshape(x.shape) / math.sqrt(n))


K_FACTOR = {4096: 1, 14336: 28, 28672: 28, 11008: 172, 13824: 108}


def _unpack(w):
    c = torch.stack((w & 15, w >> 4), -1).flatten(-2).double()
    return torch.where(c >= 8, c - 16, c)


def _quant(x):
    s = _f16(x.abs().amax(-1, keepdim=True) / 7)
    return _f16(x / s).round().clamp(-8, 7), s


def _matmul_w(x, w, quant=_quant):
    q, s = quant(x)
    return (q @ _unpack(w[0]).T) * s * w[1].double()


def _linear_asym(x, w):
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    s = _f16(_f16(hi - lo) / 15)
    z = _f16(-lo / s).round()
    q = (_f16(x / s).round() + z).clamp(0, 15)
    return ((q - z) @ _unpack(w[0]).T) * s * w[1].double()


def _swiglu(gate, up):
    gate, up = _f16(gate), _f16(up)
    return _f16(_f16(gate * torch.sigmoid(gate)) * up)


def _norm(x):
    return _f16(x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5))


def _rope(x, cos, sin):
    half = D // 2
    return _f16(_f16(x * cos) + _f16(torch.cat((-x[..., half:], x[..., :half]), -1) * sin))


def _attend(q, k, v, mask=None, causal=False):
    """[T, D] queries of one head over [S, D] keys."""
    s = q @ k.T / math.sqrt(D)
    if causal:
        s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
    if mask is not None:
        s = s.masked_fill(mask[None, :] == 0, -math.inf)
    return torch.softmax(s, -1) @ v


def _cached(data, param, pages, length):
    """K and V [2, Hk, length, D] of one request's pages."""
    codes = data[pages, 0].permute(1, 2, 0, 3, 4).flatten(2, 3)[:, :, :length]
    prm = param[pages, 0].permute(1, 2, 0, 3, 4).flatten(2, 3)[:, :, :length].double()
    c = torch.stack((codes & 15, codes >> 4), -1).flatten(-2).double()
    return c * prm[..., :1] - prm[..., 1:]


def _kv_round(x):
    """The value that the int4 cache gives back for x."""
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    s = _f16(_f16(hi - lo).clamp_min(1e-5) / 15)
    return _f16(_f16(x - lo) / s).round().clamp(0, 15) * s + lo


def _exact_layer(t, case):
    h, f, hq, hk = (LAYER[n] for n in ("hidden", "ffn", "heads", "kv_heads"))
    b, length = case["batch"], case["length"]
    decode = case["kind"] == "decode_layer"
    tok = 1 if decode else length
    x = t["h"].double().view(b * tok, h)
    qkv = _f16(_matmul_w(_norm(x), t["qkv"])).view(b, tok, hq + 2 * hk, D)
    pos = torch.arange(length, length + 1) if decode else torch.arange(length)
    freq = pos.float()[:, None] / (500000.0 ** (torch.arange(0, D, 2).float() / D))[None]
    freq = torch.cat((freq, freq), -1).to(DEV)
    cos, sin = freq.cos().half().double()[:, None], freq.sin().half().double()[:, None]
    q, k, v = qkv[:, :, :hq], qkv[:, :, hq:hq + hk], qkv[:, :, hq + hk:]
    q, k = _rope(q, cos, sin), _rope(k, cos, sin)
    att = torch.empty(b, tok, hq, D, dtype=torch.float64, device=DEV)
    if decode:
        q, k = _rotate(q, 1), _rotate(k, 1)
        per = -(-(length + 1) // PAGE)
        for i in range(b):
            pages = torch.arange(per, device=DEV) * b + i
            kc, vc = _cached(t["pages"], t["scales"], pages, length)
            for j in range(hk):
                kk = torch.cat((kc[j], _kv_round(k[i, :, j])))
                vv = torch.cat((vc[j], _kv_round(v[i, :, j])))
                g = hq // hk
                att[i, 0, j * g:(j + 1) * g] = _attend(q[i, 0, j * g:(j + 1) * g], kk, vv)
    else:
        for i in range(b):
            for j in range(hq):
                g = j * hk // hq
                att[i, :, j] = _attend(q[i, :, j], k[i, :, g], v[i, :, g], causal=True)
    rot = _rotate(_f16(att).transpose(-1, -2).contiguous(), 1).transpose(-1, -2).reshape(b * tok, h)
    x = _f16(x + _f16(_matmul_w(rot, t["o"])))
    gu = _matmul_w(_norm(x), t["gu"])
    a = _swiglu(gu[:, :f], gu[:, f:])
    x = x + _matmul_w(_rotate(a, K_FACTOR[f]) * t["sign"].double(), t["down"])
    return dict(out=x.view(b, tok, h), pages=None, scales=None)


@torch.no_grad()
def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "qlinear":
        x = _rotate(t["x"], K_FACTOR[case["k"]]) * t["sign"].double()
        return _linear_asym(x, t["w"]) if case["asym"] else _matmul_w(x, t["w"])
    if kind == "mlp":
        gu = _matmul_w(t["x"].double(), t["gu"])
        f = case["ffn"]
        a = _swiglu(gu[:, :f], gu[:, f:])
        return _matmul_w(_rotate(a, K_FACTOR[f]) * t["sign"].double(), t["down"])
    if kind == "moe":
        linear = _linear_asym if case["asym"] else _matmul_w
        x = t["x"][0].double()
        # the router's logits are fp16 by its interface
        logits = (x @ t["gate"].double().T).half()
        top, idx = torch.softmax(logits.double(), -1).topk(2, -1)
        top = (top / top.sum(-1, keepdim=True)).half().double()
        out = torch.zeros_like(x)
        for e in range(8):
            tok, choice = (idx == e).nonzero(as_tuple=True)
            if tok.numel() == 0:
                continue
            w = [(t[n][0][e], t[n][1][e]) for n in ("gate_w", "up_w", "down_w")]
            a = _swiglu(linear(x[tok], w[0]), linear(x[tok], w[1]))
            a = _rotate(a, 28) * t["sign"][e].double()
            out.index_add_(0, tok, linear(a, w[2]) * top[tok, choice, None])
        return dict(out=out.view(t["x"].shape), logits=logits.double())
    if kind == "decode_attention":
        out = torch.empty(t["q"].shape, dtype=torch.float64, device=DEV)
        g = case["heads"] // case["kv_heads"]
        ptr = t["kv_indptr"].tolist()
        for i, length in enumerate(t["lens"].tolist()):
            pages = t["kv_indices"][ptr[i]:ptr[i + 1]].long()
            k, v = _cached(t["kv_data"], t["kv_param"], pages, length)
            for j in range(case["kv_heads"]):
                out[i, j * g:(j + 1) * g] = _attend(t["q"][i, j * g:(j + 1) * g].double(), k[j],
                                                    v[j])
        return out
    if kind == "prefill_attention":
        q, k, v, mask = t["q"].double(), t["k"].double(), t["v"].double(), t["mask"]
        out = torch.zeros_like(q)
        for i in range(case["batch"]):
            first = 0 if mask is None else int((mask[i] == 0).sum())
            for j in range(case["heads"]):
                n = j * case["kv_heads"] // case["heads"]
                out[i, first:, j] = _attend(q[i, first:, j], k[i, first:, n], v[i, first:, n],
                                            causal=True)
        return out
    return _exact_layer(t, case)
