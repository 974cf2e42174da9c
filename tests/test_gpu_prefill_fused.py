"""The fused prefill of the decoder layer against its op-by-op path (which
test_gpu_prefill_layer.py checks against the oracle): the same hidden states
and cache bytes, bit for bit, with and without padding, at the edges of pages
and row blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _layer(hidden, Hq, Hkv, ffn):
    from signrot_amd.transformers.decode_layer import W4A4LlamaDecodeLayer
    return W4A4LlamaDecodeLayer.random(hidden, Hq, Hkv, D, ffn, seed=5)


def _cos_sin(B, T, per_request):
    from signrot_amd.transformers.decode_layer import rope_cos_sin
    if not per_request:
        return rope_cos_sin(range(T), D, 500000.0, "cuda")
    cs = [rope_cos_sin(range(3 * b, 3 * b + T), D, 500000.0, "cuda") for b in range(B)]
    return torch.cat([c for c, _ in cs]), torch.cat([s for _, s in cs])


def _run(layer, h, B, T, page, cos, sin, mask, trace):
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    cache = MultiLayerPagedKVCache4Bit(B, page, T, "cuda", 1, layer.n_kv, D,
                                       group_size=layer.n_heads // layer.n_kv)
    cache.pages.zero_()
    cache.scales.zero_()
    out = layer.prefill(h, cache, cos, sin, attention_mask=mask, trace=trace)
    return out, cache.pages, cache.scales


# heads whose rows split a wave between kinds (9 and 5 slots), one token, page
# edges, more rows than rmsnorm's per-row form takes
@pytest.mark.parametrize("B,T,Hq,Hkv,page", [(1, 1, 8, 2, 16), (3, 40, 8, 2, 32),
                                             (2, 33, 8, 1, 16), (1, 300, 16, 4, 64),
                                             (2, 64, 8, 8, 64)])
@pytest.mark.parametrize("per_request", [False, True])
def test_fused_prefill_bitexact(B, T, Hq, Hkv, page, per_request):
    hidden = Hq * D
    layer = _layer(hidden, Hq, Hkv, 896)
    h = torch.randn(B, T, hidden, device="cuda", generator=torch.Generator("cuda").manual_seed(T))
    h = h.half()
    cos, sin = _cos_sin(B, T, per_request)
    keep = h.clone()
    fused = _run(layer, h, B, T, page, cos, sin, None, None)
    ops = _run(layer, h, B, T, page, cos, sin, None, {})
    assert torch.equal(h, keep)
    for a, b, what in zip(fused, ops, ("hidden", "codes", "params")):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


def test_fused_prefill_masked_bitexact():
    B, T, page = 3, 40, 32
    layer = _layer(1024, 8, 2, 896)
    h = torch.randn(B, T, 1024, device="cuda").half()
    lens = torch.tensor([40, 33, 36], device="cuda")
    mask = (torch.arange(T, device="cuda")[None] >= (T - lens)[:, None]).int()
    cos, sin = _cos_sin(B, T, False)
    fused = _run(layer, h, B, T, page, cos, sin, mask, None)
    ops = _run(layer, h, B, T, page, cos, sin, mask, {})
    for a, b in zip(fused, ops):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_fused_prefill_refuses_a_filled_layer():
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    layer = _layer(1024, 8, 2, 896)
    cos, sin = _cos_sin(1, 8, False)
    cache = MultiLayerPagedKVCache4Bit(1, 16, 16, "cuda", 1, 2, D, group_size=4)
    h = torch.randn(1, 8, 1024, device="cuda").half()
    layer.prefill(h, cache, cos, sin)
    with pytest.raises(ValueError):
        layer.prefill(h, cache, cos, sin)
    assert cache.length == 8


def test_prefill_through_cache_adapter():
    """A cache that has only the HF methods takes the prefill too."""
    from signrot_amd.transformers import HFCacheAdapter, MultiLayerPagedKVCache4Bit
    T, layer = 33, _layer(1024, 8, 2, 896)
    h = torch.randn(1, T, 1024, device="cuda").half()
    cos, sin = _cos_sin(1, T, False)
    outs = []
    for wrap in (lambda c: c, HFCacheAdapter):
        cache = MultiLayerPagedKVCache4Bit(1, 16, T, "cuda", 1, 2, D, group_size=4)
        cache.pages.zero_()
        cache.scales.zero_()
        outs.append((layer.prefill(h, wrap(cache), cos, sin), cache.pages, cache.scales))
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _prefill(layer, h, cos, sin, **cache_kw):
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    B, T, _ = h.shape
    cache = MultiLayerPagedKVCache4Bit(B, 16, T, "cuda", 1, layer.n_kv, D,
                                       group_size=layer.n_heads // layer.n_kv, **cache_kw)
    return layer.prefill(h, cache, cos, sin)


def test_prefill_reads_the_weights_themselves():
    """A prefill keeps nothing of the weights: it follows a change that leaves
    the tensors' version counters alone, takes buffers that have none, and
    leaves no derived copy on the layer."""
    layer, T = _layer(1024, 8, 2, 896), 33
    h = torch.randn(1, T, 1024, device="cuda").half()
    cos, sin = _cos_sin(1, T, False)
    before = set(vars(layer))
    _prefill(layer, h, cos, sin)
    assert set(vars(layer)) == before
    layer.w_gu.data.copy_(layer.w_gu.flip(0))
    layer.s_gu.data.copy_(layer.s_gu.flip(0) * 2)
    got = _prefill(layer, h, cos, sin)
    fresh = _layer(1024, 8, 2, 896)
    fresh.load_state_dict(layer.state_dict())
    assert torch.equal(got, _prefill(fresh, h, cos, sin))
    with torch.inference_mode():
        inf = _layer(1024, 8, 2, 896)
        inf.load_state_dict(layer.state_dict())
    assert torch.equal(got, _prefill(inf, h, cos, sin))


def test_prefill_first_in_capture_then_eager():
    """The layer's first prefill recorded into a graph, an eager one before
    the first replay: each computes its own."""
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    layer, T = _layer(1024, 8, 2, 896), 64
    h = torch.randn(1, T, 1024, device="cuda").half()
    cos, sin = _cos_sin(1, T, False)
    want = _prefill(layer, h, cos, sin)
    new = _layer(1024, 8, 2, 896)
    cache = MultiLayerPagedKVCache4Bit(1, 16, T, "cuda", 1, 2, D, group_size=4)
    cache.refresh_specs(T)
    cache.freeze_specs(True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = new.prefill(h, cache, cos, sin)
    assert torch.equal(_prefill(new, h, cos, sin), want)
    for _ in range(3):
        graph.replay()
        assert torch.equal(out, want)


def test_refused_prefill_leaves_the_cache_alone():
    """A call that is refused for its cos / sin leaves the cache as it was: the
    corrected one then gives what a first call gives."""
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    layer, B, T = _layer(1024, 8, 2, 896), 2, 33
    h = torch.randn(B, T, 1024, device="cuda").half()
    cos, sin = _cos_sin(B, T, False)
    want = _run(layer, h, B, T, 16, cos, sin, None, None)
    cache = MultiLayerPagedKVCache4Bit(B, 16, T, "cuda", 1, 2, D, group_size=4)
    cache.pages.zero_()
    cache.scales.zero_()
    for c, s in ((cos.float(), sin.float()), (cos[:, 1:], sin[:, 1:]), (cos, sin[:, 1:]),
                 (cos.cpu(), sin.cpu()), (torch.cat([cos] * 3), torch.cat([sin] * 3))):
        with pytest.raises(RuntimeError):
            layer.prefill(h, cache, c, s)
        assert cache.length == 0 and not any(cache._filled)
    out = layer.prefill(h, cache, cos, sin)
    assert cache.length == T
    for a, b in zip((out, cache.pages, cache.scales), want):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_prefill_calls_what_is_put_in_place():
    """Hooks on a norm, another norm, a cache's own update() and gradients of
    the residual stream are seen by a prefill as by the op-by-op path."""
    from signrot_amd.nn.normalization import RMSNorm
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    T = 33
    h = torch.randn(1, T, 1024, device="cuda").half()
    cos, sin = _cos_sin(1, T, False)
    want = _prefill(_layer(1024, 8, 2, 896), h, cos, sin)

    for norm in ("input_layernorm", "post_attention_layernorm"):
        layer, seen = _layer(1024, 8, 2, 896), []
        getattr(layer, norm).register_forward_hook(lambda m, a, out: seen.append(out.shape))
        assert torch.equal(_prefill(layer, h, cos, sin), want) and len(seen) == 1
        layer = _layer(1024, 8, 2, 896)
        getattr(layer, norm).register_forward_pre_hook(lambda m, a: (a[0] * 0,))
        assert not torch.equal(_prefill(layer, h, cos, sin), want)
        layer = _layer(1024, 8, 2, 896)

        class Double(RMSNorm):
            def forward(self, x):
                return super().forward(x * 2) * 0 + super().forward(x)
        setattr(layer, norm, Double(1024))
        assert torch.equal(_prefill(layer, h, cos, sin), want)
        setattr(layer, norm, torch.nn.Identity())
        assert not torch.equal(_prefill(layer, h, cos, sin), want)
    layer, seen = _layer(1024, 8, 2, 896), []
    handle = torch.nn.modules.module.register_module_forward_hook(
        lambda m, a, out: seen.append(type(m)))
    try:
        assert torch.equal(_prefill(layer, h, cos, sin), want)
    finally:
        handle.remove()
    assert seen.count(RMSNorm) == 2

    calls = []

    class Own(MultiLayerPagedKVCache4Bit):
        def update(self, k, v, *a, **kw):
            calls.append(k.shape)
            return super().update(k, v, *a, **kw)
    cache = Own(1, 16, T, "cuda", 1, 2, D, group_size=4)
    assert torch.equal(layer.prefill(h, cache, cos, sin), want) and len(calls) == 1

    hg = h.clone().requires_grad_()
    out = _prefill(layer, hg, cos, sin)
    assert torch.equal(out, want) and out.requires_grad
    out.float().sum().backward()
    assert torch.equal(hg.grad, torch.ones_like(hg))   # through the residual adds


@pytest.mark.parametrize("dtype", [None, torch.float32])
def test_fused_prefill_key_rotations(dtype):
    """Caches whose keys are not rotated, or rotated in fp32."""
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    layer, B, T = _layer(1024, 8, 2, 896), 2, 40
    h = torch.randn(B, T, 1024, device="cuda").half()
    cos, sin = _cos_sin(B, T, True)
    outs = []
    for trace in (None, {}):
        cache = MultiLayerPagedKVCache4Bit(B, 16, T, "cuda", 1, 2, D, group_size=4,
                                           hadamard_dtype=dtype)
        cache.pages.zero_()
        cache.scales.zero_()
        outs.append((layer.prefill(h, cache, cos, sin, trace=trace), cache.pages, cache.scales))
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _wide_layer(hidden, Hq, Hkv, ffn):
    """Random codes straight on the GPU (random() draws the weights on the CPU)."""
    from signrot_amd.transformers.decode_layer import W4A4LlamaDecodeLayer
    layer = W4A4LlamaDecodeLayer(hidden, Hq, Hkv, D, ffn).to("cuda")
    g = torch.Generator("cuda").manual_seed(7)
    for name in ("qkv", "o", "gu", "down"):
        w, s = getattr(layer, f"w_{name}"), getattr(layer, f"s_{name}")
        w.copy_(torch.randint(0, 256, w.shape, dtype=torch.uint8, device="cuda", generator=g))
        s.copy_(torch.rand(s.shape, device="cuda", generator=g) * 2e-3 + 1e-3)
    layer.down_sign.copy_(torch.randint(0, 2, (ffn,), device="cuda", generator=g) * 2 - 1)
    return layer


# 8B widths; an FFN of 172 x 64, whose rotation has no SwiGLU form
@pytest.mark.parametrize("ffn", [14336, 11008])
@pytest.mark.parametrize("B,T,padded", [(1, 300, False), (2, 130, True), (1, 2048, False)])
def test_fused_prefill_model_widths(ffn, B, T, padded):
    layer = _wide_layer(4096, 32, 8, ffn)
    h = torch.randn(B, T, 4096, device="cuda", generator=torch.Generator("cuda").manual_seed(T))
    cos, sin = _cos_sin(B, T, False)
    mask = None
    if padded:
        pad = torch.tensor([[0], [37]], device="cuda")
        mask = (torch.arange(T, device="cuda")[None] >= pad).int()
    fused = _run(layer, h.half(), B, T, 256, cos, sin, mask, None)
    ops = _run(layer, h.half(), B, T, 256, cos, sin, mask, {})
    for a, b, what in zip(fused, ops, ("hidden", "codes", "params")):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), what


def test_prefill_from_two_streams():
    """One layer, a cache per request, first prefills from two streams at once."""
    layer, T = _wide_layer(4096, 32, 8, 14336), 512
    hs = [torch.randn(1, T, 4096, device="cuda").half() for _ in range(2)]
    cos, sin = _cos_sin(1, T, False)
    torch.cuda.synchronize()
    streams, outs = [torch.cuda.Stream() for _ in hs], []
    for h, s in zip(hs, streams):
        with torch.cuda.stream(s):
            outs.append(_prefill(layer, h, cos, sin))
    torch.cuda.synchronize()
    for h, out in zip(hs, outs):
        assert torch.equal(out, _prefill(layer, h, cos, sin))


def test_prefill_refuses_other_key_rotations():
    """A key rotation in a type that the Hadamard kernel has not is refused by
    a prefill, and nothing comes into the cache."""
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    layer, T = _layer(1024, 8, 2, 896), 8
    cos, sin = _cos_sin(1, T, False)
    h = torch.randn(1, T, 1024, device="cuda").half()
    cache = MultiLayerPagedKVCache4Bit(1, 16, T, "cuda", 1, 2, D, group_size=4,
                                       hadamard_dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="only float16 and float32"):
        layer.prefill(h, cache, cos, sin)
    assert cache.length == 0 and not any(cache._filled)
