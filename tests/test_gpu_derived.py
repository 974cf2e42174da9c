"""The interleaved gate/up weights that a decode step and the MoE block keep:
they follow the weights, a capture and other streams do not leave them
unwritten, and a copied module has its own."""
import copy
import pickle

import pytest
import torch
from test_gpu_prefill_fused import _cos_sin, _layer

pytestmark = pytest.mark.gpu

D, T, FFN = 128, 33, 896


def _decoder(inference=False):
    """(module, call, names of its gate/up buffers): a decode step from a
    synthetic context."""
    from signrot_amd.transformers import MultiLayerPagedKVCache4Bit
    layer = _layer(1024, 8, 2, FFN)
    h = torch.randn(2, 1, 1024, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    h = h.half()
    cos, sin = _cos_sin(1, T + 1, False)
    cos, sin = cos[:, T:].contiguous(), sin[:, T:].contiguous()
    caches = []

    def call(m):
        cache = MultiLayerPagedKVCache4Bit(2, 16, T + 1, "cuda", 1, 2, D, group_size=4)
        cache.pages.zero_().add_(37)
        cache.scales.zero_().add_(0.25)
        cache.mark_prefilled(T)
        cache.refresh_specs(T + 1)
        cache.freeze_specs(True)
        caches.append(cache)   # a captured step's buffers stay
        return lambda: m(h, cache, cos, sin)
    return layer, call, ("w_gu", "s_gu")


def _moe():
    from signrot_amd.nn import SignRotMoEBlock
    E, hidden, inter = 4, 256, 6144
    g = torch.Generator("cuda").manual_seed(3)
    u8 = lambda *s: torch.randint(0, 256, s, dtype=torch.uint8, device="cuda", generator=g)  # noqa: E731
    f16 = lambda *s: (torch.rand(s, device="cuda", generator=g) * 2e-3 + 1e-3).half()  # noqa: E731
    gate = torch.nn.Linear(hidden, E, bias=False, dtype=torch.float16, device="cuda")
    gate.requires_grad_(False).weight.copy_(torch.randn(E, hidden, device="cuda", generator=g))
    blk = SignRotMoEBlock(gate, top_k=2, norm_topk_prob=True, w_gate=u8(E, inter, hidden // 2),
                          s_gate=f16(E, inter), w_up=u8(E, inter, hidden // 2), s_up=f16(E, inter),
                          w_down=u8(E, hidden, inter // 2), s_down=f16(E, hidden))
    x = torch.randn(1, 24, hidden, device="cuda", generator=g).half()
    return blk, lambda m: (lambda: m(x)[0]), ("w_gate", "s_gate")


@pytest.fixture(params=[_decoder, _moe])
def made(request):
    module, call, names = request.param()
    with torch.no_grad():
        yield module, call, names, call(copy.deepcopy(module))()


def test_first_in_capture_then_eager(made):
    module, call, _, want = made
    step, eager = call(module), call(module)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    assert torch.equal(eager(), want)      # before the first replay
    for _ in range(3):
        graph.replay()
        assert torch.equal(out, want)
    assert torch.equal(eager(), want)


def test_follows_the_weights(made):
    module, call, (w, s), want = made
    step = call(module)
    assert torch.equal(step(), want)
    old = getattr(module, w).clone()
    getattr(module, w).copy_(old.flip(0))                   # in place
    changed = step()
    assert not torch.equal(changed, want)
    cur = getattr(module, w)                                # another tensor, same address
    fresh = cur.data                                        # and version
    fresh.copy_(old)
    while fresh._version < cur._version:
        fresh.add_(0)
    assert (fresh.data_ptr(), fresh._version) == (cur.data_ptr(), cur._version)
    module._buffers[w] = fresh
    assert torch.equal(step(), want)
    other = copy.deepcopy(module)                           # and copies of the module
    getattr(other, s).mul_(2)
    assert torch.equal(call(module)(), want) and not torch.equal(call(other)(), want)
    assert torch.equal(call(pickle.loads(pickle.dumps(module)))(), want)


def test_inference_mode_buffers(made):
    module, call, (w, s), want = made
    with torch.inference_mode():
        bufs = {n: b.clone() for n, b in module._buffers.items() if b is not None}
    for n, b in bufs.items():
        module._buffers[n] = b
    assert torch.equal(call(module)(), want)


def test_two_streams(made):
    module, call, _, want = made
    steps, outs = [call(module) for _ in range(2)], []
    torch.cuda.synchronize()
    for step in steps:
        with torch.cuda.stream(torch.cuda.Stream()):
            outs.append(step())
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)
