"""Prefill attention of short causal prompts (32-row blocks of 4 heads) against
float32 attention: lengths at the edges of tiles and of the rule that picks the
form, groups of 4 and 8, left padding down to one live token, strided inputs;
and the same bits whatever form a prompt's batch takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _ref(q, k, v, mask):
    B, T, Hq, _ = q.shape
    g = Hq // k.shape[2]
    out = torch.zeros(B, T, Hq, D, device="cuda")
    causal = torch.ones(T, T, dtype=torch.bool, device="cuda").tril()
    for b in range(B):
        ok = causal if mask is None else causal & (mask[b] != 0)[None, :]
        for h in range(Hq):
            s = q[b, :, h].float() @ k[b, :, h // g].float().T * D ** -0.5
            p = torch.softmax(s.masked_fill(~ok, -1e30), -1)
            o = p @ v[b, :, h // g].float()
            if mask is not None:
                o = o * (mask[b] != 0)[:, None]
            out[b, :, h] = o
    return out


# (8, 8) etc: query heads, KV heads.  32-row blocks, 64-key tiles, 128-key steps
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (16, 2), (32, 8), (4, 1)])
@pytest.mark.parametrize("B,T", [(1, 1), (1, 31), (2, 64), (1, 65), (1, 256), (1, 257), (2, 300),
                                 (1, 384), (1, 449), (3, 400), (1, 700), (1, 1025)])
@pytest.mark.parametrize("padded", [False, True])
def test_short_prompts(Hq, Hkv, B, T, padded):
    from signrot_amd import _CUDA as C
    gen = torch.Generator("cuda").manual_seed(T + Hq)
    heads = torch.randn(B, T, Hq + 2 * Hkv, D, device="cuda", generator=gen).half()
    q, k, v = heads.split((Hq, Hkv, Hkv), dim=2)   # strided views
    q = q * 2
    mask = None
    if padded:
        pad = torch.tensor([(7 * b + 1) * T // 9 for b in range(B)], device="cuda")
        pad[0] = T - 1                             # one live token
        mask = (torch.arange(T, device="cuda")[None] >= pad[:, None]).int()
    out = C.prefill_attention(q, k, v, mask).float()
    want = _ref(q, k, v, mask)
    # fp16 probabilities and outputs: 2^-11 relative each
    assert torch.allclose(out, want, rtol=4e-3, atol=4e-3)
    if mask is not None:
        assert torch.all(out[mask == 0] == 0)


# one prompt on its own, and among others that take it out of the rule for 32-row blocks
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (32, 8), (64, 8)])
@pytest.mark.parametrize("T", [1, 65, 128, 257, 300, 512, 700, 1024, 2048])
def test_same_bits_in_any_batch(Hq, Hkv, T):
    from signrot_amd import _CUDA as C
    gen = torch.Generator("cuda").manual_seed(T + Hq)
    B = 1 + 512 // (-(-T // 32) * (Hq // 4)) + 1
    q, k, v = (torch.randn(B, T, h, D, device="cuda", generator=gen).half()
               for h in (Hq, Hkv, Hkv))
    want = C.prefill_attention(q, k, v, None)
    for b in {0, B - 1}:
        got = C.prefill_attention(*(t[b:b + 1].contiguous() for t in (q, k, v)), None)
        assert torch.equal(got[0], want[b])
    # and with a mask that hides nothing
    ones = torch.ones(1, T, dtype=torch.int32, device="cuda")
    assert torch.equal(C.prefill_attention(q[:1], k[:1], v[:1], ones)[0], want[0])
