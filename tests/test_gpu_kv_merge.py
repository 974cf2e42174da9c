"""The merge of the split decode attention's partial states at the edges of its
first batch of chunks (16) and of one chunk per thread (128)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


# chunk counts past the number of tokens leave empty chunks (m = -inf, d = 0)
@pytest.mark.parametrize("tokens,chunks", [(300, 2), (300, 15), (300, 16), (300, 17), (1, 33),
                                           (700, 128), (700, 129), (64, 1024)])
def test_merge_against_partial_states(tokens, chunks):
    from signrot_amd import _CUDA as C
    B, Hq, H, page = 2, 4, 2, 32
    g = torch.Generator("cuda").manual_seed(chunks)
    n = -(-tokens // page)
    data = torch.randint(0, 256, (B * n, 1, 2, H, page, D // 2), dtype=torch.uint8, device="cuda",
                         generator=g)
    param = torch.rand(B * n, 1, 2, H, page, 2, device="cuda", generator=g).half() * 0.2
    indptr = torch.arange(0, B * n + 1, n, dtype=torch.int32, device="cuda")
    indices = torch.arange(B * n, dtype=torch.int32, device="cuda")
    last = torch.full((B,), (tokens - 1) % page + 1, dtype=torch.int32, device="cuda")
    q = torch.randn(B, Hq, D, device="cuda", generator=g).half()
    tmp = torch.empty(B, Hq, chunks, D + 4, device="cuda")
    C.batch_decode_i4(None, q, data, param, indptr, indices, last, 0, tmp, chunks)
    rec = tmp.double()
    o = torch.empty_like(q)
    C.batch_decode_i4(o, q, data, param, indptr, indices, last, 0, tmp, chunks)
    m, d = rec[..., D], rec[..., D + 1]
    w = torch.exp2(m - m.amax(-1, keepdim=True))  # -inf: weight 0
    den = (d * w).sum(-1)[..., None]
    want = (rec[..., :D] * w[..., None]).sum(-2) / den
    # half an fp16 ulp (normal and subnormal), and the fp32 sums of `chunks`
    # terms with an exp2f of a few ulps each, on the sum of absolute terms
    mag = (rec[..., :D].abs() * w[..., None]).sum(-2) / den
    tol = want.abs() * 2.0 ** -11 + 2.0 ** -25 + (2 * chunks + 8) * 2.0 ** -24 * mag
    assert ((o.double() - want).abs() <= tol).all()
