"""Large products on either side of the rule between 256 x 256 and 256 x 128
tiles, ragged in both directions: the fp16 linear (bias, residual), the int32
product and the SwiGLU form against row blocks of at most 32 rows, which
another kernel multiplies, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# (square, 256 x 128) tiles: (192, 384), (101, 201) ragged, (128, 256), (560, 1120)
@pytest.mark.parametrize("M,N", [(2048, 6144), (1030, 5121), (2048, 4096), (1200, 28672)])
def test_tile_rule_bitexact(M, N):
    from signrot_amd import _CUDA as C
    K = 544
    g = torch.Generator(DEV).manual_seed(M + N)
    a = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    b = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    sa = (torch.rand(M, device=DEV, generator=g) * 0.05 + 1e-3).half()
    sb = (torch.rand(N, device=DEV, generator=g) * 0.01 + 1e-4).half()
    bias = (torch.randn(N, device=DEV, generator=g) * 0.5).half()
    res = (torch.randn(M, N, device=DEV, generator=g) * 3).half()
    rows = [0, 255, 256, M // 2, M - 33]
    out = C.w4a4_linear(a, sa, b, sb, bias)
    outr = C.w4a4_linear_residual(a, sa, b, sb, res, bias)
    prod = C.matmul(a, b)
    for r in rows:
        s = slice(r, min(r + 32, M))
        part, ps = a[s].contiguous(), sa[s].contiguous()
        assert torch.equal(prod[s], C.matmul(part, b))
        want = C.w4a4_linear(part, ps, b, sb, bias)
        assert torch.equal(out[s], want)
        assert torch.equal(outr[s], want + res[s])
    if N % 16 == 0:
        sw = C.w4a4_linear_swiglu(a, sa, b, sb)
        for r in rows:
            s = slice(r, min(r + 32, M))
            assert torch.equal(sw[s], C.w4a4_linear_swiglu(a[s].contiguous(), sa[s].contiguous(),
                                                           b, sb))


# 516 square tiles (three rounds) against 1032 (five): square below K = 4096;
# 320 (two) against 640 (three): below 2048
@pytest.mark.parametrize("M,N,K", [(1281, 22016, 1024), (1281, 22016, 4064), (1281, 22016, 4096),
                                   (1100, 16384, 2016), (1100, 16384, 2048)])
def test_tile_rule_short_k(M, N, K):
    from signrot_amd import _CUDA as C
    g = torch.Generator(DEV).manual_seed(K)
    a = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    b = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    sa = (torch.rand(M, device=DEV, generator=g) * 0.05 + 1e-3).half()
    sb = (torch.rand(N, device=DEV, generator=g) * 0.01 + 1e-4).half()
    out, sw = C.w4a4_linear(a, sa, b, sb), C.w4a4_linear_swiglu(a, sa, b, sb)
    for r in (0, 1024, M - 32):
        part, ps = a[r:r + 32].contiguous(), sa[r:r + 32].contiguous()
        assert torch.equal(out[r:r + 32], C.w4a4_linear(part, ps, b, sb))
        assert torch.equal(sw[r:r + 32], C.w4a4_linear_swiglu(part, ps, b, sb))
