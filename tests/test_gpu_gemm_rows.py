"""Dense linears of 33 to 192 rows on gemm_rows_kernel (all rows in one tile,
unsplit or split over K) against the int32 product of another kernel and the
separate dequant, bit for bit: the edges of the row blocks and of the rules
that choose the kernel, ragged N and K, bias, residual, SwiGLU and asymmetric
activations."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
EDGES = [33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193]


@pytest.fixture(scope="module")
def C():
    from signrot_amd import _CUDA
    return _CUDA


def _data(M, N, K):
    g = torch.Generator(DEV).manual_seed(M + N + K)
    a = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    b = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    sa = (torch.rand(M, device=DEV, generator=g) * 0.05 + 1e-3).half()
    sb = (torch.rand(N, device=DEV, generator=g) * 0.01 + 1e-4).half()
    bias = (torch.randn(N, device=DEV, generator=g) * 0.5).half()
    res = (torch.randn(M, N, device=DEV, generator=g) * 3).half()
    z = torch.randint(-8, 16, (M,), dtype=torch.int8, device=DEV, generator=g)
    return a, b, sa, sb, bias, res, z


# unsplit: 193 and 224 column tiles (one ragged), K of two ragged steps;
# split over K: 32, 40 (ragged), 64 and 9 tiles, even and ragged chunks
@pytest.mark.parametrize("N,K", [(24577, 288), (28672, 1024), (4096, 10272), (5099, 12288),
                                 (8192, 16416), (1032, 28672)])
@pytest.mark.parametrize("M", EDGES)
def test_rows_linear_bitexact(C, M, N, K):
    a, b, sa, sb, bias, res, z = _data(M, N, K)
    want = C.sym_dequant(C.matmul(a, b), sa, sb)
    assert torch.equal(C.w4a4_linear(a, sa, b, sb), want)
    assert torch.equal(C.w4a4_linear(a, sa, b, sb, bias), want + bias)
    inplace = res.clone()
    C.w4a4_linear_residual(a, sa, b, sb, inplace, bias, out=inplace)
    assert torch.equal(inplace, (want + bias) + res)
    wsum = C.sum_i4(b).view(-1)
    prod = C.matmul_ui4_si4(a, b) - z.int()[:, None] * wsum[None]
    assert torch.equal(C.w4a4_linear_asym(a, sa, z, b, sb, wsum, bias),
                       C.sym_dequant(prod, sa, sb) + bias)


# 97, 161 (ragged) and 224 column tiles
@pytest.mark.parametrize("N,K", [(12304, 544), (20496, 288), (28672, 1024)])
@pytest.mark.parametrize("M", EDGES)
def test_rows_swiglu_bitexact(C, M, N, K):
    a, b, sa, sb, *_ = _data(M, N, K)
    h = C.sym_dequant(C.matmul(a, b), sa, sb).view(M, N // 16, 2, 8)
    want = C.swiglu(h[:, :, 0].contiguous().view(M, N // 2), h[:, :, 1].contiguous().view(M, N // 2))
    assert torch.equal(C.w4a4_linear_swiglu(a, sa, b, sb), want)


def test_rows_split_small_workspace(C):
    """A workspace smaller than the split needs: the unsplit kernels, same bits."""
    from signrot_amd import _native
    M, N, K = 50, 4096, 14336
    a, b, sa, sb, *_ = _data(M, N, K)
    nbytes = int(_native.lib().srq_w4a4_linear_ws_bytes(M, N, K))
    assert nbytes > 0
    want = C.w4a4_linear(a, sa, b, sb)
    ws = torch.empty(nbytes - 16, dtype=torch.uint8, device=DEV)
    out = torch.empty(M, N, dtype=torch.float16, device=DEV)
    _native.call("srq_w4a4_linear_ws", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(),
                 None, M, N, K, out.data_ptr(), ws.data_ptr(), ws.numel(),
                 torch.cuda.current_stream().cuda_stream)
    assert torch.equal(out, want)
