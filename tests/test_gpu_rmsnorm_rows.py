"""RMSNorm + quantizer on both sides of the block-per-row rule (256 rows, 2048
columns): the fused codes are those of the quantizer over the norm's output,
and the norm is within fp16 rounding of 64 bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 255, 256, 301])
@pytest.mark.parametrize("cols", [8, 512, 2040, 2048, 2056, 4104, 8192])
def test_rmsnorm_quant_rows(rows, cols):
    from signrot_amd import _CUDA
    g = torch.Generator("cuda").manual_seed(rows * 8192 + cols)
    x = (3 * torch.randn(rows, cols, device="cuda", generator=g)).half()
    eps = 1e-5
    n = _CUDA.rmsnorm(x, eps, cols)
    xd = x.double()
    want = xd / ((xd * xd).sum(-1, keepdim=True) / cols + eps).sqrt()
    # half an fp16 ulp of rounding and a few fp32 ones of the sum: one ulp
    ulp = 2.0 ** (torch.floor(torch.log2(want.abs().clamp_min(2.0 ** -14))) - 10)
    assert bool(((n.double() - want).abs() <= ulp).all())
    q, s = _CUDA.rmsnorm_quant(x, eps, cols)
    qw, sw = _CUDA.sym_quant_dynamic(n)
    assert torch.equal(q, qw) and torch.equal(s, sw)


def _lane_order_norm(x, eps, waves):
    """rmsnorm with its fp32 sum in the kernel's order: a row over 64 * waves
    lanes in vectors of 8, a lane's squares one after the other (each exact in
    fp32), then halves added lane by lane, then the waves pairwise."""
    rows, cols = x.shape
    lanes = 64 * waves
    f = np.zeros((rows, -(-cols // (8 * lanes)) * 8 * lanes), np.float32)
    f[:, :cols] = x.astype(np.float32)
    f = f.reshape(rows, -1, lanes, 8)
    acc = np.zeros((rows, lanes), np.float32)
    for i in range(f.shape[1]):
        for e in range(8):
            acc = acc + f[:, i, :, e] * f[:, i, :, e]
    acc = acc.reshape(rows, waves, 64)
    while acc.shape[2] > 1:
        h = acc.shape[2] // 2
        acc = acc[:, :, :h] + acc[:, :, h:]
    acc = acc[:, :, 0]
    while acc.shape[1] > 1:
        acc = acc[:, 0::2] + acc[:, 1::2]
    inv = np.float32(1) / np.sqrt(acc / np.float32(cols) + np.float32(eps))
    return (x.astype(np.float32) * inv).astype(np.float16)


@pytest.mark.parametrize("rows,cols,waves", [(255, 4096, 4), (256, 4096, 1), (300, 2048, 1),
                                             (256, 8192, 1)])
def test_rmsnorm_sum_order(rows, cols, waves):
    """The order of the sum, bit for bit: a block per row below 256 rows, a
    wave per row from there, the order that a layer's prefill has always had."""
    from signrot_amd import _CUDA
    rng = np.random.default_rng(cols + rows)
    x = (3 * rng.standard_normal((rows, cols))).astype(np.float16)
    want = _lane_order_norm(x, 1e-5, waves)
    assert (want != _lane_order_norm(x, 1e-5, 5 - waves)).any()   # the other order shows
    xd = torch.from_numpy(x).cuda()
    got = _CUDA.rmsnorm(xd, 1e-5, cols)
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16))
    q, s = _CUDA.rmsnorm_quant(xd, 1e-5, cols)
    qw, sw = _CUDA.sym_quant_dynamic(torch.from_numpy(want).cuda())
    assert torch.equal(q, qw) and torch.equal(s, sw)
