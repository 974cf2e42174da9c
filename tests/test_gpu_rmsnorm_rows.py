"""RMSNorm + quantizer on both sides of the block-per-row rule (256 rows, 2048
columns): the fused codes are those of the quantizer over the norm's output,
and the norm is within fp16 rounding of 64 bits."""
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
