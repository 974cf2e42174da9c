"""The prefill's q/k/v pass where a block takes several passes over a token's
rows, against the op-by-op path, bit for bit."""
import pytest
import torch
from test_gpu_prefill_fused import _cos_sin, _layer, _run

pytestmark = pytest.mark.gpu


# 24 rows a token (two passes): 2 blocks a token below 2048 tokens, 1 from there
@pytest.mark.parametrize("T", [2047, 2048])
def test_prefill_passes_bitexact(T):
    layer = _layer(2048, 16, 4, 896)
    h = torch.randn(1, T, 2048, device="cuda", generator=torch.Generator("cuda").manual_seed(T))
    cos, sin = _cos_sin(1, T, False)
    fused = _run(layer, h.half(), 1, T, 64, cos, sin, None, None)
    ops = _run(layer, h.half(), 1, T, 64, cos, sin, None, {})
    for a, b in zip(fused, ops):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
