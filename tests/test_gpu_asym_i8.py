"""The register form of the asymmetric quantizer against the general one (which
an unaligned input takes), and int8 zero points against torch's cast, over
rows of every kind: constant, all-positive (zero points far below -128),
all-negative, tiny, huge, infinite, NaN."""
import numpy as np
import pytest
import torch

from tests.gpu_util import outlier_input, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    from signrot_amd import _CUDA
    return _CUDA


def _rows(cols, rows=40, seed=0):
    rng = np.random.default_rng(seed + cols)
    x = outlier_input(rng, rows, cols, n_out=min(4, cols // 4), mag=30.0)
    f = rng.standard_normal((rows, cols)).astype(np.float32)
    x[1] = 0
    x[2] = np.float16(1.5)
    x[3] = (np.abs(f[3]) * 0.01 + 100).astype(np.float16)     # zero point about -10^4
    x[4] = (-np.abs(f[4]) * 0.01 - 100).astype(np.float16)    # about 10^4
    x[5] = (f[5] * 1e-6).astype(np.float16)
    x[6] = (f[6] * 2e4).astype(np.float16)
    x[7, 3] = np.inf
    x[8, cols - 1] = -np.inf
    x[9, 2] = np.nan
    x[10] = np.nan
    x[11] = np.inf
    for i, base in enumerate((3, 10, 20, 33, 40, 60)):        # zero points around +-128, +-511
        x[12 + 2 * i] = (f[12] * 0.3 + base).astype(np.float16)
        x[13 + 2 * i] = (f[13] * 0.3 - base).astype(np.float16)
    return x


def _same_zero(a, b):
    """Equal, a zero of either sign counting as zero, NaN as NaN."""
    return torch.equal(torch.nan_to_num(a + 0, nan=-7.0), torch.nan_to_num(b + 0, nan=-7.0))


@pytest.mark.parametrize("cols", [8, 136, 2048, 2056, 4096, 8200, 14336, 16384, 16392])
@pytest.mark.parametrize("clip", [1.0, 0.8])
def test_register_form_and_int8_zero(C, cols, clip):
    x = to_dev(_rows(cols))
    rows = x.shape[0]
    buf = torch.empty(rows * cols + 1, dtype=torch.float16, device="cuda")
    odd = buf[1:].view(rows, cols)
    odd.copy_(x)
    q, s, z = C.asym_quant_dynamic(x, clip)
    qg, sg, zg = C.asym_quant_dynamic(odd, clip)
    assert torch.equal(s.view(torch.int16), sg.view(torch.int16)) and _same_zero(z, zg)
    assert torch.equal(q, qg)
    for src in (x, odd):
        q8, s8, z8 = C.asym_quant_dynamic(src, clip, True)
        assert z8.dtype == torch.int8 and torch.equal(z8, z.to(torch.int8))
        assert torch.equal(q8, q) and torch.equal(s8.view(torch.int16), s.view(torch.int16))


@pytest.mark.parametrize("cols", [136, 14336])
def test_moe_signs(C, cols):
    x = to_dev(_rows(cols, seed=1))
    rows, E = x.shape[0], 3
    rng = np.random.default_rng(cols)
    sign = to_dev(rng.choice([-1, 1], (E, cols)).astype(np.int8))
    ids = to_dev(rng.integers(-1, E + 1, rows).astype(np.int32))   # some outside the table
    inside = (ids >= 0) & (ids < E)
    flip = torch.where(inside[:, None], sign[ids.clamp(0, E - 1).long()], 1)
    q, s, z = C.asym_quant_dynamic_moe(x, sign, ids)
    q2, s2, z2 = C.asym_quant_dynamic(torch.where(flip < 0, -x, x))
    assert torch.equal(q, q2) and torch.equal(s.view(torch.int16), s2.view(torch.int16))
    assert _same_zero(z, z2)
    q8, _, z8 = C.asym_quant_dynamic_moe(x, sign, ids, 1.0, True)
    assert torch.equal(q8, q) and torch.equal(z8, z.to(torch.int8))


# the three rotations with an asymmetric form, more rows than two blocks per CU
@pytest.mark.parametrize("n,k", [(14336, 28), (28672, 28), (11008, 172), (5120, 40)])
def test_rotation_int8_zero(C, n, k):
    from signrot_amd.functional import hadamard_matrices as hm
    hk = getattr(hm, f"get_had{k}")().half().cuda().contiguous()
    x = to_dev(np.tile(_rows(n), (14, 1)))
    q, s, z = C.had_sign_asym_quant(x, hk, k)
    q8, s8, z8 = C.had_sign_asym_quant(x, hk, k, None, 1.0, True)
    assert torch.equal(z8, z.to(torch.int8))
    assert torch.equal(q8, q) and torch.equal(s8.view(torch.int16), s.view(torch.int16))
    rot = C.online_hadamard(x, hk, k)
    q2, s2, z2 = C.asym_quant_dynamic(rot)
    assert torch.equal(q, q2) and torch.equal(s.view(torch.int16), s2.view(torch.int16))
    assert _same_zero(z, z2)
