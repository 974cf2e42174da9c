"""GPU parity of the MFMA rotation for n = K x m outside the 512 / 1024 chunk
forms (hadamard_kron.hip): every launch form (K up to 32, 64, 112, 176; m =
64 ... 512), one row, more rows than blocks, values that the quantizers treat
apart, sign vectors of any alignment."""
import numpy as np
import pytest
import torch

from oracle import hadamard as oh
from oracle import quant as oq
from tests.gpu_util import assert_bitexact, outlier_input, to_dev, to_np

pytestmark = pytest.mark.gpu

SHAPES = [(12, 64), (28, 128), (20, 256), (40, 64), (52, 128), (60, 256), (36, 512),
          (108, 64), (108, 128), (140, 64), (148, 128), (156, 128), (172, 64)]


@pytest.fixture(scope="module")
def C():
    from signrot_amd import _CUDA
    return _CUDA


def _hadk(k):
    from signrot_amd.functional import hadamard_matrices as hm
    return getattr(hm, f"get_had{k}")().half().cuda().contiguous()


def _exact(x, hadk, k, sign):
    """float64: hadK . FWHT / sqrt(n), with the fp16 rounding between them."""
    n = x.shape[-1]
    m = n // k
    y = torch.from_numpy(x).cuda().double().view(-1, k, m)
    h = 1
    while h < m:
        y = y.view(-1, k, m // (2 * h), 2, h)
        y = torch.stack((y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]), -2)
        y = y.reshape(-1, k, m)
        h *= 2
    y = (y / np.sqrt(n)).half().double()
    return ((hadk.double() @ y).view(-1, n) * torch.from_numpy(sign).cuda().double()).cpu().numpy()


@pytest.mark.parametrize("k,m", SHAPES)
@pytest.mark.parametrize("rows", [1, 1030])
def test_kron_rotation_and_quantizers(C, k, m, rows):
    n = k * m
    rng = np.random.default_rng(n + rows)
    x = outlier_input(rng, rows, n, n_out=8, mag=50.0)
    if rows > 8:
        x[1] = 0                           # scale 0
        x[2] = 0
        x[2, 11] = np.float16(2.0 ** -24)  # scale underflows
        x[3] *= np.float16(100)
        x[4, 5] = np.float16(np.inf)       # non-finite rows take the exact route
        x[5, n - 1] = np.float16(np.nan)
        x[6, m] = np.float16(np.inf)
        x[6, 2 * m] = np.float16(-np.inf)
        x[7] = np.float16(1.5)
    hk = _hadk(k)
    sign_np = rng.choice([-1, 1], n).astype(np.int8)
    xd, sd = to_dev(x), to_dev(sign_np)
    rot = C.online_hadamard(xd, hk, k, sd)
    fin = [r for r in range(rows) if rows == 1 or r not in (4, 5, 6)]
    got = to_np(rot)[fin].astype(np.float64)
    want = _exact(x[fin], hk, k, sign_np)
    # one fp16 rounding of the K-mix, plus what y moves when its fp32 sum lies
    # at a rounding edge: an ulp of y (rare), K of them at most
    ymax = np.abs(want).max(axis=1, keepdims=True) + 2.0 ** -14
    assert np.all(np.abs(got - want) <= np.spacing(np.abs(want).astype(np.float16)) + 4e-3 * ymax)
    # share of outputs that differ at all: an fp32 sum around an outlier of 50
    # is off by about 50 * 2^-25, which moves y (about sqrt(m) >= 8, fp16
    # spacing 2^-8) over a rounding edge in about 2 * 50 * 2^-25 / 2^-8 = 7.6e-4
    # cases, by one ulp(y) = ulp(out) / sqrt(k); an output sums k of them
    assert np.mean(got != want.astype(np.float16)) < 1e-3 * (1 + np.sqrt(k))
    for clip in (1.0, 0.8):
        q, s = C.had_sign_quant(xd, hk, k, sd, clip)
        qw, sw = oq.sym_quant_dynamic(to_np(rot), clip)
        assert_bitexact(to_np(s), sw, f"scale, clip {clip}")
        assert_bitexact(to_np(q), qw, f"codes, clip {clip}")
        assert C.had_asym_fusable(n, k)
        q, s, z = C.had_sign_asym_quant(xd, hk, k, sd, clip)
        q2, s2, z2 = C.asym_quant_dynamic(rot, clip)
        assert torch.equal(s.view(torch.int16), s2.view(torch.int16)), f"asym scale, clip {clip}"
        assert torch.equal(torch.nan_to_num(z), torch.nan_to_num(z2)), f"zero, clip {clip}"
        assert torch.equal(q, q2), f"asym codes, clip {clip}"


def test_kron_sign_values_and_alignment(C):
    """No sign, a sign vector at an odd address, and other factors than +-1
    (the op multiplies by whatever int8 it is given)."""
    k, m, rows = 172, 64, 5
    n = k * m
    rng = np.random.default_rng(0)
    xd, hk = to_dev(outlier_input(rng, rows, n, n_out=8, mag=50.0)), _hadk(k)
    plain = C.online_hadamard(xd, hk, k, None)
    vals = to_dev(rng.choice([-1, 1, 0, 2, -3], n).astype(np.int8))
    buf = torch.empty(n + 16, dtype=torch.int8, device="cuda")
    odd = buf[3:n + 3]
    odd.copy_(vals)
    want = (plain.float() * vals.float()).half()
    for s in (vals, odd):
        out = C.online_hadamard(xd, hk, k, s)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        q, sc = C.had_sign_quant(xd, hk, k, s)
        q2, sc2 = C.sym_quant_dynamic(want)
        assert torch.equal(q, q2) and torch.equal(sc, sc2)


def test_kron_matches_general_kernel(C):
    """A hadK table at an address that the MFMA form refuses takes the LDS
    kernel: the same rotation up to the order of the fp32 sums."""
    k, m, rows = 108, 128, 3
    n = k * m
    rng = np.random.default_rng(1)
    xd, hk = to_dev(outlier_input(rng, rows, n, n_out=8, mag=50.0)), _hadk(k)
    buf = torch.empty(k * k + 1, dtype=torch.float16, device="cuda")
    off = buf[1:].view(k, k)
    off.copy_(hk)
    a, b = C.online_hadamard(xd, hk, k), C.online_hadamard(xd, off, k)
    assert torch.mean((a != b).float()) < 5e-3
    assert torch.allclose(a.float(), b.float(), rtol=2e-3, atol=2e-3)
    q, s, z = C.had_sign_asym_quant(xd, off, k)
    q2, s2, z2 = C.asym_quant_dynamic(b)
    assert torch.equal(q, q2) and torch.equal(s, s2) and torch.equal(z, z2)
