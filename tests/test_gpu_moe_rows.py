"""The expert-offset GEMMs with few rows per expert (gemm_rows_kernel: tiles of
32, 64 or 96 rows) against the dense linear of each expert, bit for bit: row
counts at the edges of the row blocks, empty experts, more tiles than
workgroups, ragged N and K, and the average row counts where the tile
changes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"

# rows per expert; the averages fall on 1, 2 and 3 row blocks and past them
COUNTS = [[1, 0, 31, 32], [33, 0, 1, 46], [64, 20, 0, 65], [97, 95, 96, 32], [1, 0, 0, 320],
          [20, 20, 20, 20], [48, 48, 48, 48], [80, 80, 80, 80], [81, 80, 80, 80]]


@pytest.fixture(scope="module")
def C():
    from signrot_amd import _CUDA
    return _CUDA


def _data(counts, N, K, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    E, R = len(counts), sum(counts)
    off = torch.tensor([0] + counts, device=DEV).cumsum(0).int()
    a = torch.randint(0, 256, (R, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    sa = (torch.rand(R, device=DEV, generator=g) * 0.01 + 1e-3).half()
    b = torch.randint(0, 256, (E, N, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    sb = (torch.rand(E, N, device=DEV, generator=g) * 0.01 + 1e-3).half()
    z = torch.randint(-8, 16, (R,), dtype=torch.int8, device=DEV, generator=g)
    return off, a, sa, b, sb, z


# K: one step, a ragged step, fewer steps than the ring, more
@pytest.mark.parametrize("N,K", [(128, 256), (144, 288), (272, 1056), (4096, 4096)])
@pytest.mark.parametrize("counts", COUNTS)
def test_moe_rows_bitexact(C, counts, N, K):
    off, a, sa, b, sb, z = _data(counts, N, K, N + K)
    bounds = off.tolist()
    plain = C.w4a4_linear_moe(a, sa, b, sb, off)
    sw = C.w4a4_linear_moe_swiglu(a, sa, b, sb, off)
    wsum = C.sum_i4(b.view(-1, K // 2)).view(len(counts), N)
    asym = C.w4a4_linear_moe_asym(a, sa, z, b, sb, wsum, off)
    gate, up = C.w4a4_linear_moe_gate_up(a, sa, b, sb, b.flip(1).contiguous(),
                                         sb.flip(1).contiguous(), off)
    for e in range(len(counts)):
        r = slice(bounds[e], bounds[e + 1])
        if counts[e] == 0:
            continue
        ae, se = a[r].contiguous(), sa[r].contiguous()
        want = C.w4a4_linear(ae, se, b[e], sb[e])
        assert torch.equal(plain[r], want), f"expert {e}"
        assert torch.equal(gate[r], want), f"gate, expert {e}"
        assert torch.equal(up[r], want.flip(1)), f"up, expert {e}"
        assert torch.equal(sw[r], C.w4a4_linear_swiglu(ae, se, b[e], sb[e])), f"swiglu, {e}"
        assert torch.equal(asym[r], C.w4a4_linear_asym(ae, se, z[r].contiguous(), b[e], sb[e],
                                                       wsum[e])), f"asym, expert {e}"


def test_moe_rows_many_experts(C):
    """More experts than workgroups, most of them empty, rows in a few."""
    E, N, K = 300, 160, 512
    counts = [0] * E
    for e, n in ((0, 3), (17, 40), (255, 1), (256, 33), (299, 2)):
        counts[e] = n
    off, a, sa, b, sb, _ = _data(counts, N, K, 1)
    out = C.w4a4_linear_moe(a, sa, b, sb, off)
    bounds = off.tolist()
    for e in (0, 17, 255, 256, 299):
        r = slice(bounds[e], bounds[e + 1])
        want = C.w4a4_linear(a[r].contiguous(), sa[r].contiguous(), b[e], sb[e])
        assert torch.equal(out[r], want), f"expert {e}"


# routers that send most rows to few experts: by the average these take 32-row to
# 160-row tiles, by the experts' rows the 128-row form, with and without its extra
# rows, among empty experts and past 64 of them
@pytest.mark.parametrize("counts", [[0, 0, 80, 0, 0, 0, 0, 0], [96, 0, 0, 64], [0] * 5 + [129, 0, 0],
                                    [0, 192, 0, 190], [250, 0, 2, 0], [1, 0, 0, 500],
                                    [0] * 70 + [640, 3, 0, 130], [128] * 4, [60, 70, 256, 0]])
@pytest.mark.parametrize("N,K", [(144, 288), (4096, 1024)])
def test_moe_skewed_bitexact(C, counts, N, K):
    test_moe_rows_bitexact(C, counts, N, K)
