"""The 160-row tiles of the expert-offset GEMMs without extra rows (asymmetric
activations, the gate and up pair) against the dense linear of each expert, bit
for bit: counts at the tile's edges, empty experts, and averages at both ends
of its range and past them."""
import pytest
import torch
from test_gpu_moe_rows import C, _data  # noqa: F401  (C is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(128, 256), (144, 1056), (4096, 4096)])
@pytest.mark.parametrize("counts", [[160, 161, 129, 40], [0, 320, 200, 20], [146] * 4,
                                    [147, 146, 146, 146], [122] * 4, [128, 127, 1, 300]])
def test_moe_160_rows_bitexact(C, counts, N, K):  # noqa: F811
    off, a, sa, b, sb, z = _data(counts, N, K, N + K)
    bounds = off.tolist()
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
        assert torch.equal(gate[r], want), f"gate, expert {e}"
        assert torch.equal(up[r], want.flip(1)), f"up, expert {e}"
        assert torch.equal(asym[r], C.w4a4_linear_asym(ae, se, z[r].contiguous(), b[e], sb[e],
                                                       wsum[e])), f"asym, expert {e}"
