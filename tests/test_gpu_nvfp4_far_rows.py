"""NVFP4 products on activation matrices past 4 GiB. The panel kernel addresses a matrix with 32-bit byte offsets and does
not take them; the weight stream's sixteen-row body does, and its rows on the far side must be their own."""
import pytest
import torch

from tests.util import MAX_REL, NORM_REL, errors

pytestmark = pytest.mark.gpu

K = 25600
LAST = 0xffffffff // (2 * K)  # rows of the largest matrix of this K that the panel kernel takes


@pytest.mark.parametrize("m", [LAST, LAST + 1, LAST + 115])
def test_dense_rows_on_both_sides_of_four_gib(m):
    from hibana_amd import synthetic
    from hibana_amd.kernels import ops
    lin = synthetic.nvfp4_linear(64, K, 3, global_scale=0.01)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, K, device="cuda", generator=g, dtype=torch.bfloat16)
    got = ops.nvfp4_linear(x, lin)
    dense = lin.dequantize()
    for rows in (slice(0, 160), slice(m - 160, m)):  # an offset that wraps reads the first rows for the last
        mx, nr = errors(got[rows], x[rows].float() @ dense.T)
        assert mx < MAX_REL and nr < NORM_REL, (m, rows, mx, nr)


def test_routed_pairs_past_four_gib():
    """fc2's activations, one row a pair: 800 800 rows of 2688."""
    from hibana_amd import synthetic
    ex = synthetic.nvfp4_experts(32, 128, 2688, 5)
    m, topk = 36400, 22
    assert m * topk * ex.n * 2 > 1 << 32
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(m, 128, device="cuda", generator=g, dtype=torch.bfloat16)
    ids = torch.rand(m, 32, device="cuda", generator=g).topk(topk).indices.to(torch.int32)  # (the pairs lie sorted by expert: every row has some on either side)
    weights = torch.rand(m, topk, device="cuda", generator=g)
    got = ex(x, ids, weights)
    for rows in (slice(0, 8), slice(m // 2, m // 2 + 8), slice(m - 8, m)):
        mx, nr = errors(got[rows], ex(x[rows], ids[rows], weights[rows]))
        assert mx < MAX_REL and nr < NORM_REL, (rows, mx, nr)
