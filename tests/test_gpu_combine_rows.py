"""The combine of a long call with a shared expert, a row a workgroup, against the short calls' form (a span of columns a
workgroup), bit for bit: columns that fill a load, a pass of a workgroup, more and less; batches' edges; dropped pairs."""
import pytest
import torch

from tests.util import random_experts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("m,topk,h", [(1024, 1, 8), (1024, 12, 2040), (1025, 13, 2048), (1024, 10, 2056), (1031, 25, 520), (1024, 3, 4104)])
def test_bf16_pairs(m, topk, h, gated):
    from hibana_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(m + topk + h)
    e_lo, e_n = 3, 9
    ids = torch.randint(0, 16, (m, topk), generator=g, device="cuda", dtype=torch.int32)  # a quarter of them outside
    ids[5], ids[6] = -1, e_lo + e_n  # rows of which nothing is left
    weights = torch.rand(m, topk, generator=g, device="cuda")
    y = torch.randn(m * topk, h, generator=g, device="cuda").bfloat16()
    y[((ids < e_lo) | (ids >= e_lo + e_n)).view(-1)] = float("nan")
    shared, x = torch.randn(m, h, generator=g, device="cuda").bfloat16(), torch.randn(m, h, generator=g, device="cuda").bfloat16()
    gate = torch.randn(h, generator=g, device="cuda") * 0.05 if gated else None
    got = ops.moe_combine_pairs(y, ids, weights, shared, x, gate, e_lo, e_n)
    assert torch.isfinite(got).all()
    half = m // 2
    parts = [ops.moe_combine_pairs(y[r0 * topk:r1 * topk], ids[r0:r1], weights[r0:r1], shared[r0:r1], x[r0:r1], gate, e_lo, e_n) for r0, r1 in ((0, half), (half, m))]
    assert torch.equal(got, torch.cat(parts))


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("m,topk,h", [(1024, 8, 1024), (1024, 9, 1024), (1024, 8, 1032), (1030, 9, 512), (1030, 9, 520), (1024, 12, 2304), (1024, 13, 2560)])
def test_bf16_pairs_around_the_lines(m, topk, h, gated):
    """Widths and selections on both sides of the lines between the two forms, and widths whose last pass few threads take."""
    test_bf16_pairs(m, topk, h, gated)


@pytest.mark.parametrize("m,topk,hidden", [(511, 9, 2048), (512, 8, 2048), (512, 9, 2048), (512, 9, 1920), (513, 12, 2304), (530, 13, 2560), (512, 9, 3200)])
def test_fp32_pairs_of_a_layer_around_the_lines(m, topk, hidden):
    """Passes of 1024 columns that are partly used, and both sides of the lines."""
    _layer_of_fp32_pairs(m, topk, hidden)


@pytest.mark.parametrize("m,topk", [(512, 2), (520, 13)])  # the first size, 2048 columns, and one more batch
def test_fp32_pairs_of_a_layer(m, topk):
    _layer_of_fp32_pairs(m, topk, 2048)


def _layer_of_fp32_pairs(m, topk, hidden):
    from hibana_amd import _lib
    from hibana_amd.kernels import ops, w3_moe
    (ex, _), (sh, _) = random_experts(16, hidden, 128, True, 5), random_experts(1, hidden, 128, True, 6)
    g = torch.Generator().manual_seed(m)
    ids = torch.stack([torch.randperm(17, generator=g)[:topk] for _ in range(m)]).to(torch.int32).cuda()  # 16: no expert
    x, weights, gate = torch.randn(m, hidden, generator=g).bfloat16().cuda(), torch.rand(m, topk, generator=g).cuda(), (torch.randn(hidden, generator=g) * 0.02).cuda()
    assert _lib.lib().hb_tune(b"w3_tile", 1) == 0
    try:
        got = w3_moe.moe_layer(ex, x, ids, weights, shared=sh, gate_vec=gate)
        pairs = w3_moe.w3_moe(ex, x, ids, weights, pairs=True)
        own = w3_moe.w3_moe(sh, x, torch.zeros(m, 1, dtype=torch.int32, device="cuda"), torch.ones(m, 1, device="cuda"), pairs=True)
    finally:
        _lib.lib().hb_tune(b"w3_tile", 0)
    assert pairs.dtype == torch.float32
    assert torch.equal(got, ops.moe_combine_pairs(pairs, ids, weights, own.bfloat16(), x, gate, 0, 16))
