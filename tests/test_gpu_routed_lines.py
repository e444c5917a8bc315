"""From how many rows an expert a routed call of few, wide experts takes the panel kernel: fc2's workgroups are then few and as long as its K, and the weight
stream serves more rows. The two kernels add in different orders, so the bits say which one ran."""
import pytest
import torch

from tests.test_gpu_expert_ranges import _by_kernel, _forced

pytestmark = pytest.mark.gpu


def _draw(m, e, k, hidden):
    g = torch.Generator().manual_seed(m)
    ids = torch.stack([torch.randperm(e, generator=g)[:k] for _ in range(m)]).int().cuda()
    return torch.randn(m, hidden, generator=g).bfloat16().cuda(), ids, torch.rand(m, k, generator=g).cuda()


# fc2's workgroups a chunk of its K: 90, 64, 32, 26, 6, 0.5, 12 (fc1 of few workgroups)
@pytest.mark.parametrize("experts,hidden,inter,rows", [(300, 640, 1280, 4), (256, 768, 1536, 3), (128, 512, 1024, 5), (160, 512, 1536, 7), (48, 768, 2816, 14), (16, 512, 8192, 60), (48, 512, 1024, 7)])
def test_nvfp4(experts, hidden, inter, rows):
    from hibana_amd import synthetic
    ex = synthetic.nvfp4_experts(experts, hidden, inter, 1)
    for m in (rows * experts // 4 - 1, rows * experts // 4):
        x, ids, w = _draw(m, experts, 4, hidden)
        by_panel, by_stream = _by_kernel(b"nvfp4_tile", lambda: ex(x, ids, w))
        assert torch.equal(ex(x, ids, w), by_panel if 4 * m >= rows * experts else by_stream)


# 150 experts and more; fewer; fc2 of few workgroups a chunk of its K; fc1 of many workgroups
@pytest.mark.parametrize("experts,hidden,inter,rows", [(180, 1664, 384, 7), (128, 512, 512, 16), (24, 512, 6144, 24), (96, 1024, 3072, 14), (64, 1536, 4096, 9)])
def test_three_bit(experts, hidden, inter, rows):
    from hibana_amd import synthetic
    from hibana_amd.kernels import w3_moe
    ex = w3_moe.tile(synthetic.w3_experts(experts, hidden, inter, True, 1), release=True)
    for m in ((rows * experts - 1) // 4, (rows * experts + 3) // 4):
        x, ids, w = _draw(m, experts, 4, hidden)
        by_panel, by_stream = _by_kernel(b"w3_tile", lambda: w3_moe.w3_moe(ex, x, ids, w))
        assert torch.equal(w3_moe.w3_moe(ex, x, ids, w), by_panel if 4 * m >= rows * experts else by_stream)


# wider than long, all workgroups at once, and the long end that keeps its own launch: either way the same bits
@pytest.mark.parametrize("experts,hidden,inter", [(64, 512, 4096), (24, 512, 4096), (32, 512, 6144)])
@pytest.mark.parametrize("rows", [16, 40])
def test_one_launch_and_two_have_the_same_bits(experts, hidden, inter, rows):
    from hibana_amd import synthetic
    ex = synthetic.nvfp4_experts(experts, hidden, inter, 1)
    x, ids, w = _draw(rows * experts // 4, experts, 4, hidden)
    out = [ex(x, ids, w).clone()]
    for form in (1, 2):
        with _forced(b"nvfp4_tile", 1), _forced(b"nvfp4_fused", form):
            out.append(ex(x, ids, w).clone())
    assert torch.isfinite(out[0]).all() and torch.equal(out[1], out[2])
