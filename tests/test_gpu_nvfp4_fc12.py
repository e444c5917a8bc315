"""fc1 and fc2 of NVFP4 experts in one launch against the two launches, and the small latent block in one call against
`router` and `block`: the same sums in the same order, so the same bits (of the block, behind a shared expert
too: tests/test_gpu_latent_layer_bits.py)."""
import contextlib

import pytest
import torch

from tests.test_gpu_nvfp4_moe import _experts
from tests.util import MAX_REL, NORM_REL, errors

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _forced(key, value):
    from hibana_amd import _lib
    assert _lib.lib().hb_tune(key, value) == 0
    try:
        yield
    finally:
        _lib.lib().hb_tune(key, 0)


# blocks that do not fill their workgroups (fc1 10 and 6 blocks, fc2 2 and 6), one chunk of K and many, workgroups that differ in
# size apart; rows an expert 1, 4, 5, 8, 9, 16 and, past 16, a second slot
@pytest.mark.parametrize("hidden,inter", [(128, 640), (1024, 384), (384, 128), (256, 2688)])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16, 17, 40])
def test_one_launch_has_the_bits_of_two(hidden, inter, gated, m):
    ex, _ = _experts(8, hidden, inter, gated, 5)
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, hidden, generator=g).bfloat16().cuda()
    ids = torch.stack([torch.cat([torch.zeros(1, dtype=torch.long), 1 + torch.randperm(7, generator=g)[:2]]) for _ in range(m)]).int().cuda()  # expert 0: every row
    w = torch.rand(m, 3, generator=g).cuda()
    out = []
    for form in (1, 2):
        with _forced(b"nvfp4_tile", 2), _forced(b"nvfp4_fused", form):
            out.append(ex(x, ids, w).clone())
    assert torch.isfinite(out[0]).all() and torch.equal(*out)


@pytest.mark.parametrize("hidden,latent,inter,experts,topk,shared", [(512, 128, 640, 16, 4, 0), (1024, 512, 384, 200, 8, 640), (2048, 1024, 2688, 64, 22, 128)])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("padded", [False, True])
def test_layer_is_router_and_block(hidden, latent, inter, experts, topk, shared, m, form, padded):
    from hibana_amd import synthetic
    from hibana_amd.kernels import nemotron_moe as small
    from hibana_amd.model.nemotron_moe import NemotronMoe
    g = torch.Generator(device="cuda").manual_seed(m)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    up, down = (synthetic.nvfp4_linear(shared, hidden, 1), synthetic.nvfp4_linear(hidden, shared, 2)) if shared else (None, None)
    block = NemotronMoe((draw(experts + latent, hidden) / hidden ** 0.5).bfloat16(), torch.rand(experts, device="cuda", generator=g), (draw(hidden, latent) / latent ** 0.5).bfloat16(),
                        synthetic.nvfp4_experts(experts, latent, inter, 3), topk, shared_up=up, shared_down=down)
    weights = block.small_weights()
    x = draw(m, hidden).bfloat16()
    slots = torch.arange(m, device="cuda", dtype=torch.int32) if padded else None  # row 0 is padding
    _, ids, w, ws = small.router(x, weights, None, topk, slots, 1)
    want = small.block(x, ws, ids, w, weights).clone()
    with _forced(b"nvfp4_fused", form):
        got = small.layer(x, weights, topk, slots, 1)
    if shared:
        mx, nr = errors(got, want)
        assert mx < MAX_REL and nr < NORM_REL
    else:
        assert torch.equal(got, want)


def test_layer_replays_in_a_graph():
    from hibana_amd import synthetic
    from hibana_amd.model.nemotron_moe import NemotronMoe
    g = torch.Generator(device="cuda").manual_seed(1)
    draw = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    block = NemotronMoe((draw(512 + 1024, 1024) / 32).bfloat16(), torch.rand(512, device="cuda", generator=g), (draw(1024, 1024) / 32).bfloat16(),
                        synthetic.nvfp4_experts(512, 1024, 1024, 3), 22, shared_up=synthetic.nvfp4_linear(640, 1024, 1), shared_down=synthetic.nvfp4_linear(1024, 640, 2))
    x = draw(6, 1024).bfloat16()
    block(x, None)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = block(x, None)
    for _ in range(4):
        x.copy_(draw(6, 1024).bfloat16())
        want = block(x, None).clone()
        graph.replay()
        assert torch.equal(out, want)
