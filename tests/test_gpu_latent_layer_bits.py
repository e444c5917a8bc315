"""The small latent block in one call against `router` and `block`: the same sums in the same order, so the same bits, also behind a shared
expert, whose up projection stands beside the plan in one form and beside fc1 in the other."""
import pytest
import torch

from tests.test_gpu_nvfp4_fc12 import _forced

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,latent,inter,experts,topk,shared", [(512, 128, 640, 16, 4, 0), (1024, 512, 384, 200, 8, 640), (2048, 1024, 2688, 64, 22, 128), (4096, 1024, 2688, 64, 22, 5376)])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("padded", [False, True])
def test_layer_has_the_bits_of_router_and_block(hidden, latent, inter, experts, topk, shared, m, form, padded):
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
    assert torch.equal(got, want)
