"""A rank's range of the experts: the rows an expert that choose between the weight stream and the panel kernel are the
call's pairs over ALL the experts its ids name, not over the few held here. The two kernels add in different orders, so
the bits say which one ran."""
import contextlib

import pytest
import torch

from tests.util import MAX_REL, NORM_REL, errors, random_experts

pytestmark = pytest.mark.gpu
E, LOCAL, BASE, TOPK = 64, 8, 16, 8


@contextlib.contextmanager
def _forced(key, value):
    from hibana_amd import _lib
    assert _lib.lib().hb_tune(key, value) == 0
    try:
        yield
    finally:
        _lib.lib().hb_tune(key, 0)


def _by_kernel(key, call):
    """(the panel kernel's result, the stream's): different bits of the same product."""
    out = []
    for tile in (1, 2):
        with _forced(key, tile):
            out.append(call().clone())
    mx, nr = errors(*out)
    assert mx < MAX_REL and nr < NORM_REL and not torch.equal(*out)
    return out


def _draw(m, hidden, seed):
    g = torch.Generator().manual_seed(seed)
    ids = torch.stack([torch.randperm(E, generator=g)[:TOPK] for _ in range(m)]).to(torch.int32).cuda()
    return torch.randn(m, hidden, generator=g).bfloat16().cuda(), ids, torch.rand(m, TOPK, generator=g).cuda()


@pytest.mark.parametrize("m,panel", [(40, False), (63, False), (64, True), (300, True)])  # 8 rows an expert: 512 pairs of 64 experts
def test_nvfp4_range_of_a_latent_block(m, panel):
    from hibana_amd import synthetic
    from hibana_amd.model.nemotron_moe import NemotronMoe
    ex = synthetic.nvfp4_experts(LOCAL, 512, 1024, 7)
    ex.base = BASE
    g = torch.Generator().manual_seed(1)
    block = NemotronMoe(torch.randn(E + 512, 512, generator=g).bfloat16().cuda(), torch.rand(E, generator=g).cuda(), torch.randn(512, 512, generator=g).bfloat16().cuda(), ex, TOPK)
    lat, ids, weights = _draw(m, 512, m)
    by_panel, by_stream = _by_kernel(b"nvfp4_tile", lambda: block.routed(lat, ids, weights))
    assert torch.equal(block.routed(lat, ids, weights), by_panel if panel else by_stream)


@pytest.mark.parametrize("m,panel", [(60, False), (383, False), (384, True)])  # 48 rows an expert: 3072 pairs of 64 experts
@pytest.mark.parametrize("entry", ["w3_moe", "moe_layer", "routed", "layer"])
def test_w3_range_of_a_gated_layer(entry, m, panel):
    from hibana_amd.kernels import w3_moe
    from hibana_amd.model.flashnext_moe import MoeLayer
    ex, _ = random_experts(LOCAL, 1024, 512, True, 3)
    ex.base = BASE
    x, ids, weights = _draw(m, 1024, m)
    g = torch.Generator().manual_seed(2)
    layer = MoeLayer(torch.randn(E, 1024, generator=g).bfloat16().cuda(), torch.zeros(1024).cuda(), ex, TOPK)
    call = {"w3_moe": lambda: w3_moe.w3_moe(ex, x, ids, weights, experts_total=E), "moe_layer": lambda: w3_moe.moe_layer(ex, x, ids, weights, experts_total=E),
            "routed": lambda: layer.routed(x, ids, weights), "layer": lambda: layer(x)}[entry]
    by_panel, by_stream = _by_kernel(b"w3_tile", call)
    assert torch.equal(call(), by_panel if panel else by_stream)
