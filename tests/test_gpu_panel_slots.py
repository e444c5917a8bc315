"""Routed calls on the panel kernel, slot by slot: the weight stream's bodies for a slot's few rows (one to four, five to
sixteen), the panel's from seventeen, at every number of K chunks around the stream's two-deep ring."""
import pytest
import torch

from oracle import layers
from tests.util import MAX_REL, NORM_REL, errors, oracle_expert_getter, random_experts

pytestmark = pytest.mark.gpu
COUNTS = [1, 3, 4, 5, 8, 15, 16, 17, 0, 32, 33, 47, 48, 49, 64, 80, 81, 96, 97, 112, 127, 128, 129, 145]  # rows of an expert each


def _call(counts, seed):
    g = torch.Generator().manual_seed(seed)
    m = sum(counts)
    ids = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))[torch.randperm(m, generator=g)].to(torch.int32)[:, None]
    return m, ids, g


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("hidden,inter", [(128, 256), (256, 384), (384, 128), (640, 512)])  # 1, 2, 3, 5 chunks of fc1; 2, 3, 1, 4 of fc2
def test_w3_slots_of_every_height(hidden, inter, gated):
    from hibana_amd import _lib
    from hibana_amd.kernels import w3_moe
    ex, per = random_experts(len(COUNTS), hidden, inter, gated, 9)
    m, ids, g = _call(COUNTS, hidden)
    x = torch.randn(m, hidden, generator=g).bfloat16()
    want = layers.routed_experts_ref(x, ids.numpy(), oracle_expert_getter(per, gated, inter), gated, e_n=len(COUNTS))
    assert _lib.lib().hb_tune(b"w3_tile", 1) == 0
    try:
        got = w3_moe.w3_moe(ex, x.cuda(), ids.cuda(), torch.ones(m, 1, device="cuda"))
        again = w3_moe.w3_moe(ex, x.cuda(), ids.cuda(), torch.ones(m, 1, device="cuda"))
    finally:
        _lib.lib().hb_tune(b"w3_tile", 0)
    mx, nr = errors(got, want)
    assert mx < MAX_REL and nr < NORM_REL, (mx, nr)
    assert torch.equal(got, again)
