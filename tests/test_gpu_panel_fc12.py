"""fc1 and fc2 of a routed call on the panel kernel in one launch against the two launches: the same sums in the same order, so the same
bits, over the slots' heights, remainders of every kind and blocks that do not fill a workgroup."""
import contextlib

import pytest
import torch

from tests.test_gpu_nvfp4_moe import _experts
from tests.util import random_experts

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _forced(**keys):
    from hibana_amd import _lib
    for k, v in keys.items():
        assert _lib.lib().hb_tune(k.encode(), v) == 0
    try:
        yield
    finally:
        for k in keys:
            _lib.lib().hb_tune(k.encode(), 0)


def _routing(m, e, seed):
    """Rows of two: every row names expert 0 (its slots are full and its last one ragged), the other choice is a skewed draw."""
    g = torch.Generator().manual_seed(seed)
    other = 1 + (torch.rand(m, generator=g) ** 2 * (e - 1)).long()
    return torch.stack([torch.zeros(m, dtype=torch.long), other], 1).int().cuda(), torch.rand(m, 2, generator=g).cuda()


# e: the rows an expert choose the height: 48, 80, 128 or 144 rows a slot
@pytest.mark.parametrize("m,e", [(17, 4), (48, 5), (97, 4), (150, 6), (200, 4), (300, 3), (700, 8), (1100, 12)])
@pytest.mark.parametrize("hidden,inter", [(128, 640), (512, 384), (256, 128)])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("form", ["w3", "nvfp4"])
def test_one_launch_has_the_bits_of_two(form, gated, hidden, inter, m, e):
    x = torch.randn(m, hidden, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
    ids, w = _routing(m, e, m + e)
    if form == "w3":
        from hibana_amd.kernels import w3_moe
        ex, _ = random_experts(e, hidden, inter, gated, 3)
        sh, _ = random_experts(1, hidden, inter, gated, 4)
        call, tile, fused = lambda: w3_moe.moe_layer(ex, x, ids, w, shared=sh), "w3_tile", "moe_fused"
    else:
        ex, _ = _experts(e, hidden, inter, gated, 5)
        call, tile, fused = lambda: ex(x, ids, w), "nvfp4_tile", "nvfp4_fused"
    with _forced(**{tile: 1}):
        one = [call().clone() for _ in range(3)]  # a read of h ahead of its arrival would not be wrong every time
        with _forced(**{fused: 2}):
            two = call().clone()
    assert torch.isfinite(two).all() and all(torch.equal(o, two) for o in one)


# A caller's workspace need only lie on sixteen bytes: rows of h then share cache lines, and fc2 may not read them in the launch that writes them.
@pytest.mark.parametrize("tile", [1, 2])
@pytest.mark.parametrize("form", ["w3", "nvfp4"])
def test_a_workspace_off_the_cache_lines_gives_the_same_bits(form, tile, monkeypatch):
    from hibana_amd import _lib
    m, e, hidden, inter = 40, 8, 1024, 384
    x = torch.randn(m, hidden, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
    ids, w = _routing(m, e, m + e)
    if form == "w3":
        from hibana_amd.kernels import w3_moe
        ex, _ = random_experts(e, hidden, inter, True, 3)
        call, keys = lambda: w3_moe.moe_layer(ex, x, ids, w), {"w3_tile": tile}
    else:
        ex, _ = _experts(e, hidden, inter, True, 5)
        call, keys = lambda: ex(x, ids, w), {"nvfp4_tile": tile, "nvfp4_fused": 1}
    with _forced(**keys):
        want = call().clone()
        asked = []
        monkeypatch.setattr(_lib, "workspace", lambda device, need, kind="moe": asked.append(torch.zeros(need + 16, dtype=torch.uint8, device=device)[16:]) or asked[-1])
        got = call().clone()
    assert asked and all(a.data_ptr() % 256 == 16 for a in asked) and torch.equal(got, want)
