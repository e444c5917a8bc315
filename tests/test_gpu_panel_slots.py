"""Routed calls on the panel kernel, slot by slot: the weight stream's bodies for a slot's few rows (one to four, five to
sixteen), the panel's from seventeen, at every number of K chunks around the stream's two-deep ring; slots of 48, 80, 128 and
144 rows, which the rows an expert choose; and the lines that give a call to the panel kernel."""
import pytest
import torch

from oracle import layers, nvfp4_format as onv
from tests.util import MAX_REL, NORM_REL, errors, oracle_expert_getter, random_experts

pytestmark = pytest.mark.gpu
COUNTS = [1, 3, 4, 5, 8, 15, 16, 17, 0, 32, 33, 47, 48, 49, 64, 80, 81, 96, 97, 112, 127, 128, 129, 145]  # rows of an expert each


def _call(counts, seed):
    g = torch.Generator().manual_seed(seed)
    m = sum(counts)
    ids = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))[torch.randperm(m, generator=g)].to(torch.int32)[:, None]
    return m, ids, g


TOTALS = [0, 31, 100]  # experts that the ids are said to name: 56, 43 and 13 rows an expert
MORE, MOST = [300], [900]  # ... and with one expert more 65 and 89


@pytest.mark.parametrize("total,more", [(t, []) for t in TOTALS] + [(0, MORE), (0, MOST)])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("hidden,inter", [(128, 256), (256, 384), (384, 128), (640, 512)])  # 1, 2, 3, 5 chunks of fc1; 2, 3, 1, 4 of fc2
def test_w3_slots_of_every_height(hidden, inter, gated, total, more):
    from hibana_amd import _lib
    from hibana_amd.kernels import w3_moe
    counts = COUNTS + more
    ex, per = random_experts(len(counts), hidden, inter, gated, 9)
    m, ids, g = _call(counts, hidden)
    x = torch.randn(m, hidden, generator=g).bfloat16()
    want = layers.routed_experts_ref(x, ids.numpy(), oracle_expert_getter(per, gated, inter), gated, e_n=len(counts))
    ones = torch.ones(m, 1, device="cuda")
    assert _lib.lib().hb_tune(b"w3_tile", 1) == 0
    try:
        got, again = (w3_moe.w3_moe(ex, x.cuda(), ids.cuda(), ones, experts_total=total) for _ in range(2))
    finally:
        _lib.lib().hb_tune(b"w3_tile", 0)
    mx, nr = errors(got, want)
    assert mx < MAX_REL and nr < NORM_REL, (mx, nr)
    assert torch.equal(got, again)


@pytest.mark.parametrize("total,more", [(t, []) for t in TOTALS] + [(0, MORE), (0, MOST)])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("hidden,inter", [(128, 256), (384, 128)])
def test_nvfp4_slots_of_every_height(hidden, inter, gated, total, more):
    from hibana_amd import _lib
    from tests.test_gpu_nvfp4_moe import _experts
    counts = COUNTS + more
    ex, (w1, s1, g1, w2, s2, g2) = _experts(len(counts), hidden, inter, gated, 4)
    m, ids, g = _call(counts, inter)
    x = torch.randn(m, hidden, generator=g).bfloat16()

    def get(i):
        return onv.unpack_fp4(w1[i], s1[i]) * g1[i], onv.unpack_fp4(w2[i], s2[i]) * g2[i]

    want = layers.routed_experts_ref(x, ids.numpy(), get, gated, e_n=len(counts))
    assert _lib.lib().hb_tune(b"nvfp4_tile", 1) == 0
    try:
        got = ex(x.cuda(), ids.cuda(), torch.ones(m, 1, device="cuda"), experts_total=total)
    finally:
        _lib.lib().hb_tune(b"nvfp4_tile", 0)
    mx, nr = errors(got, want)
    assert mx < MAX_REL and nr < NORM_REL, (mx, nr)


@pytest.mark.parametrize("m,panel", [(255, False), (256, True)])  # 16 rows an expert of 64, 0.79 M pairs x blocks
def test_w3_calls_from_sixteen_rows_an_expert(m, panel):
    """The two kernels add in different orders, so the bits say which one ran."""
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import w3_moe
    ex = synthetic.w3_experts(64, 2048, 1024, True, 3)  # 768 blocks an expert
    g = torch.Generator().manual_seed(m)
    ids = torch.stack([torch.randperm(64, generator=g)[:4] for _ in range(m)]).to(torch.int32).cuda()
    x, weights = torch.randn(m, 2048, generator=g).bfloat16().cuda(), torch.rand(m, 4, generator=g).cuda()
    results = []
    for tile in (0, 1, 2):
        assert _lib.lib().hb_tune(b"w3_tile", tile) == 0
        try:
            results.append(w3_moe.w3_moe(ex, x, ids, weights))
        finally:
            _lib.lib().hb_tune(b"w3_tile", 0)
    got, by_panel, by_stream = results
    assert not torch.equal(by_panel, by_stream) and torch.equal(got, by_panel if panel else by_stream)


def _most_rows(ex, m, x, topk=1):
    """The rows of the highest slot of the plan that the last call left in its workspace."""
    from hibana_amd import _lib
    torch.cuda.synchronize()
    head = _lib.workspace(x.cuda().device, 0).view(torch.int32)[:16 + 4 * (m * topk + 4096)].cpu()
    return int(head[16:16 + 4 * int(head[0])].view(-1, 4)[:, 2].max())


# rows an expert and the slots' height: 144 rows past the lines of the lower ones, however many, except where slots of 128 rows all
# run at once (two workgroups on each of 256 compute units) and 144 hold no whole expert; the three-bit format's 80 rows serve up to 60
# rows an expert at once and up to 72 past one round
@pytest.mark.parametrize("fmt,experts,inter,rows,height", [
    ("w3", 40, 512, 140, 144), ("w3", 40, 512, 150, 128), ("w3", 40, 1536, 150, 144), ("w3", 40, 1536, 250, 144), ("w3", 40, 1536, 260, 144),
    ("w3", 40, 1536, 700, 144), ("w3", 32, 128, 300, 128), ("w3", 40, 2048, 71, 80), ("w3", 40, 2048, 73, 128), ("w3", 40, 512, 59, 80),
    ("w3", 40, 512, 61, 128), ("nvfp4", 40, 512, 140, 144), ("nvfp4", 40, 512, 150, 128), ("nvfp4", 40, 1536, 150, 144),
    ("nvfp4", 40, 1536, 260, 144), ("nvfp4", 40, 2048, 45, 80), ("nvfp4", 40, 2048, 47, 128)])
def test_height_by_the_rows_an_expert(fmt, experts, inter, rows, height):
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import w3_moe
    ex = synthetic.w3_experts(experts, 128, inter, True, 3) if fmt == "w3" else synthetic.nvfp4_experts(experts, 128, 2 * inter, 3)
    counts = [2 * rows] + [rows] * (experts - 2)
    m, ids, g = _call(counts, rows)
    x, ones = torch.randn(m, 128, generator=g).bfloat16().cuda(), torch.ones(m, 1, device="cuda")
    key = b"w3_tile" if fmt == "w3" else b"nvfp4_tile"
    assert _lib.lib().hb_tune(key, 1) == 0
    try:
        w3_moe.w3_moe(ex, x, ids.cuda(), ones) if fmt == "w3" else ex(x, ids.cuda(), ones)
    finally:
        _lib.lib().hb_tune(key, 0)
    assert _most_rows(ex, m, x) == min(height, 2 * rows)


@pytest.mark.parametrize("fmt", ["w3", "nvfp4"])
def test_low_slots_refuse_nothing(fmt):
    """Ids that all lie in a small share of the experts: 3.3 million pairs are more slots of 48 rows than a call may have, and fewer
    of 128."""
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import w3_moe
    m, topk, named = 51200, 64, 200000
    ex = synthetic.w3_experts(64, 128, 128, True, 3) if fmt == "w3" else synthetic.nvfp4_experts(64, 128, 128, 3)
    g = torch.Generator(device="cuda").manual_seed(1)
    ids = torch.rand(m, 64, device="cuda", generator=g).argsort(1).to(torch.int32)
    x, weights = torch.randn(m, 128, device="cuda", generator=g).bfloat16(), torch.rand(m, topk, device="cuda", generator=g)
    call = (lambda total: w3_moe.w3_moe(ex, x, ids, weights, experts_total=total)) if fmt == "w3" else (lambda total: ex(x, ids, weights, experts_total=total))
    key = b"w3_tile" if fmt == "w3" else b"nvfp4_tile"
    assert _lib.lib().hb_tune(key, 1) == 0  # the panel kernel for both
    try:
        assert torch.equal(call(named), call(0))
    finally:
        _lib.lib().hb_tune(key, 0)
