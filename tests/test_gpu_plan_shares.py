"""The plan of a call of many pairs, made by workgroups that each place a share of them: pair counts around the shares' edges
(256 pairs from all ids, 1024 from a table of counts) and around the sizes where one form hands over to the next, against the
oracle's stable sort."""
import pytest
import torch

from tests.test_gpu_workspace import _check_plan, _read_plan
from tests.util import random_experts

pytestmark = pytest.mark.gpu
E = 64


@pytest.fixture(scope="module")
def experts():
    return random_experts(E, 128, 128, True, 21)[0], random_experts(1, 128, 128, True, 22)[0]


@pytest.mark.parametrize("m,topk", [(1023, 1), (1024, 1), (1025, 1), (320, 4), (427, 6), (4097, 1), (8191, 1), (8192, 1), (8193, 1), (1303, 7), (16384, 4), (65537, 1)])
@pytest.mark.parametrize("base,count,shared", [(0, E, True), (16, 33, False)])
def test_shares_of_a_plan(experts, m, topk, base, count, shared):
    from hibana_amd import _lib
    from hibana_amd.kernels import w3_moe
    ex, sh = experts
    part = w3_moe.W3Experts(ex.planes13[base:base + count], ex.scales13[base:base + count], ex.row13[base:base + count], ex.planes2[base:base + count],
                            ex.scales2[base:base + count], ex.row2[base:base + count], ex.codebook, ex.lut, ex.fc2_codebook, ex.fc2_lut, base=base)
    g = torch.Generator().manual_seed(m + base)
    ids = torch.randint(0, E + 2, (m, topk), generator=g).to(torch.int32)  # 64, 65: no expert; a row may name one twice
    ids[m // 3:m // 2] = 20  # a run on one expert, over several shares
    x, weights = torch.randn(m, 128, generator=g).bfloat16().cuda(), torch.rand(m, topk, generator=g).cuda()
    assert _lib.lib().hb_tune(b"w3_tile", 2) == 0  # the weight stream: slots of 16 rows
    try:
        if shared:
            w3_moe.moe_layer(part, x, ids.cuda(), weights, shared=sh)
        else:
            w3_moe.w3_moe(part, x, ids.cuda(), weights)
    finally:
        _lib.lib().hb_tune(b"w3_tile", 0)
    torch.cuda.synchronize()
    head, entries, slots, order = _read_plan(_lib.workspace(x.device, 0), w3_moe._struct(part), m, topk, shared)
    _check_plan(head, entries, slots, order, ids.numpy(), topk, base, count, m if shared else 0)


@pytest.mark.parametrize("m,topk", [(1366, 6), (2731, 3), (5000, 4), (65537, 1), (1365, 6)])  # 8196, 8193, 20000, 65537 pairs; 8190, which one workgroup plans
def test_three_launches_of_a_plan_beside_a_rounding_job(experts, m, topk):
    """E4M3 activations are rounded by further workgroups: from 8192 pairs the plan is counted, scanned and placed in a launch each."""
    from hibana_amd import _lib
    from hibana_amd.kernels import w3_moe
    ex, sh = experts
    g = torch.Generator().manual_seed(m)
    ids = torch.randint(0, E + 2, (m, topk), generator=g).to(torch.int32)
    ids[m // 3:m // 2] = 20
    x, weights = torch.randn(m, 128, generator=g).bfloat16().cuda(), torch.rand(m, topk, generator=g).cuda()
    w3_moe.moe_layer(ex, x, ids.cuda(), weights, shared=sh, e4m3=True)
    torch.cuda.synchronize()
    head, entries, slots, order = _read_plan(_lib.workspace(x.device, 0), w3_moe._struct(ex), m, topk, True)
    _check_plan(head, entries, slots, order, ids.numpy(), topk, 0, E, m)
