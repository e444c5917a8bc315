"""The gated layer from its input rows (`w3_moe.moe_layer_rows`): the router's product in the library's own launch (up to
ROUTER_ROWS rows) or handed in (beyond), then the chain of `moe_layer_logits` / `moe_layer_budget` / padded `route_topk`.

Rows and router hold small integers, so every logit is exact in FP32 whatever the order of its sum and the BF16 rounding
is the same wherever it is made: the layer must give the bits of the chain on torch's logits."""
import pytest
import torch

from tests.util import random_experts

pytestmark = pytest.mark.gpu


def _setup(e, hidden, m, seed):
    ex, _ = random_experts(e, hidden, 128, True, seed)
    shared, _ = random_experts(1, hidden, 128, True, seed + 1)
    g = torch.Generator().manual_seed(seed + 2)
    x = torch.randint(-2, 3, (m, hidden), generator=g).bfloat16().cuda()
    router = torch.randint(-1, 2, (e, hidden), generator=g).bfloat16().cuda()
    return ex, shared, x, router, (torch.randn(hidden, generator=g) * 0.05).cuda()


# row tiles of sixteen and their remainders, the last row of the library's product and the first beyond it; a hidden size
# whose K steps do not divide among the wavefronts (36 over sixteen), a router that ends inside a 16-column tile
@pytest.mark.parametrize("m", [1, 2, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize("e,hidden", [(30, 1152), (64, 256)])
def test_layer_from_rows_is_the_chain_on_its_logits(e, hidden, m):
    from hibana_amd.kernels import ops, w3_moe
    ex, shared, x, router, gate = _setup(e, hidden, m, 500 + e)
    logits = torch.mm(x, router.T)
    got = w3_moe.moe_layer_rows(ex, x, router, 6, shared=shared, gate_vec=gate)
    assert torch.equal(got, w3_moe.moe_layer_logits(ex, x, logits.float(), 6, shared=shared, gate_vec=gate))
    got = w3_moe.moe_layer_rows(ex, x, router, 6, 2, 12, shared=shared, gate_vec=gate)
    assert torch.equal(got, w3_moe.moe_layer_budget(ex, x, logits, 6, 2, 12, shared=shared, gate_vec=gate))
    slots = torch.ones(m, dtype=torch.int32, device="cuda")
    slots[m // 2] = 0  # a padded row names no expert
    ids, weights = ops.route_topk(logits, 6, slots)
    got = w3_moe.moe_layer_rows(ex, x, router, 6, slots=slots, shared=shared, gate_vec=gate)
    assert torch.equal(got, w3_moe.moe_layer(ex, x, ids, weights, shared=shared, gate_vec=gate))


@pytest.mark.parametrize("m", [10, 70])  # the router's product in the library and handed in
def test_verify_forwards_that_are_no_whole_requests(m):
    """Without slots the requests' length means nothing; with them the last request may be cut short."""
    from types import SimpleNamespace

    from hibana_amd.kernels import ops, w3_moe
    from hibana_amd.model.flashnext_moe import MoeLayer
    ex, shared, x, router, gate = _setup(30, 1152, m, 900)
    layer = MoeLayer(router, gate, ex, 6, shared=shared)
    assert torch.equal(layer(x, SimpleNamespace(mode="verify", seq_slots=None, verify_steps=4)), layer(x))
    slots = torch.ones(-(-m // 4), dtype=torch.int32, device="cuda")
    slots[1] = 0
    ids, weights = ops.route_topk(torch.mm(x, router.T), 6, slots, 4)
    got = layer(x, SimpleNamespace(mode="verify", seq_slots=slots, verify_steps=4))
    assert torch.equal(got, w3_moe.moe_layer(ex, x, ids, weights, shared=shared, gate_vec=gate))
    with pytest.raises(ValueError):
        layer(x, SimpleNamespace(mode="verify", seq_slots=slots[1:], verify_steps=4))


@pytest.mark.parametrize("m", [3, 70])
def test_a_router_off_the_vector_boundary(m):
    """A router sliced out of a larger tensor need not start on a 16-byte boundary."""
    from hibana_amd.model.flashnext_moe import MoeLayer
    ex, shared, x, router, gate = _setup(30, 256, m, 700)
    slice_ = torch.cat([router.new_zeros(4), router.flatten()])[4:].view_as(router)
    assert slice_.data_ptr() % 16 == 8 and slice_.is_contiguous()
    assert torch.equal(MoeLayer(slice_, gate, ex, 6, shared=shared)(x), MoeLayer(router, gate, ex, 6, shared=shared)(x))


@pytest.mark.parametrize("m", [256, 257, 263, 640])
def test_layer_routes_several_rows_a_workgroup(m):
    """From more rows than compute units the routing launch gives a workgroup eight rows; the last one to arrive plans."""
    from hibana_amd import synthetic
    from hibana_amd.kernels import ops, w3_moe
    ex = synthetic.w3_experts(48, 256, 128, True, 3)
    g = torch.Generator().manual_seed(m)
    x, logits = torch.randn(m, 256, generator=g).bfloat16().cuda(), (torch.randn(m, 48, generator=g) * 2).cuda()
    ids, wts = ops.route_topk(logits, 6)
    want = w3_moe.moe_layer(ex, x, ids, wts)
    for _ in range(2):
        got, got_ids, got_w = w3_moe.moe_layer_logits(ex, x, logits, 6, return_routing=True)
        assert torch.equal(got_ids, ids) and torch.equal(got_w, wts) and torch.equal(got, want)
