"""Weight objects that have served a call - and so keep the structure of their tensors' addresses that the library takes -
can be copied and pickled, and a copy's structure names the copy's tensors. No kernel runs: CPU tensors will do."""
import copy
import pickle

import pytest
import torch

from hibana_amd.kernels import nemotron_moe, w3_moe
from hibana_amd.model.flashnext_moe import MoeLayer


def _experts():
    ex = w3_moe.W3Experts(None, None, torch.ones(2, 256), None, None, torch.ones(2, 128), (1.0,), 1, (2.0,), 2, 0, torch.zeros(64, dtype=torch.uint8),
                          torch.zeros(64, dtype=torch.uint8), (256, 128), (128, 128))
    w3_moe._struct(ex)  # what a call does first
    return ex


def _small():
    small = nemotron_moe.SmallWeights(torch.ones(6, 512, dtype=torch.bfloat16), torch.zeros(2), torch.ones(512, 4, dtype=torch.bfloat16))
    small.struct()
    return small


WAYS = {"copy": copy.copy, "deepcopy": copy.deepcopy, "pickle": lambda o: pickle.loads(pickle.dumps(o))}


@pytest.mark.parametrize("way", WAYS)
def test_experts_that_served_a_call(way):
    ex = _experts()
    twin = WAYS[way](ex)
    got, want = w3_moe._struct(twin), w3_moe._struct(ex)
    assert (got.fc1, got.fc2) == (twin.tiled13.data_ptr(), twin.tiled2.data_ptr()) and got is not want
    assert (got.fc1 == want.fc1) == (way == "copy")
    assert (got.experts, got.base, got.hidden, got.inter, got.hidden_out, got.gated) == (want.experts, want.base, want.hidden, want.inter, want.hidden_out, want.gated)


@pytest.mark.parametrize("way", ["copy", "deepcopy", "pickle"])
def test_a_layer_that_served_a_call(way):
    layer = MoeLayer(torch.ones(2, 128, dtype=torch.bfloat16), torch.zeros(128), _experts(), 1)
    twin = WAYS[way](layer)
    assert torch.equal(twin.router, layer.router) and w3_moe._struct(twin.w3).fc1 == twin.w3.tiled13.data_ptr()


@pytest.mark.parametrize("way", WAYS)
def test_small_weights_that_served_a_call(way):
    small = _small()
    twin = WAYS[way](small)
    assert twin.struct().fc2 == twin.fc2.data_ptr() and (twin.struct().fc2 == small.struct().fc2) == (way == "copy")
