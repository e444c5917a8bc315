"""NVFP4 dense calls of few blocks, whose row tiles go to two or four workgroups: the bodies of four, eight and sixteen rows, one
slot and several, K from one chunk to more than the splits, block counts on both sides of the lines (64 and 128 blocks times slots)
and off the eight dies."""
import numpy as np
import pytest
import torch

from oracle import layers, nvfp4_format as onv
from tests.test_gpu_nvfp4 import _linear, _matrix
from tests.util import MAX_REL, NORM_REL, errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("relu2", [False, True])
@pytest.mark.parametrize("n,k", [(64, 128), (192, 384), (576, 2048), (4096, 256), (4160, 1152), (8192, 128), (8256, 256)])
def test_row_tiles_of_a_block(n, k, relu2):
    from hibana_amd.kernels import ops
    packed, scales = _matrix(n, k, n + k, hi=8.0)
    lin = _linear(packed, scales, alpha=0.3, inv=1.0)
    dense = onv.unpack_fp4(packed, scales)
    for m in (1, 3, 4, 5, 8, 9, 16):
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16()
        got = ops.nvfp4_linear(x.cuda(), lin, relu2=relu2)
        mx, nr = errors(got, layers.nvfp4_dense_ref(x, dense, np.float32(0.3), relu2=relu2))
        assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)
        assert torch.equal(ops.nvfp4_linear(x.cuda(), lin, relu2=relu2), got), m


@pytest.mark.parametrize("m", [17, 32, 33, 64])
def test_long_k_in_several_slots(m):
    """32 chunks and more on few blocks: the weight stream's passes side by side, each block's tiles on several workgroups."""
    from hibana_amd.kernels import ops
    packed, scales = _matrix(1024, 4608, m, hi=8.0)
    lin = _linear(packed, scales, alpha=0.3, inv=1.0)
    x = torch.randn(m, 4608, generator=torch.Generator().manual_seed(m)).bfloat16()
    mx, nr = errors(ops.nvfp4_linear(x.cuda(), lin), layers.nvfp4_dense_ref(x, onv.unpack_fp4(packed, scales), np.float32(0.3)))
    assert mx < MAX_REL and nr < NORM_REL, (mx, nr)
