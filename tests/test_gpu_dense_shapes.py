"""Dense calls of at most sixteen rows where the rule for their workgroups' shape turns: blocks just below and from 768, fewer
chunks of K than a split of four or eight has shares, rows on both sides of the few-row bodies. The shape decides how K is
split and how many blocks a workgroup takes, never what is summed: each against the product of the dequantized matrix (in
FP64 on the CPU for the columns at the start, around the last run of blocks and at the end)."""
import pytest
import torch

from tests.util import MAX_REL, NORM_REL, errors

pytestmark = pytest.mark.gpu
ROWS = [1, 4, 5, 8, 9, 16]


def _columns(n):
    return torch.unique(torch.cat([torch.arange(64), torch.arange(n // 2, n // 2 + 64), torch.arange(n - 5 * 64, n)]))


def _check(lin, call, n, k):
    cols = _columns(n)
    dense = lin.dequantize()[cols.cuda()].double().cpu()
    for m in ROWS:
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16()
        got = call(x.cuda())
        assert got.shape == (m, n)
        mx, nr = errors(got[:, cols.cuda()], x.double() @ dense.T)
        assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)


@pytest.mark.parametrize("blocks", [130, 766, 770])
@pytest.mark.parametrize("chunks", [1, 3, 4, 7, 8, 12, 31, 32])
def test_w3_shapes(blocks, chunks):
    from types import SimpleNamespace
    from hibana_amd import synthetic
    from hibana_amd.kernels import w3
    n, k = blocks * 64, chunks * 128
    for codebook in ("lloyd", "lloyd2"):
        lin = synthetic.w3_matrix(n, k, 3, codebook=codebook)
        dense = w3.dequantize(lin)
        tiled = w3.tile(lin)
        _check(SimpleNamespace(dequantize=lambda: dense), lambda x: w3.w3_linear(x, tiled), n, k)


@pytest.mark.parametrize("blocks", [5, 300, 302, 767, 768])
@pytest.mark.parametrize("chunks", [1, 3, 7, 8, 11, 12])
def test_nvfp4_shapes(blocks, chunks):
    from hibana_amd import synthetic
    from hibana_amd.kernels import ops
    n, k = blocks * 64, chunks * 128
    lin = synthetic.nvfp4_linear(n, k, 3)
    _check(lin, lambda x: ops.nvfp4_linear(x, lin), n, k)


def _general_split(blocks, chunks, want):
    """How many ways the rule for any launch splits K: until there are `want` wavefronts, four chunks each at least."""
    ks = 1
    while ks < 16 and blocks * ks < want and chunks // (2 * ks) >= 4:
        ks *= 2
    return ks


# sizes that keep the general rule's split
@pytest.mark.parametrize("rows,blocks,chunks", [(1, 768, 16), (4, 800, 40), (4, 1200, 12), (2, 2374, 9), (1, 258, 8), (4, 512, 14), (16, 770, 8), (8, 800, 16),
                                                (12, 1026, 16), (16, 2374, 4)])
@pytest.mark.parametrize("codebook", ["lloyd", "lloyd2"])
def test_w3_shapes_that_split_k_as_any_launch(rows, blocks, chunks, codebook):
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import w3
    mat = synthetic.w3_matrix(blocks * 64, chunks * 128, 3, codebook=codebook)
    x = torch.randn(rows, chunks * 128, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
    got = w3.w3_linear(x, mat)
    try:
        assert _lib.lib().hb_tune(b"w3_ksplit", _general_split(blocks, chunks, 8192)) == 0
        want = w3.w3_linear(x, mat)
    finally:
        _lib.lib().hb_tune(b"w3_ksplit", 0)
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,blocks,chunks", [(1, 258, 12), (2, 400, 8), (1, 512, 15), (8, 302, 10), (4, 514, 7), (4, 768, 40), (8, 1200, 12), (1, 2374, 24)])
def test_nvfp4_shapes_that_split_k_as_any_launch(rows, blocks, chunks):
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import ops
    lin = synthetic.nvfp4_linear(blocks * 64, chunks * 128, 3)
    x = torch.randn(rows, chunks * 128, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
    got = ops.nvfp4_linear(x, lin)
    try:
        assert _lib.lib().hb_tune(b"nvfp4_ksplit", _general_split(blocks, chunks, 4096)) == 0
        want = ops.nvfp4_linear(x, lin)
    finally:
        _lib.lib().hb_tune(b"nvfp4_ksplit", 0)
    assert torch.equal(got, want)
