"""A three-bit dense call of at most four rows on few blocks: a block's row tiles on two or four workgroups, around the
numbers of blocks where the division changes and where the blocks do not fill the last turn of the compute dies."""
import pytest
import torch

from tests.util import MAX_REL, NORM_REL, errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128, 1152, 4096, 4224, 8192, 8320])  # 2, 18, 64 blocks in four parts, 66, 128 in two, 130 whole
@pytest.mark.parametrize("k", [128, 640, 2560])
def test_parts_of_a_block_against_the_product_and_the_sixteen_row_body(n, k):
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import w3
    mat = synthetic.w3_matrix(n, k, n + k)
    dense = w3.dequantize(mat).double()
    for m in (1, 2, 3, 4, 5):
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
        q, s = w3.quant_groups(x)
        got, got8 = w3.w3_linear(x, mat), w3.w3_linear(q, mat, s)
        mx, nr = errors(got, x.double() @ dense.T)
        assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)
        mx, nr = errors(got8, (q.double().reshape(m, -1, 32) * s.double()[:, :, None]).reshape(m, k) @ dense.T)
        assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)
        assert _lib.lib().hb_tune(b"w3_few", 2) == 0
        try:
            full = w3.w3_linear(x, mat)
        finally:
            _lib.lib().hb_tune(b"w3_few", 0)
        mx, nr = errors(got, full)
        assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)


@pytest.mark.parametrize("n", [128, 1152, 4096, 4224, 8192])  # 2, 18 and 64 blocks in four parts, 66 and 128 in two
@pytest.mark.parametrize("k", [128, 640, 2048, 5120])  # one chunk of K, fewer and more chunks than splits
def test_parts_of_a_block_on_the_sixteen_row_bodies(n, k):
    from hibana_amd import synthetic
    from hibana_amd.kernels import w3
    mat = synthetic.w3_matrix(n, k, n + k)
    dense = w3.dequantize(mat).double()
    for m in (5, 7, 8, 13, 16):
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
        q, s = w3.quant_groups(x)
        for _ in range(3):  # a read of the ring ahead of its data would not be wrong every time
            mx, nr = errors(w3.w3_linear(x, mat), x.double() @ dense.T)
            assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)
            mx, nr = errors(w3.w3_linear(q, mat, s), (q.double().reshape(m, -1, 32) * s.double()[:, :, None]).reshape(m, k) @ dense.T)
            assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)
