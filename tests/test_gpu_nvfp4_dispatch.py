"""Which kernel serves a dense NVFP4 product of more than sixteen rows, around the lines of the rule. The two kernels add in
different orders, so the bits say which one ran."""
import pytest
import torch

from tests.util import MAX_REL, NORM_REL, errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,m,room,relu2,stream", [
    (2048, 5120, 17, True, 0, True), (2048, 5120, 48, True, 1, True), (5120, 5120, 48, True, 0, True),  # long K, few blocks
    (5120, 5120, 49, True, 0, False),                                                                   # 80 blocks x 4 passes: more than fit at once
    (1024, 8192, 256, False, 0, True), (1024, 8192, 257, False, 0, False),                              # 16 blocks x 16 passes, x 17
    (2048, 4096, 17, True, 0, True),                                                                    # the fewest chunks of K (below, the two split K alike and give the same bits)
    (512, 12800, 64, True, 1, False), (512, 12800, 64, False, 1, True),                                 # K shared where there is room for it
    (2048, 5120, 16, True, 0, True),
])
def test_which_kernel_serves_a_call(n, k, m, room, relu2, stream):
    from hibana_amd import _lib, synthetic
    lib = _lib.lib()
    lin = synthetic.nvfp4_linear(n, k, n + k, global_scale=0.02)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
    need = lib.hb_nvfp4_gemm_room_bytes(m, n, k) if room else 0
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None

    def call(tile):
        y = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
        assert lib.hb_tune(b"nvfp4_tile", tile) == 0
        try:
            _lib.check(lib.hb_nvfp4_gemm_ws(_lib.ptr(x), m, _lib.ptr(lin.tiled), lin.global_scale, n, k, relu2, _lib.ptr(y), _lib.ptr(ws), need, _lib.stream()), "gemm")
        finally:
            lib.hb_tune(b"nvfp4_tile", 0)
        return y

    got, by_panel, by_stream = call(0), call(1), call(2)
    assert not torch.equal(by_panel, by_stream)
    assert torch.equal(got, by_stream if stream else by_panel)
    want = (x.float() @ lin.dequantize().T).bfloat16().float()
    mx, nr = errors(got, torch.relu(want) ** 2 if relu2 else want)
    assert mx < MAX_REL and nr < (2 * NORM_REL if relu2 else NORM_REL), (mx, nr)  # the square doubles a relative error


@pytest.mark.parametrize("n,k,m,room,stream", [
    (1024, 2048, 128, True, True), (1024, 3072, 129, True, False),                                      # 128 blocks x passes, shared tiles; past them
    (4096, 3072, 32, True, True),
    (512, 8192, 64, True, True), (512, 8192, 64, False, True), (512, 8320, 64, True, False),            # K up to 64 chunks, with room and without
    (448, 6144, 128, True, True), (448, 6144, 129, True, False), (448, 6272, 64, True, False),          # fewer blocks than dies: eight passes, 48 chunks
])
def test_which_kernel_serves_a_call_of_few_blocks(n, k, m, room, stream):
    test_which_kernel_serves_a_call(n, k, m, room, 0, stream)


@pytest.mark.parametrize("n,k,m", [(4096, 1536, 17), (4096, 3072, 32), (2112, 3200, 48), (1024, 2048, 33), (576, 640, 40), (8192, 512, 9), (2048, 5120, 12),
                                   (4160, 1152, 8), (1024, 4096, 3), (64, 128, 1)])
def test_shared_tiles_add_as_one_workgroup_does(n, k, m):
    """A block's tiles on two or four workgroups (one slot and several) against the same K split in one: the same bits."""
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import ops
    lib = _lib.lib()
    lin = synthetic.nvfp4_linear(n, k, n + k, global_scale=0.02)
    x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
    split, most = 1, 16 if m > 8 and k // 128 >= 24 else 8
    while 2 * split <= min(most, k // 128):
        split *= 2
    assert lib.hb_tune(b"nvfp4_tile", 2) == 0
    try:
        got = ops.nvfp4_linear(x, lin)
        assert lib.hb_tune(b"nvfp4_ksplit", split) == 0
        want = ops.nvfp4_linear(x, lin)
    finally:
        lib.hb_tune(b"nvfp4_tile", 0)
        lib.hb_tune(b"nvfp4_ksplit", 0)
    assert torch.equal(got, want)
