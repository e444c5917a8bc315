"""The panel kernel (more than sixteen rows a weight block) at the edges of its cuts: one row more or less than whole row
tiles and slots, a single 64-row block and a single chunk of K, row tiles that only wide workgroups hold, K shared inside a
workgroup and among workgroups, calls of several shapes over one workspace."""
import numpy as np
import pytest
import torch

from oracle import layers, nvfp4_format as onv, w3_format as ow3
from tests.test_gpu_nvfp4 import _linear, _matrix
from tests.util import MAX_REL, NORM_REL, errors, random_w3, to_device_w3

pytestmark = pytest.mark.gpu
ROWS = [17, 32, 33, 64, 65, 80, 96, 97, 112, 113, 128, 129, 257]


@pytest.mark.parametrize("n,k", [(64, 128), (192, 640), (576, 1280), (320, 6400)])  # the last: K shared among workgroups up to 200 rows
def test_nvfp4_rows_around_whole_tiles(n, k):
    """Every call on one workspace, whose head the calls before it (other shapes, other cuts) have used and left zero."""
    from hibana_amd.kernels import ops
    packed, scales = _matrix(n, k, n + k, hi=8.0)
    lin = _linear(packed, scales, alpha=0.3, inv=1.0)
    dense = onv.unpack_fp4(packed, scales)
    for m in ROWS + ROWS[::-1]:
        x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16()
        mx, nr = errors(ops.nvfp4_linear(x.cuda(), lin), layers.nvfp4_dense_ref(x, dense, np.float32(0.3)))
        assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)


@pytest.mark.parametrize("codebook", ["lloyd", "lloyd2"])  # three-bit and two-bit tiles
@pytest.mark.parametrize("n,k", [(128, 128), (640, 640), (384, 1280)])
def test_w3_rows_around_whole_tiles(n, k, codebook):
    from hibana_amd import _lib
    from hibana_amd.kernels import w3
    packed, *_ = random_w3(n, k, 7, codebook)
    dev = to_device_w3(packed)
    dense = ow3.dequantize(packed)
    assert _lib.lib().hb_tune(b"w3_tile", 1) == 0  # (these matrices are too small for the kernel to be the faster one)
    try:
        for m in [1, 16] + [m for m in ROWS if m <= w3.MAX_ROWS]:
            x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16()
            got = w3.w3_linear(x.cuda(), dev)
            mx, nr = errors(got, layers.dense_ref(x, dense))
            assert mx < MAX_REL and nr < NORM_REL, (m, mx, nr)
            assert torch.equal(w3.w3_linear(x.cuda(), dev), got), m
    finally:
        _lib.lib().hb_tune(b"w3_tile", 0)


@pytest.mark.parametrize("m", [20, 21, 48, 77, 128])
def test_w3_calls_the_library_gives_to_the_panel(m):
    """n large enough for the built-in choice (24576 rows: 384 blocks), which is the panel kernel from 21 rows and the weight
    stream at 20: the two scale and add in different orders, so the bits say which one ran. Either way the product of the
    dequantized matrix."""
    from hibana_amd import _lib
    from hibana_amd.kernels import w3
    packed, *_ = random_w3(24576, 256, 3, "lloyd")
    dev = to_device_w3(packed)
    x = torch.randn(m, 256, generator=torch.Generator().manual_seed(m)).bfloat16()
    results = []
    for tile in (0, 1, 2):
        assert _lib.lib().hb_tune(b"w3_tile", tile) == 0
        try:
            results.append(w3.w3_linear(x.cuda(), dev))
        finally:
            _lib.lib().hb_tune(b"w3_tile", 0)
    got, panel, stream = results
    assert not torch.equal(panel, stream)
    assert torch.equal(got, panel if m > 20 else stream)
    mx, nr = errors(got, layers.dense_ref(x, ow3.dequantize(packed)))
    assert mx < MAX_REL and nr < NORM_REL, (mx, nr)


def test_nvfp4_calls_of_several_shapes_share_a_workspace():
    """Shared tiles' counters lie at a fixed place of the workspace: calls whose tiles number differently, one after the
    other on a stream, never take another's partial results for counters (a result nobody adds up is never stored)."""
    from hibana_amd import _lib
    from hibana_amd.kernels import ops
    shapes = [(5120, 2688), (512, 12800), (1024, 512), (320, 6400), (2688, 1024), (64, 128), (4096, 1280), (1024, 12800)]
    rows = (33, 200, 64, 512, 77, 333)
    assert sum(_lib.lib().hb_nvfp4_gemm_room_bytes(m, n, k) > 0 for m in rows for n, k in shapes) >= 12  # calls that share K, among calls that do not
    mats = []
    for i, (n, k) in enumerate(shapes):
        packed, scales = _matrix(n, k, i, hi=8.0)
        mats.append((_linear(packed, scales, alpha=0.3, inv=1.0), torch.from_numpy(onv.unpack_fp4(packed, scales)).cuda()))
    for m in rows:
        for (n, k), (lin, dense) in zip(shapes, mats):
            x = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
            junk = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")  # what the result's memory may hold before
            del junk
            got = ops.nvfp4_linear(x, lin)
            mx, nr = errors(got, ((x.float() @ dense.T) * 0.3).bfloat16())
            assert mx < MAX_REL and nr < NORM_REL, (m, n, k, mx, nr)


@pytest.mark.parametrize("m,n,k", [(64, 25600, 1280), (64, 512, 12800)])  # a cut that shares no K, one that does
def test_nvfp4_linear_holds_the_room_its_cut_uses(m, n, k, monkeypatch):
    from hibana_amd import _lib, synthetic
    from hibana_amd.kernels import ops
    asked, real = [], _lib.workspace
    monkeypatch.setattr(_lib, "workspace", lambda device, need, kind="moe": asked.append(need) or real(device, need, kind))
    ops.nvfp4_linear(torch.zeros(m, k, dtype=torch.bfloat16, device="cuda"), synthetic.nvfp4_linear(n, k, 1))
    room = _lib.lib().hb_nvfp4_gemm_room_bytes(m, n, k)
    assert asked == ([room] if room else []) and (room > 0) == (k == 12800)


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("mode,shift", [(1, 0), (2, 0), (2, 4)])  # FP32 and BF16 pair outputs; BF16 ones that start off a 16-byte boundary (shift: elements)
def test_routed_slots_around_whole_row_tiles(gated, mode, shift):
    """An expert a row count: every number of row tiles of a slot, a row more or less, two slots, none; the rows leave as whole
    lines where the output allows, else four columns at a time."""
    import ctypes as C
    from hibana_amd import _lib
    from hibana_amd.kernels import w3_moe
    from tests.util import oracle_expert_getter, random_experts
    counts = [1, 15, 16, 17, 33, 48, 0, 64, 65, 81, 97, 112, 127, 128, 129, 250]
    hidden, inter, m = 256, 384, sum(counts)
    ex, per = random_experts(len(counts), hidden, inter, gated, 5)
    w3_moe.tile(ex)
    g = torch.Generator().manual_seed(m)
    ids = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts))[torch.randperm(m, generator=g)].to(torch.int32)[:, None]
    x = torch.randn(m, hidden, generator=g).bfloat16()
    want = layers.routed_experts_ref(x, ids.numpy(), oracle_expert_getter(per, gated, inter), gated, e_n=len(counts))
    lib, st = _lib.lib(), w3_moe._struct(ex)
    dtype = torch.float32 if mode == 1 else torch.bfloat16
    guard = 64
    out = torch.full((m * hidden + shift + guard,), 7.0, dtype=dtype, device="cuda")
    need = w3_moe._workspace_bytes(st, m, 1, False)
    xd, idd, wd = x.cuda(), ids.cuda(), torch.ones(m, 1, device="cuda")
    assert lib.hb_tune(b"w3_tile", 1) == 0
    try:
        _lib.check(lib.hb_w3_moe_among(C.byref(st), 0, _lib.ptr(xd), _lib.ptr(idd), _lib.ptr(wd), m, 1, mode, C.c_void_p(out.data_ptr() + shift * out.element_size()),
                                       _lib.ptr(_lib.workspace(xd.device, need)), need, _lib.stream()), "w3_moe")
    finally:
        lib.hb_tune(b"w3_tile", 0)
    mx, nr = errors(out[shift:shift + m * hidden].view(m, hidden), want)
    assert mx < MAX_REL and nr < NORM_REL, (mx, nr)
    assert bool((out[:shift] == 7).all()) and bool((out[shift + m * hidden:] == 7).all())


@pytest.mark.parametrize("n,k", [(64, 128), (192, 640), (576, 1280), (320, 6400)])
def test_nvfp4_rows_around_whole_tiles_on_the_panel(n, k):
    """The same with the panel kernel for every size (few blocks are the weight stream's otherwise)."""
    from hibana_amd import _lib
    assert _lib.lib().hb_tune(b"nvfp4_tile", 1) == 0
    try:
        test_nvfp4_rows_around_whole_tiles(n, k)
    finally:
        _lib.lib().hb_tune(b"nvfp4_tile", 0)
