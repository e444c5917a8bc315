"""The dense SwiGLU block on its three-bit copies in one call (`w3.w3_mlp`): gate | up with the SiLU product and its E4M3 rounding in the
first launch's epilogue, bit for bit against the three calls it stands for (the same sums in the same order), around the lines of its shapes."""
import pytest
import torch

from tests.test_gpu_w3_mlp import _apart, _copies

pytestmark = pytest.mark.gpu


# h's 64-column blocks: 2, 32 and 128 in halves, 34 in three launches from five rows (long K), 42 in halves on 40 chunks, 130 and 256 whole, 258 and 384 in
# halves, 386 and 700 whole, 516 in halves. Splits of K a wavefront: one to four, the first of unequal length (11 and 41 chunks)
@pytest.mark.parametrize("hidden,inter", [(128, 128), (640, 2048), (1408, 1024), (256, 8192), (4096, 2176), (5248, 2688), (384, 8320), (5248, 8448), (1024, 16384),
                                          (512, 16512), (128, 24576), (1408, 24576), (256, 24704), (2560, 25600), (1152, 33024), (640, 44800)])
def test_one_call_has_the_bits_of_three(hidden, inter):
    from hibana_amd.kernels import w3
    gate_up, down = _copies(hidden, inter)
    for m in (1, 3, 4, 5, 12, 16, 17):
        x = torch.randn(m, hidden, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
        want = _apart(x, gate_up, down, 0)
        for _ in range(3):  # a read of the ring or of the exchange ahead of its data would not be wrong every time
            assert torch.equal(w3.w3_mlp(x, gate_up, down), want), m


@pytest.mark.parametrize("pairs", [32, 64, 192, 384])  # 32: gate and up meet inside a block, three launches
def test_gate_and_up_in_runs_have_the_bits_of_three(pairs):
    from hibana_amd.kernels import w3
    gate_up, down = _copies(256, 384)
    for m in (2, 9):
        x = torch.randn(m, 256, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
        assert torch.equal(w3.w3_mlp(x, gate_up, down, pairs), _apart(x, gate_up, down, pairs)), m


def test_rows_of_zeros_infinities_and_nan_have_the_bits_of_three():
    from hibana_amd.kernels import w3
    gate_up, down = _copies(256, 384)
    for m in (3, 7):
        x = torch.randn(m, 256, generator=torch.Generator().manual_seed(m)).bfloat16()
        x[0] = 0
        x[1, 5], x[2, 7] = float("inf"), float("nan")
        x = x.cuda()
        got, want = w3.w3_mlp(x, gate_up, down), _apart(x, gate_up, down, 0)
        assert torch.equal(got[0], torch.zeros_like(got[0])) and torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))


@pytest.mark.parametrize("m", [4, 17])
@pytest.mark.parametrize("change", [{"n": 96}, {"down_bits": 4}, {"down": 8}, {"y": 1}])  # (pointers: bytes off their boundary)
def test_what_the_down_projection_refuses_launches_nothing(change, m):
    from hibana_amd import _lib
    gate_up, down = _copies(256, 384)
    x = torch.randn(m, 256, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
    from hibana_amd.kernels import w3
    w3.tile(gate_up), w3.tile(down)
    scratch, y = torch.full((m * 384 // 8 * 41,), 0x7f, dtype=torch.uint8, device="cuda"), torch.zeros(m, 256, dtype=torch.bfloat16, device="cuda")
    call = {"x": x.data_ptr(), "m": m, "gate_up": gate_up.tiled.data_ptr(), "gate_up_rows": gate_up.row_scale.data_ptr(), "gate_up_lut": gate_up.lut, "inter": 384, "hidden": 256,
            "gate_up_bits": 3, "pairs": 0, "down": down.tiled.data_ptr(), "down_rows": down.row_scale.data_ptr(), "down_lut": down.lut, "n": 256, "down_bits": 3,
            "scratch": scratch.data_ptr(), "scratch_bytes": scratch.numel(), "y": y.data_ptr(), "stream": _lib.stream()}
    for k, v in change.items():
        call[k] = call[k] + v if k in ("down", "y") else v
    assert _lib.lib().hb_w3_mlp(*call.values()) == _lib.HB_EINVAL
    torch.cuda.synchronize()
    assert bool((scratch == 0x7f).all())
