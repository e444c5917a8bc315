"""The dense SwiGLU block on its three-bit copies in one call (`w3.w3_mlp`): gate | up with the SiLU product and its E4M3 rounding in the
first launch's epilogue, against the three calls it stands for, around the lines of its shapes."""
import pytest
import torch

from tests.util import errors

pytestmark = pytest.mark.gpu

# The two have the same bits (tests/test_gpu_w3_mlp_bits.py); this limit allows for FP32 sums in another order, whose BF16 rounding may move a group's largest
# value, and with it the scale and the rounding of all its 32 codes.
REL = 1e-3


def _copies(hidden, inter, codebook="lloyd"):
    from hibana_amd import synthetic
    return synthetic.w3_matrix(2 * inter, hidden, hidden + inter, codebook=codebook), synthetic.w3_matrix(hidden, inter, hidden + inter + 1)


def _apart(x, gate_up, down, pairs):
    from hibana_amd.kernels import ops, w3
    q, s = ops.silu_mul_quant_groups(w3.w3_linear(x, gate_up), pairs, torch_chain=True)
    return w3.w3_linear(q, down, s)


# h's 64-column blocks: 2, 32 and 128 in halves, 34 in three launches (long K), 130 and 256 whole, 258 and 384 in halves two ways, 386 whole two ways
@pytest.mark.parametrize("hidden,inter", [(128, 128), (640, 2048), (256, 8192), (4096, 2176), (384, 8320), (1024, 16384), (512, 16512), (128, 24576), (256, 24704)])
def test_one_call_against_the_three_it_stands_for(hidden, inter):
    from hibana_amd.kernels import w3
    gate_up, down = _copies(hidden, inter)
    for m in (1, 3, 4, 5, 12, 16, 17):
        x = torch.randn(m, hidden, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
        want = _apart(x, gate_up, down, 0)
        for _ in range(3):  # a read of the ring or of the exchange ahead of its data would not be wrong every time
            mx, nr = errors(w3.w3_mlp(x, gate_up, down), want.double())
            assert nr < REL, (m, mx, nr)


@pytest.mark.parametrize("pairs", [32, 64, 192, 384])  # 32: gate and up meet inside a block, three launches
def test_gate_and_up_in_runs(pairs):
    from hibana_amd.kernels import w3
    gate_up, down = _copies(256, 384)
    for m in (2, 9):
        x = torch.randn(m, 256, generator=torch.Generator().manual_seed(m)).bfloat16().cuda()
        mx, nr = errors(w3.w3_mlp(x, gate_up, down, pairs), _apart(x, gate_up, down, pairs).double())
        assert nr < REL, (m, mx, nr)


def test_rows_of_zeros_infinities_and_nan():
    from hibana_amd.kernels import w3
    gate_up, down = _copies(256, 384)
    for m in (3, 7):
        x = torch.randn(m, 256, generator=torch.Generator().manual_seed(m)).bfloat16()
        x[0] = 0
        x[1, 5], x[2, 7] = float("inf"), float("nan")
        x = x.cuda()
        got, want = w3.w3_mlp(x, gate_up, down), _apart(x, gate_up, down, 0)
        assert torch.equal(got[0], torch.zeros_like(got[0])) and torch.equal(torch.isnan(got), torch.isnan(want))
        assert errors(got[3:], want[3:].double())[1] < REL if m > 3 else True


def test_a_two_bit_copy_and_refused_calls():
    from hibana_amd.kernels import w3
    gate_up, down = _copies(256, 384, codebook="lloyd2")
    x = torch.randn(4, 256, generator=torch.Generator().manual_seed(4)).bfloat16().cuda()
    assert torch.equal(w3.w3_mlp(x, gate_up, down), _apart(x, gate_up, down, 0))
    for bad in (x.float(), x[:, :128], x[:0], x.repeat(33, 1)):
        with pytest.raises(ValueError):
            w3.w3_mlp(bad, gate_up, down)
    with pytest.raises(ValueError):
        w3.w3_mlp(x, gate_up, down, pairs=40)
    with pytest.raises(RuntimeError):
        w3.w3_mlp(x.cpu(), gate_up, down)
