"""The package imports under a torch that was built without a GPU backend (its configuration, checkpoint and host code run on
the CPU); only a kernel call needs one."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
import torch
for name in [n for n in dir(torch._C) if n.startswith("_cuda_")]:
    delattr(torch._C, name)
import hibana_amd
from hibana_amd import _lib
from hibana_amd.kernels import b12x_moe, nemotron_moe, ops, w3, w3_moe
from hibana_amd.model import flashnext_moe, mlp
from hibana_amd.weights import linear, modelopt, w3_checkpoint
try:
    ops.silu_and_mul(torch.zeros(2, 8, dtype=torch.bfloat16))
except RuntimeError as error:
    assert "GPU" in str(error)
else:
    raise SystemExit("a kernel call without a GPU must raise")
print("imported")
"""


def test_import_without_gpu_backend():
    run = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and run.stdout.strip() == "imported", run.stderr
