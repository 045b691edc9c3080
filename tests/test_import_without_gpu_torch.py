"""The package imports on a torch that was built without GPU support (its native module lacks the GPU accessors): the host
side (packing, plans, saved weights) is of use there, and a GPU call says what is missing by itself."""
import subprocess
import sys

PROGRAM = """
import torch
for name in [n for n in dir(torch._C) if n.startswith("_cuda_")]:
    delattr(torch._C, name)
import slimkernels_amd.torch as ops
assert ops.W2A8Linear is not None
try:
    ops.quantize_act_int8(torch.zeros((1, 128), dtype=torch.float16), 128)
except (ValueError, RuntimeError) as e:
    print("refused:", e)
else:
    raise SystemExit("a CPU tensor was taken")
"""


def test_import_without_the_gpu_accessors():
    done = subprocess.run([sys.executable, "-c", PROGRAM], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr[-2000:]
    assert "refused:" in done.stdout


# ... nor has it a native host side (which links against GPU support): what is refused is refused for the tensor it is
CALLS = """
import sys
import torch
for name in [n for n in dir(torch._C) if n.startswith("_cuda_")]:
    delattr(torch._C, name)
sys.modules["slimkernels_amd.torch._native"] = None      # (an ImportError)
import slimkernels_amd.torch as ops
from slimkernels_amd.torch import w4
from slimkernels_amd.torch.ops import W2A16Linear, w2a16_gemm
x = torch.zeros((2, 128), dtype=torch.float16)
w = ops.W2A8Weight(x, x, None, 2, 64, 128, 128)
calls = [lambda: ops.quantize_act_int8(x, 128), lambda: ops.W2A8Linear(w)(x), lambda: ops.W2A8Linear(w)(x[:1]), lambda: W2A16Linear(w)(x),
         lambda: w2a16_gemm(x, w), lambda: w4.W4A8Linear(w4.W4A8Weight(w, 64, 128, 128))(x)]
for i, call in enumerate(calls):
    try:
        call()
    except ValueError as e:
        assert "must live on the GPU" in str(e), (i, e)
    else:
        raise SystemExit(f"call {i} took a CPU tensor")
assert ops.w2a8_gemm_grouped([]) == []
print("all refused")
"""


def test_calls_without_a_native_host_side():
    done = subprocess.run([sys.executable, "-c", CALLS], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0 and "all refused" in done.stdout, done.stderr[-2000:]
