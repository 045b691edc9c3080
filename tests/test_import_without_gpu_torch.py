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
