"""The many-rows kernel of the weight-only form (csrc/gemm_w2a16_tiled.hip) against the float64 restatement, at the
tolerance of tests/test_w2a16.py: tile edges, remainders, K splits (even ones and ones that leave the last split short or
empty), both activation types, zero-points beyond the two bits of a code."""
import numpy as np
import pytest
import torch

from slimkernels_amd import workloads
import parity_utils as pu
from test_w2a16 import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,g,mode,xdt,out,split", [
    (48, 64, 128, 128, "sym", "float16", "float16", 1),        # two steps, one strip of four
    (64, 256, 256, 64, "asym", "bfloat16", "bfloat16", 1),
    (65, 264, 1024, 128, "ref", "float16", "bfloat16", 1),     # one row past a tile, a fifth strip
    (100, 1001, 1024, 256, "asym", "float16", "float16", 0),   # ragged N: 2-byte stores or scalar partial sums
    (129, 320, 1920, 128, "sym", "bfloat16", "float16", 3),    # 30 steps in three splits of 10
    (130, 192, 1920, 64, "asym", "float16", "bfloat16", 3),
    (200, 128, 3584, 256, "sym", "float16", "float16", 3),     # 56 steps: splits of 19, 19 and 18
    (300, 512, 4096, 128, "asym", "bfloat16", "bfloat16", 0),
    (1030, 4160, 256, 128, "sym", "float16", "float16", 0),    # many tiles
])
def test_w2a16_many_rows_against_the_oracle(gpu_ops, oracle, M, N, K, g, mode, xdt, out, split):
    print(f"W2A16 many rows M={M} N={N} K={K} g={g} {mode} {xdt} -> {out} split={split}", flush=True)
    case = pu.small_case(M, N, K, g, mode, seed=M * 7 + N, out_dtype=out)
    packed, scales, zero = pu.quantized_weight(case)
    x = torch.from_numpy(workloads.make_activation(case)).to(getattr(torch, xdt))
    want, mag = oracle.w2a16_reference_forward(x.view(torch.int16).numpy().view(np.uint16 if xdt == "bfloat16" else np.float16),
                                               oracle.np_unpack(packed), scales, zero, g, x_bf16=xdt == "bfloat16")
    w, _ = pu.device_inputs(gpu_ops, case, packed, scales, zero, workloads.make_activation(case))
    y = gpu_ops.w2a16_gemm(x.cuda(), w, pu.torch_dtype(case), split_k=split)
    _check(y, want, mag, out == "bfloat16", "W2A16 many rows")
    wide = torch.zeros((M, K + 8), dtype=x.dtype, device="cuda")
    wide[:, :K] = x.cuda()
    y2 = gpu_ops.w2a16_gemm(wide[:, :K], w, pu.torch_dtype(case), split_k=split)
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


@pytest.mark.parametrize("xdt", ["float16", "bfloat16"])
def test_w2a16_many_rows_with_zero_points_beyond_the_codes(gpu_ops, oracle, xdt):
    M, N, K, g = 70, 128, 256, 64
    case = pu.small_case(M, N, K, g, "asym", seed=11)
    packed, scales, _ = pu.quantized_weight(case)
    zero = np.random.default_rng(3).integers(0, 256, scales.shape).astype(np.uint8)
    x = torch.from_numpy(workloads.make_activation(case)).to(getattr(torch, xdt))
    want, mag = oracle.w2a16_reference_forward(x.view(torch.int16).numpy().view(np.uint16 if xdt == "bfloat16" else np.float16),
                                               oracle.np_unpack(packed), scales, zero, g, x_bf16=xdt == "bfloat16")
    w = gpu_ops.repack_w2(packed, scales, zero, g)
    _check(gpu_ops.w2a16_gemm(x.cuda(), w, torch.bfloat16, split_k=1), want, mag, True, "W2A16 large zero-points")
