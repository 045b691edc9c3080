"""The many-rows kernel of the weight-only form (csrc/gemm_w2a16_tiled.hip) at the tolerance of tests/test_w2a16.py: both
tile heights, K halves inside a workgroup, K splits, ragged edges, both activation types, zero-points beyond the two
bits of a code.  The shapes are past the sizes where the few-rows kernel is the faster one (about 2100 strips of 64
channels x blocks of 16 rows), too large for the oracle's loops: its sum, sum_g scale * sum_k x * (code - zp), and the sum
of the terms' magnitudes are taken in float64 on the GPU, and one row is held to the oracle itself."""
import numpy as np
import pytest
import torch

from slimkernels_amd import _lib, workloads
import parity_utils as pu
from test_w2a16 import _check
from test_w2a16_plan import plan

pytestmark = pytest.mark.gpu


def _run(gpu_ops, oracle, M, N, K, g, mode, xdt, out, split, zero=None):
    case = pu.small_case(M, N, K, g, mode, seed=M * 7 + N, out_dtype=out)
    packed, scales, zero_q = pu.quantized_weight(case)
    wide_zero = zero is not None
    zero = zero_q if zero is None else zero(np.asarray(scales).shape)
    x = torch.from_numpy(workloads.make_activation(case)).to(getattr(torch, xdt)).cuda()
    if wide_zero:
        w = gpu_ops.repack_w2(packed, scales, zero, g)
    else:
        w, _ = pu.device_inputs(gpu_ops, case, packed, scales, zero, workloads.make_activation(case))
    codes = oracle.np_unpack(packed)
    zp = np.broadcast_to(np.asarray(zero), np.asarray(scales).shape)
    deq = torch.from_numpy(codes).cuda().double().reshape(N, K // g, g)
    deq -= torch.from_numpy(zp.T.copy()).cuda().double()[:, :, None]
    deq *= torch.from_numpy(np.asarray(scales, np.float16).T.copy()).cuda().double()[:, :, None]
    deq = deq.reshape(N, K)
    want = (x.double() @ deq.t()).cpu().numpy()
    mag = (x.double().abs() @ deq.abs_().t()).cpu().numpy()
    del deq
    bits = x[:1].view(torch.int16).cpu().numpy().view(np.uint16 if xdt == "bfloat16" else np.float16)
    row, _ = oracle.w2a16_reference_forward(bits, codes, scales, zp, g, x_bf16=xdt == "bfloat16")
    np.testing.assert_allclose(want[:1], row, rtol=1e-9, atol=1e-9 * np.abs(row).max())
    y = gpu_ops.w2a16_gemm(x, w, pu.torch_dtype(case), split_k=split)
    _check(y, want, mag, out == "bfloat16", "W2A16 many rows")
    wide = torch.zeros((M, K + 8), dtype=x.dtype, device="cuda")
    wide[:, :K] = x
    y2 = gpu_ops.w2a16_gemm(wide[:, :K], w, pu.torch_dtype(case), split_k=split)
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


@pytest.mark.parametrize("M,N,K,g,mode,xdt,out,split", [
    (300, 16448, 256, 128, "sym", "float16", "float16", 1),       # 128-row tiles, four steps, one strip in the last channel tile
    (1000, 16384, 512, 128, "ref", "float16", "bfloat16", 0),     # 128-row tiles
    (1000, 16384, 512, 64, "asym", "bfloat16", "bfloat16", 0),
    (250, 16384, 2048, 64, "asym", "bfloat16", "bfloat16", 1),    # two K halves in a workgroup
    (130, 14337, 2048, 128, "asym", "float16", "float16", 1),     # the same, ragged N: 2-byte stores
    (65, 28680, 4096, 256, "sym", "bfloat16", "float16", 1),      # the same, one row past a tile
    (300, 4096, 14336, 128, "sym", "float16", "float16", 0),      # halves and splits
    (300, 4097, 14336, 128, "asym", "bfloat16", "bfloat16", 5),   # splits of unequal length, scalar partial sums
    (700, 4096, 7168, 256, "asym", "float16", "float16", 0),
])
def test_w2a16_many_rows_against_the_oracle(gpu_ops, oracle, M, N, K, g, mode, xdt, out, split):
    print(f"W2A16 many rows M={M} N={N} K={K} g={g} {mode} {xdt} -> {out} split={split}", flush=True)
    _run(gpu_ops, oracle, M, N, K, g, mode, xdt, out, split)


@pytest.mark.parametrize("xdt", ["float16", "bfloat16"])
def test_w2a16_many_rows_with_zero_points_beyond_the_codes(gpu_ops, oracle, xdt):
    _run(gpu_ops, oracle, 300, 16448, 256, 64, "asym", xdt, "bfloat16", 1,
         zero=lambda shape: np.random.default_rng(3).integers(0, 256, shape).astype(np.uint8))


def test_w2a16_many_rows_with_a_split_count_that_does_not_divide(gpu_ops, oracle):
    """48 pairs of steps in nine splits: six each, so the ninth has no work and is not launched."""
    assert plan(33, 16384, 6144, 128, 9) == (64, 8, 1)
    _run(gpu_ops, oracle, 33, 16384, 6144, 128, "asym", "float16", "float16", 9)


def test_w2a16_partial_sums_are_not_kept(gpu_ops):
    """A call whose K is split leaves nothing behind on the weight or in the allocator."""
    w = gpu_ops.W2A16Linear.from_float(torch.randn((4096, 8192), device="cuda", dtype=torch.float16), 128).weight
    x = torch.randn((300, 8192), device="cuda", dtype=torch.float16)
    assert plan(300, 4096, 8192, 128)[1] > 1
    out = torch.empty((300, 4096), device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    gpu_ops.w2a16_gemm(x, w, out=out)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before
    assert torch.equal(out, gpu_ops.w2a16_gemm(x, w))


def test_w2a16_prompt_without_workspace(gpu_ops):
    """NULL for the workspace of a prompt the library would rather split: it runs unsplit, with the bits of split_k = 1."""
    L = _lib.lib()
    M, N, K, g = 300, 14336, 4096, 128
    w = gpu_ops.W2A16Linear.from_float(torch.randn((N, K), device="cuda", dtype=torch.float16), g).weight
    x = torch.randn((M, K), device="cuda", dtype=torch.float16)
    assert plan(M, N, K, g)[1] > 1 and plan(M, N, K, g, 0, 0)[1] == 1
    out = torch.zeros((M, N), device="cuda", dtype=torch.float16)
    stream = torch.cuda.current_stream()
    _lib.check(L.slimk_w2a16_gemm(x.data_ptr(), K, _lib.F16, w.w_r.data_ptr(), w.s_r.data_ptr(), None, w.zp_const, M, N, K, g,
                                  out.data_ptr(), N, _lib.F16, None, 0, 0, stream.cuda_stream))
    assert torch.equal(out, gpu_ops.w2a16_gemm(x, w, split_k=1))


@pytest.mark.parametrize("M,N,K,g,rows", [(16384, 1, 128, 128, 64), (16384, 4, 128, 64, 64), (16384, 7, 128, 128, 64), (16384, 8, 128, 128, 64),
                                          (8192, 100, 128, 128, 64), (20000, 103, 128, 64, 128), (700, 14337, 2048, 128, 64)])
def test_w2a16_bias_of_rows_that_are_no_whole_pieces(gpu_ops, M, N, K, g, rows):
    """A bias of fewer than eight channels, or of a number that is no multiple of eight, in an unsplit call of the many-rows kernel:
    the sum of two tensors, bit for bit.  (The bias lies inside a longer tensor.)"""
    assert plan(M, N, K, g)[:2] == (rows, 1)
    print(f"W2A16 bias M={M} N={N} K={K} g={g}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N)
    layer = gpu_ops.W2A16Linear.from_float(torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16), g)
    x = torch.randn((M, K), generator=gen, device="cuda", dtype=torch.float16)
    bias = torch.randn((N + 128,), generator=gen, device="cuda", dtype=torch.float16)[64:64 + N]
    plain = layer(x)
    layer.bias = bias
    assert torch.equal(layer(x).view(torch.int16), (plain + bias).view(torch.int16))
