"""Every form the many-rows kernels run in (tile height, K splits, workgroups per CU, K halves), each at a size the planner
sends to it, which is asserted; on activations with a mean (behind a ReLU).

Digit form (csrc/gemm_mx.hip): against float64 from the same integers and scales, and bit for bit against the int8 tiled
kernel, which reproduces the oracle's bits, where K is in one piece and the levels are symmetric.  Weight-only form
(csrc/gemm_w2a16_tiled.hip): as tests/test_w2a16_tiled.py."""
import ctypes

import numpy as np
import pytest
import torch

from slimkernels_amd import _lib
import parity_utils as pu
from test_w2a16_plan import plan
from test_w2a16_tiled import _run

pytestmark = pytest.mark.gpu


def digits_plan(M, N, K, g):
    rows, splits = ctypes.c_int(), ctypes.c_int()
    _lib.check(_lib.lib().slimk_w2a8_linear_plan(M, N, K, g, ctypes.byref(rows), ctypes.byref(splits)))
    return rows.value, splits.value


def _weight(gpu_ops, N, K, g, mode, gen):
    """(packed, scales, zero) on the GPU; the groups are shifted, so that every zero-point 0..3 occurs with "asym"."""
    w = torch.randn((N, K // g, g), generator=gen, device="cuda")
    if mode == "asym":
        w += torch.randn((N, K // g, 1), generator=gen, device="cuda") * 1.5
    return gpu_ops.quantize_weight_gpu((w * 0.02).half().reshape(N, K).contiguous(), g, mode)


@pytest.mark.parametrize("out", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K,g,mode,rows,splits", [
    (65, 72, 1088, 64, "asym", 64, 1),           # 64-row tiles, two workgroups a CU; half a stage at the end
    (65, 72, 3200, 128, "asym", 64, 4),          # splits of 7, 7, 7 and 4 stages: odd numbers of groups
    (999, 8201, 1088, 64, "sym", 64, 1),         # 64-row tiles, three workgroups a CU
    (999, 8201, 1024, 128, "asym", 64, 1),
    (999, 8200, 1152, 128, "sym", 64, 1),
    (999, 3001, 6144, 64, "asym", 64, 4),        # the same with K split
    (900, 3000, 6144, 128, "sym", 64, 4),
    (300, 4100, 4096, 128, "asym", 64, 3),       # two workgroups a CU with K split
    (999, 14593, 1088, 64, "sym", 128, 1),       # 128-row tiles, nine stages
    (999, 14593, 1088, 64, "asym", 128, 1),
    (1000, 14592, 1152, 128, "sym", 128, 1),
    (999, 14600, 1152, 128, "asym", 128, 1),
    (1000, 14592, 1024, 256, "asym", 128, 1),    # a group of 256 over two stages
    (1000, 4104, 3072, 64, "sym", 128, 3),       # 128-row tiles with K split: eight stages each
    (999, 4105, 3072, 64, "asym", 128, 3),
    (1000, 4105, 4096, 128, "sym", 128, 3),      # 11, 11 and 10 stages
    (999, 4104, 4096, 128, "asym", 128, 3),
    (999, 4104, 4096, 256, "asym", 128, 3),      # splits of whole groups of 256
])
def test_digits(gpu_ops, M, N, K, g, mode, rows, splits, out):
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    print(f"digits form M={M} N={N} K={K} g={g} {mode} {out}", flush=True)
    assert digits_plan(M, N, K, g) == (rows, splits)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    packed, scales, zero = _weight(gpu_ops, N, K, g, mode, gen)
    w = gpu_ops.repack_w2(packed, scales, zero if mode == "asym" else None, g, zp_const=2)
    x = torch.randn((M, K), generator=gen, device="cuda").relu().half()
    dtype = getattr(torch, out)
    y = w2a8_linear_digits(x, w, dtype)
    qa = gpu_ops.quantize_act_int8(x, g)
    if mode == "sym" and splits == 1:
        assert torch.equal(y.view(torch.int16), gpu_ops.w2a8_gemm(qa, w, dtype, kernel="tiled", split_k=1).view(torch.int16))
    # float64, a drain of the kernel at a time (64 or 128 elements): the products are whole numbers below 2^53
    step = min(g, 128)
    shifts = torch.tensor([6, 4, 2, 0], device="cuda", dtype=torch.uint8)     # element 4 j lies in bits 7:6 of byte j
    stages = (K // 64 + 1) // 2
    per_split = -(-stages // splits)
    per_split += per_split % 2 if g == 256 else 0
    want = torch.zeros((M, N), dtype=torch.float64, device="cuda")
    run, held = torch.zeros_like(want), torch.zeros_like(want)    # a split's running sum; what it and its terms come to, in all
    for d in range(K // step):
        lo, group = d * step, d * step // g
        if lo % (per_split * 128) == 0:
            run.zero_()
        codes = ((packed[:, lo // 4:(lo + step) // 4, None] >> shifts) & 3).reshape(N, step).double()
        q = qa.q[:, lo:lo + step].double()
        sc, zp = scales[group].double(), zero[group].double() if mode == "asym" else torch.full((N,), 2.0, device="cuda", dtype=torch.float64)
        term = (q @ (codes - zp[:, None]).t().contiguous()) * sc
        offset = (2 - zp).abs() * sc * q.sum(1, keepdim=True).abs()
        want += term
        run += term
        held += run.abs() + term.abs() + 2 * offset + want.abs()
    want *= qa.s_a.double()[:, None]
    held *= qa.s_a.double()[:, None]
    # half an ULP of the output, the product with the token scale, and three roundings a drain
    ulp = torch.from_numpy(pu.ulp_of(want.float().cpu().numpy(), out == "bfloat16")).cuda()
    bad = (y.double() - want).abs() > 0.5 * ulp * (1 + 2.0 ** -7) + 2.0 ** -24 * (3 * held + want.abs())
    assert not bad.any(), int(bad.sum())


@pytest.mark.parametrize("lead,N,K,g,mode,bias,out", [
    ((4, 65), 4096, 8192, 64, "asym", True, "bfloat16"),     # fewer than 512 tiles, K split
    ((2, 48), 4096, 20480, 128, "sym", False, "float16"),    # 96 rows of a long reduction
    ((1025,), 14592, 512, 128, "sym", True, "float16"),      # 512 tiles and more
])
def test_layer_calls_on_the_digit_route(gpu_ops, monkeypatch, lead, N, K, g, mode, bias, out):
    from slimkernels_amd.torch import ops
    dtype = getattr(torch, out)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    b = torch.randn((N,), generator=gen, device="cuda").to(dtype) if bias else None
    layer = gpu_ops.W2A8Linear.from_float(torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16) * 0.02, g, mode,
                                          bias=b, out_dtype=dtype)
    x = torch.randn((*lead, K), generator=gen, device="cuda").to(dtype)
    rows = x.reshape(-1, K)
    assert ops.linear_digits_applies(rows.shape[0], layer.weight)
    int8 = ops.w2a8_gemm(ops.quantize_act_int8(rows, g), layer.weight, dtype)
    digits = ops.w2a8_linear_digits(rows, layer.weight, dtype)
    want = (digits + b if bias else digits).reshape(*lead, N)
    monkeypatch.setattr(ops, "w2a8_gemm", None)               # (the layer must not come by there)
    assert torch.equal(layer(x), want)
    if len(lead) == 2:                                        # rows that are not where reshape can leave them
        swapped = x.transpose(0, 1).contiguous().transpose(0, 1)
        assert not swapped.is_contiguous() and torch.equal(layer(swapped), want)
    assert torch.equal(layer(x.float()), want)                # (taken to the output type)
    # the two paths' outputs are the same numbers, rounded apart at most where sums were split
    assert ((digits.float() - int8.float()).norm() / int8.float().norm()).item() < 2.0 ** -12


@pytest.mark.parametrize("M,N,K,g,mode,xdt,out,split,form", [
    (735, 11008, 2048, 128, "sym", "float16", "float16", 0, (64, 1, 1)),       # four waves, 64 rows
    (735, 11009, 2048, 64, "asym", "bfloat16", "bfloat16", 1, (64, 1, 1)),
    (735, 11008, 2048, 256, "sym", "bfloat16", "float16", 1, (64, 1, 1)),
    (700, 11009, 2048, 128, "asym", "float16", "bfloat16", 1, (64, 1, 1)),
    (300, 11008, 2048, 128, "asym", "float16", "float16", 2, (64, 2, 1)),      # the same with K split
    (300, 11008, 2048, 256, "sym", "bfloat16", "float16", 2, (64, 2, 1)),
    (436, 4097, 4096, 64, "asym", "bfloat16", "bfloat16", 4, (64, 4, 1)),
    (435, 4104, 4096, 64, "sym", "float16", "bfloat16", 4, (64, 4, 1)),
    (200, 14337, 2048, 64, "asym", "float16", "float16", 2, (128, 2, 1)),      # 128 rows with K split
    (300, 4096, 8192, 128, "asym", "bfloat16", "float16", 0, (64, 3, 2)),      # halves and splits
])
def test_w2a16(gpu_ops, oracle, M, N, K, g, mode, xdt, out, split, form):
    print(f"W2A16 form M={M} N={N} K={K} g={g} {mode} {xdt} -> {out} split={split}", flush=True)
    assert plan(M, N, K, g, split) == form
    _run(gpu_ops, oracle, M, N, K, g, mode, xdt, out, split)


@pytest.mark.parametrize("xdt", ["float16", "bfloat16"])
def test_w2a16_four_waves_with_zero_points_beyond_the_codes(gpu_ops, oracle, xdt):
    assert plan(100, 16384, 256, 64, 1) == (64, 1, 1)
    _run(gpu_ops, oracle, 100, 16384, 256, 64, "asym", xdt, "bfloat16", 1,
         zero=lambda shape: np.random.default_rng(3).integers(0, 256, shape).astype(np.uint8))


def test_split_forms_recorded_into_a_graph(gpu_ops):
    """A split call of each many-rows kernel on its tiled form replays to the eager bits, with eager work in between."""
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    assert digits_plan(1000, 4104, 4096, 128) == (128, 3) and plan(300, 4096, 8192, 128) == (64, 3, 2)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    w8 = gpu_ops.W2A8Linear.from_float(torch.randn((4104, 4096), generator=gen, device="cuda", dtype=torch.float16), 128, "asym").weight
    w16 = gpu_ops.W2A16Linear.from_float(torch.randn((4096, 8192), generator=gen, device="cuda", dtype=torch.float16), 128).weight
    x8 = torch.randn((1000, 4096), generator=gen, device="cuda", dtype=torch.float16)
    x16 = torch.randn((300, 8192), generator=gen, device="cuda", dtype=torch.float16)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = [w2a8_linear_digits(x8, w8), gpu_ops.w2a16_gemm(x16, w16)]
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = [w2a8_linear_digits(x8, w8), gpu_ops.w2a16_gemm(x16, w16)]
    for _ in range(3):
        for y in got:
            y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for y, e in zip(got, want):
            assert torch.equal(y.view(torch.int16), e.view(torch.int16))
        w2a8_linear_digits(x8[:300], w8)
        gpu_ops.w2a16_gemm(x16[:100], w16)
