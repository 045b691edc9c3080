"""The digit form of a layer call (csrc/gemm_mx.hip): activations split into an fp4 and an fp6 digit, exact group sums on
the block-scaled matrix cores.  Held to the oracle within the output criterion of the path: every element within one
ULP or rtol 1e-3, or within the fp32 re-association bound (per-group zero-points reach the running sums in terms of their
own, K may be split across workgroups); with a uniform zero-point and K in one piece the outputs are the oracle's bits."""
import numpy as np
import pytest
import torch

from slimkernels_amd import _lib, workloads
import parity_utils as pu

FAKE = 0x10000


def test_every_int8_value_is_the_sum_of_its_two_digits():
    fp4 = np.array([0, 0.5, 1, 1.5, 2, 3, 4, 6])                     # e2m1
    fp6 = np.array([(m / 8 if e == 0 else (1 + m / 8) * 2.0 ** (e - 1)) for e in range(4) for m in range(8)])   # e2m3
    for q in range(-127, 128):
        a4 = np.sign(q) * fp4[np.argmin(np.abs(fp4 - abs(q) / 32))]
        assert abs(q - 32 * a4) <= 16
        assert abs(q - 32 * a4) / 8 in fp6, q


def test_validation_and_sizes():
    L = _lib.lib()
    # (x, ldx, x_dtype, w_r, s_r, zp_r, zp_const, M, N, K, group, out, ldo, out_dtype, act, act_bytes, ws, ws_bytes, stream)
    names = ["x", "ldx", "xdt", "w", "s", "zp", "zpc", "M", "N", "K", "g", "out", "ldo", "odt", "act", "actb", "ws", "wsb", "st"]
    ok = [FAKE, 4096, 0, FAKE, FAKE, None, 2, 64, 256, 4096, 128, FAKE, 256, 0, FAKE, 1 << 30, None, 0, None]

    def call(**kw):
        a = list(ok)
        for k, v in kw.items():
            a[names.index(k)] = v
        return L.slimk_w2a8_linear(*a)

    assert call(x=None) == 1 and call(act=None) == 1
    assert call(M=0) == 2 and call(g=100) == 2 and call(zpc=4) == 2 and call(ldx=4000) == 2 and call(ldo=100) == 2
    assert call(xdt=2) == 4 and call(odt=5) == 4
    assert call(ldx=4100) == 3 and call(x=FAKE + 2) == 3 and call(act=FAKE + 4) == 3 and call(out=FAKE + 1) == 3
    assert call(actb=1000) == 5
    assert L.slimk_w2a8_linear_workspace_bytes(64, 256, 4096, 128) > 0 and call() == 5      # few tiles: K is split
    assert call(K=32768 + 64, ldx=40000, g=64) == 7                                          # a row no longer fits a workgroup
    assert L.slimk_w2a8_linear_activation_bytes(64, 256, 32768 + 64, 64) == 0
    assert L.slimk_w2a8_linear_route(4096, 4096, 32768 + 64, 64, 0) == 0
    # digits: 2560 bytes per 32 rows x 64 elements, an odd step count rounded up; then sums and token scales
    assert L.slimk_w2a8_linear_activation_bytes(33, 256, 192, 64) == 2 * 4 * 2560 + 512 + 256
    assert L.slimk_w2a8_linear_route(1, 4096, 4096, 128, 0) == 0


def test_routes_only_name_what_the_kernels_take():
    import random
    L = _lib.lib()
    rng = random.Random(5)
    routed = 0
    for _ in range(3000):
        g = rng.choice([64, 128, 256])
        K = g * rng.randint(1, 40960 // g)
        M, N = int(2 ** rng.uniform(0, 13)), int(2 ** rng.uniform(0, 15))
        zp = rng.randint(0, 1)
        if L.slimk_w2a8_linear_route(M, N, K, g, zp):
            routed += 1
            assert M >= 96 and g <= 128 and K <= 32512
            assert L.slimk_w2a8_linear_activation_bytes(M, N, K, g) >= (M + 31) // 32 * ((K + 127) // 128) * 2 * 2560
            assert L.slimk_w2a8_linear_workspace_bytes(M, N, K, g) < 1 << 28
        if K % 128 == 0:      # the weight-only form's own choice of a split is one that a caller may ask for
            split = L.slimk_w2a16_gemm_auto_split_k(M, N, K, g)
            assert split == 1 or 1 < split <= 64 and split * 4 <= K // max(g, 128)
    assert routed > 100


@pytest.mark.gpu
def test_recorded_into_a_graph(gpu_ops):
    """Split calls of both tiled forms replay to the eager bits, with eager work between the replays."""
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    w = gpu_ops.W2A8Linear.from_float(torch.randn((320, 4096), generator=gen, device="cuda", dtype=torch.float16), 128, "asym").weight
    x = torch.randn((200, 4096), generator=gen, device="cuda", dtype=torch.float16)
    assert _lib.lib().slimk_w2a8_linear_workspace_bytes(200, 320, 4096, 128) > 0
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = [w2a8_linear_digits(x, w), gpu_ops.w2a16_gemm(x, w, split_k=4)]
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = [w2a8_linear_digits(x, w), gpu_ops.w2a16_gemm(x, w, split_k=4)]
    for _ in range(3):
        for y in got:
            y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for y, e in zip(got, want):
            assert torch.equal(y.view(torch.int16), e.view(torch.int16))
        w2a8_linear_digits(x[:100], w)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g,mode,out", [
    (1, 64, 64, 64, "sym", "float16"),             # one row, one step: half a stage
    (31, 100, 192, 64, "asym", "bfloat16"),        # an odd number of steps, a ragged N, per-group zero-points
    (33, 256, 128, 128, "ref", "float16"),         # one stage; uniform zero-point 1
    (64, 320, 1088, 64, "sym", "bfloat16"),        # two channel tiles, one of a single strip; an odd number of steps
    (65, 1001, 768, 256, "asym", "float16"),       # groups of two stages, three to a split-free launch; 2-byte stores
    (77, 256, 4096, 128, "sym", "float16"),        # K split across workgroups
    (130, 264, 3328, 256, "sym", "bfloat16"),      # split in whole groups of 256
    (257, 72, 2048, 64, "asym", "float16"),        # rows dealt to the XCDs (from 256 on), split
    (1025, 14592, 320, 64, "sym", "float16"),      # 128-row tiles (513 of them), the last one a single row
    (1000, 16640, 256, 128, "asym", "bfloat16"),   # 128-row tiles with per-group zero-points
])
def test_digits_against_the_oracle(gpu_ops, oracle, M, N, K, g, mode, out):
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    print(f"digits M={M} N={N} K={K} g={g} {mode} {out}", flush=True)
    case = pu.small_case(M, N, K, g, mode, seed=M + N, out_dtype=out, outliers=M % 2 == 1)
    packed, scales, zero = pu.quantized_weight(case)
    x = workloads.make_activation(case)
    bf16 = out == "bfloat16"
    big = M * N * (K // g) > 1 << 26               # (the oracle's group sums would be gigabytes: the strict criterion alone)
    ref = oracle.reference_forward(x, packed, scales, zero, g, out_bf16=bf16, want_acc=not big)
    w, xd = pu.device_inputs(gpu_ops, case, packed, scales, zero, x)
    y = w2a8_linear_digits(xd, w, pu.torch_dtype(case))
    bound = None
    if not big:
        # per-group zero-points: the sums centred on 2 and the rest (zp - 2) * rowsum are each larger than their difference
        zp = np.broadcast_to(np.asarray(zero, np.int64), (K // g, N))
        rs = ref["q"].reshape(M, K // g, g).astype(np.int64).sum(2)
        folded = np.abs(rs)[:, None, :] * np.abs(zp - (2 if mode == "asym" else zp)).T[None]
        bound = pu.reorder_bound(np.abs(ref["acc"].astype(np.int64)) + 2 * folded, scales, ref["s_a"])
    if big:
        # every element within one ULP or rtol 1e-3 but a few whose terms cancel, which the sums' magnitude bounds:
        # K / g * 2^-24 * s_a * sum_g scale * 127 * 3 * g, far below a dropped term
        bound = (K // g * 2.0 ** -24 * ref["s_a"].astype(np.float64)[:, None] * 3 * 127 * g *
                 np.asarray(scales, np.float64).sum(0)[None, :])
    pu.assert_out_close(pu.out_tensor_bits(y), ref["out_bits"], bf16, reorder_bound=bound, what="digits")
    if mode != "asym" and g < 256 and _lib.lib().slimk_w2a8_linear_workspace_bytes(M, N, K, g) == 0:
        np.testing.assert_array_equal(pu.out_tensor_bits(y), np.ascontiguousarray(ref["out_bits"]).view(np.uint16))
    # a strided activation and reused scratch give the same bits
    wide = torch.zeros((M, K + 64), dtype=xd.dtype, device="cuda")
    wide[:, :K] = xd
    y2 = w2a8_linear_digits(wide[:, :K], w, pu.torch_dtype(case))
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


def _activation(case, kind):
    """What a ReLU or a gating leaves (no value below zero), and values around 3: both have a mean far from zero."""
    x = workloads.make_activation(case)
    return {"relu": np.maximum(x, np.float16(0)), "shifted": (x.astype(np.float32) + 3 * np.abs(x).mean()).astype(np.float16)}[kind]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["relu", "shifted"])
@pytest.mark.parametrize("M,N,K,g,mode,out", [
    (40, 8256, 1024, 128, "sym", "float16"),       # 64-row tiles, four of them two row blocks short
    (513, 4160, 1088, 64, "ref", "bfloat16"),      # an odd number of steps; uniform zero-point 1
    (300, 16640, 512, 64, "sym", "bfloat16"),      # 325 64-row tiles
    (600, 16640, 512, 128, "sym", "float16"),      # 128-row tiles
])
def test_activations_with_a_mean_uniform_zero_points(gpu_ops, oracle, M, N, K, g, mode, out, kind):
    """The zero-point is in the group sums: without K splits every output is the oracle's, bit for bit."""
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    print(f"digits, bits of the oracle M={M} N={N} K={K} g={g} {mode} {out} {kind}", flush=True)
    assert _lib.lib().slimk_w2a8_linear_workspace_bytes(M, N, K, g) == 0
    case = pu.small_case(M, N, K, g, mode, seed=M + N, out_dtype=out)
    packed, scales, zero = pu.quantized_weight(case)
    x = _activation(case, kind)
    ref = oracle.reference_forward(x, packed, scales, zero, g, out_bf16=out == "bfloat16", want_acc=False)
    w, xd = pu.device_inputs(gpu_ops, case, packed, scales, zero, x)
    y = w2a8_linear_digits(xd, w, pu.torch_dtype(case))
    np.testing.assert_array_equal(pu.out_tensor_bits(y), np.ascontiguousarray(ref["out_bits"]).view(np.uint16))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["relu", "shifted"])
@pytest.mark.parametrize("M,N,K,g,mode", [
    (300, 4096, 4096, 128, "sym"),
    (300, 4096, 4096, 64, "asym"),
    (256, 2048, 8192, 128, "asym"),
    (1024, 8192, 2048, 128, "asym"),
    (1024, 8192, 2112, 64, "asym"),
])
def test_activations_with_a_mean_are_no_less_exact_than_on_the_int8_path(gpu_ops, oracle, M, N, K, g, mode, kind):
    """Against float64 from the same integers and scales: no more outputs than the int8 path has are other than the
    correctly rounded ones (0.1 % of the outputs apart, which is what the two paths' own splits of K may add), and every
    output is within its rounding and the rounding of the running sums.  These never hold more than the zero-point terms of
    two drains beside the groups so far, and a term of a group costs at most 2^-24 of what they hold."""
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    print(f"digits against float64 M={M} N={N} K={K} g={g} {mode} {kind}", flush=True)
    case = pu.small_case(M, N, K, g, mode, seed=M + N)
    packed, scales, zero = pu.quantized_weight(case)
    x = _activation(case, kind)
    w, xd = pu.device_inputs(gpu_ops, case, packed, scales, zero, x)
    qa = gpu_ops.quantize_act_int8(xd, g)
    # float64 products of a group are whole numbers below 2^53: exact
    G = K // g
    q = qa.q.double().reshape(M, G, g).transpose(0, 1).contiguous()
    sc = torch.from_numpy(np.asarray(scales, np.float16)).cuda().double()
    zp = torch.from_numpy(np.broadcast_to(np.asarray(zero), (G, N)).astype(np.float64)).cuda()
    codes = torch.from_numpy(oracle.np_unpack(packed)).cuda().double().reshape(N, G, g)
    want = torch.zeros((M, N), dtype=torch.float64, device="cuda")
    held = torch.zeros_like(want)                  # the sum over the groups of what the running sums hold, at most
    for i in range(G):
        term = (q[i] @ (codes[:, i] - zp[i][:, None]).t().contiguous()) * sc[i]
        want += term
        offset = (2 - zp[i]).abs() * sc[i] * q[i].sum(1, keepdim=True).abs()
        held += want.abs() + term.abs() + 2 * offset
    s_a = qa.s_a.double()[:, None]
    want, held = want * s_a, held * s_a
    best = want.half()
    digits = w2a8_linear_digits(xd, w)
    off = {"digits": (digits != best).sum().item(), "int8": (gpu_ops.w2a8_gemm(qa, w) != best).sum().item()}
    print(f"  not correctly rounded: {off} of {M * N}", flush=True)
    assert off["digits"] <= off["int8"] + M * N // 1000, off
    # half an ULP, the product with the token scale, and three roundings a drain (the fold and the two terms of a pair; a
    # split's sums are added once more, which the third covers)
    ulp = torch.from_numpy(pu.ulp_of(want.float().cpu().numpy(), False)).cuda()
    tol = 0.5 * ulp * (1 + 2.0 ** -12) + 2.0 ** -24 * (3 * held + want.abs())
    bad = (digits.double() - want).abs() > tol
    assert not bad.any(), int(bad.sum())


@pytest.mark.gpu
def test_split_call_keeps_nothing_and_takes_dirty_scratch(gpu_ops):
    """The partial sums of a split call are the call's own memory, whatever it held; nothing stays behind on the weight or in
    the allocator, and the arrival counters are left at zero."""
    from slimkernels_amd.torch.ops import _raw_stream, w2a8_linear_digits
    L = _lib.lib()
    M, N, K, g = 300, 4096, 4096, 128
    w = gpu_ops.W2A8Linear.from_float(torch.randn((N, K), device="cuda", dtype=torch.float16), g, "sym").weight
    x = torch.randn((M, K), device="cuda", dtype=torch.float16)
    act_bytes, ws_bytes = L.slimk_w2a8_linear_activation_bytes(M, N, K, g), L.slimk_w2a8_linear_workspace_bytes(M, N, K, g)
    assert act_bytes % 256 == 0 and ws_bytes > _lib.COUNTER_BLOCK_BYTES
    out = torch.empty((M, N), device="cuda", dtype=torch.float16)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    w2a8_linear_digits(x, w, out=out)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before and not w.workspaces
    act = torch.full((act_bytes,), 0xff, device="cuda", dtype=torch.uint8)
    ws = torch.full((ws_bytes,), 0xff, device="cuda", dtype=torch.uint8)
    for _ in range(2):
        dirty = torch.zeros_like(out)
        _lib.check(L.slimk_w2a8_linear(x.data_ptr(), K, _lib.F16, w.w_r.data_ptr(), w.s_r.data_ptr(), None, w.zp_const, M, N, K, g,
                                       dirty.data_ptr(), N, _lib.F16, act.data_ptr(), act_bytes, ws.data_ptr(), ws_bytes,
                                       _raw_stream(torch.cuda.current_device())))
        assert torch.equal(dirty, out)
    tiles = N // 256 * ((M + 127) // 128)          # (64-row tiles would be more)
    assert not ws[:4 * tiles].any()


def test_route_knows_short_reductions_and_per_group_zero_points():
    """512 and more 128-row tiles: with K < 512 symmetric layers stay on the int8 path (2317 x 8400 x 256 24.3 against 25.1
    us), layers with per-group zero-points do not (32.3 against 25.6).  Fewer tiles: the two paths' predictions know the
    zero-points too (600 x 11008 x 4096: 46.4 / 44.2 us symmetric, less than the 6 % in hand, 52.9 / 48.7 with zero-points)."""
    route = _lib.lib().slimk_w2a8_linear_route
    for M, N, g in ((2317, 8400, 128), (7173, 6000, 128), (2189, 22352, 64)):
        assert [route(M, N, 256, g, zp) for zp in (0, 1)] == [0, 1]
        assert [route(M, N, 512, g, zp) for zp in (0, 1)] == [1, 1]
    assert [route(600, 11008, 4096, 128, zp) for zp in (0, 1)] == [0, 1]
    assert [route(512, 28672, 8192, 64, zp) for zp in (0, 1)] == [1, 1]


@pytest.mark.parametrize("M,N,K,g,zp,taken", [
    (4936, 1024, 18240, 64, 0, 0),      # 220 us through the digits, 193 not
    (3574, 2296, 28160, 128, 0, 0),     # 329 / 307
    (134, 23552, 1856, 64, 0, 0),       # 28.2 / 25.5: an odd number of steps
    (207, 12544, 1984, 64, 0, 0),       # 23.7 / 21.6
    (4936, 1024, 18240, 64, 1, 1),      # per-group zero-points gain whatever the rows (1200..16384: 17 %)
    (4096, 2048, 8192, 128, 1, 1),
    (160, 20480, 2048, 128, 0, 1),      # 23 / 31
    (700, 3072, 24576, 64, 0, 1),       # 105 / 121
])
def test_route_beyond_what_the_predictions_were_fitted_on(M, N, K, g, zp, taken):
    assert _lib.lib().slimk_w2a8_linear_route(M, N, K, g, zp) == taken


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g,mode,out", [
    (96, 16384, 8192, 64, "asym", "bfloat16"),     # the fewest rows
    (129, 16384, 1088, 64, "sym", "float16"),      # a short reduction of an odd number of steps, one row in the last tile
    (255, 20481, 1024, 128, "asym", "float16"),    # the shortest; 2-byte stores
    (513, 2056, 9728, 64, "asym", "bfloat16"),     # few channels, a last strip of eight
])
def test_newly_routed_calls_give_the_int8_paths_results(gpu_ops, M, N, K, g, mode, out):
    """Calls of 96 rows and more below 4096 channels or elements, or up to 256 rows, that the layer takes through the digits:
    exact group sums on both paths, fp32 folds in another order, outputs rounded once (2^-11 / 2^-8 of a value at most)."""
    dtype = getattr(torch, out)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M)
    weight = torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16) * 0.02
    bias = torch.randn((N,), generator=gen, device="cuda").to(dtype)
    layer = gpu_ops.W2A8Linear.from_float(weight, g, mode, bias=bias, out_dtype=dtype)
    assert _lib.lib().slimk_w2a8_linear_route(M, N, K, g, int(mode == "asym"))
    x = (torch.randn((M, K), generator=gen, device="cuda") + 0.3).to(dtype)
    with torch.no_grad():
        y = layer(x).double()
    ref = (gpu_ops.w2a8_gemm(gpu_ops.quantize_act_int8(x, g), layer.weight, dtype) + bias).double()
    assert (y - ref).norm() <= (3e-4 if dtype == torch.float16 else 2.4e-3) * ref.norm()
