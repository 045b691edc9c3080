"""The native host side of the calls (slimkernels_amd/torch/_native.cpp) against the general Python code of the same calls: the
same bits wherever it takes a call, and None, which hands the call to that code, wherever it does not."""
import math
import random
import types

import pytest
import torch

from slimkernels_amd import _lib
from slimkernels_amd.torch import ops, w4


def _without_native(monkeypatch, fn):
    """fn() through the general code."""
    real = ops._host()
    names = ("linear", "linear16", "linear4", "quantize", "gemm", "grouped")
    with monkeypatch.context() as m:
        m.setattr(ops, "_fast", types.SimpleNamespace(**{n: lambda *a: None for n in names}))
        y = fn()
    assert ops._fast is real
    return y


def test_cpu_tensors_and_other_objects_are_left_to_the_general_code():
    host = ops._host()
    x = torch.zeros((2, 128), dtype=torch.float16)
    w = ops.W2A8Weight(x, x, None, 2, 64, 128, 128)
    assert host.linear(x, w, torch.float16, None) is None and host.linear16(x, w, torch.float16, None) is None
    assert host.linear(None, w, torch.float16, None) is None and host.linear(x, w, "float16", None) is None and host.linear(x, w) is None
    assert host.linear4(x, object(), torch.float16, None) is None and host.gemm(object(), w, torch.float16) is None
    assert host.quantize(x, 128, 1, True) is None and host.quantize(3, 128, 1, True) is None
    assert host.grouped([], torch.float16) is None and host.grouped([(x, w)], torch.float16) is None
    assert host.grouped(iter([]), torch.float16) is None
    with pytest.raises(ValueError, match="must live on the GPU"):
        ops.quantize_act_int8(x, 128)
    with pytest.raises(TypeError):
        host.bind({}, None)
    with pytest.raises(KeyError):
        host.bind({}, print)


def test_the_same_rules_as_the_general_code():
    """Which kernels a shape goes to, asked of the native host side and of the predicates of ops.py and w4.py: the layers' bits alone
    would not show the two running different kernels."""
    rules, rng = ops._host().rules, random.Random(3)
    seen = set()
    for _ in range(4000):
        g = rng.choice([64, 128, 256])
        M = int(math.exp(rng.uniform(0, math.log(6000))))
        N, K = int(math.exp(rng.uniform(math.log(16), math.log(30000)))), g * rng.randint(1, 28672 // g)
        zp = rng.randint(0, 2)
        w = ops.W2A8Weight(None, None, object() if zp == 2 else None, 2 if zp != 1 else 1, N, K, g)
        digits, sums, ws, act, one_pass = rules(M, N, K, g, zp)
        assert digits == (M > 1 and ops.linear_digits_applies(M, w)) and sums == ops.needs_rowsum(M, w), (M, N, K, g, zp)
        assert one_pass == w4.one_pass_applies(M, w4.W4A8Weight(w, N, K, g)), (M, K, g)
        name, args = ("slimk_w2a8_gemm_fused_workspace_bytes", (0,)) if M == 1 and ops.fused_applies(1, K) else \
            ("slimk_w2a8_linear_workspace_bytes", ()) if digits else ("slimk_w2a8_gemm_workspace_bytes", (_lib.KERNEL_AUTO, 0))
        assert ws == ops._query(name, M, N, K, g, *args)
        assert act == (ops._query("slimk_w2a8_linear_activation_bytes", M, N, K, g) if digits else 0)
        seen.add((digits, sums, one_pass, ws > 0))
    assert len(seen) >= 8
    assert rules(1, 2, 3) is None and rules(1.0, 64, 64, 64, 0) is None


LAYERS = {"2": ops.W2A8Linear, "16": ops.W2A16Linear, "4": w4.W4A8Linear}


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["2", "4", "16"])
@pytest.mark.parametrize("lead,N,K,g,mode,out,bias", [
    ((1,), 4096, 4096, 128, "sym", "float16", True),          # one launch (2-bit)
    ((1, 1), 320, 14336, 128, "asym", "bfloat16", False),     # K split: the workspace is made by the first call
    ((), 320, 512, 64, "sym", "float16", False),              # a vector
    ((5,), 1000, 1024, 64, "asym", "bfloat16", True),
    ((2, 20), 1001, 8192, 128, "sym", "float16", True),       # 40 rows, K split
    ((300,), 4096, 8192, 128, "asym", "float16", False),      # the digit form (2-bit)
    ((7, 100), 520, 2048, 64, "sym", "bfloat16", True),
])
def test_layers(gpu_ops, monkeypatch, kind, lead, N, K, g, mode, out, bias):
    dtype = getattr(torch, out)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    weight = torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16) * 0.02
    b = torch.randn((N,), generator=gen, device="cuda").to(dtype) if bias else None
    layer = LAYERS[kind].from_float(weight, g, mode, bias=b, out_dtype=dtype)
    x = torch.randn((*lead, K), generator=gen, device="cuda").to(dtype)
    want = _without_native(monkeypatch, lambda: layer(x))
    call = {"2": ops._host().linear, "4": ops._host().linear4, "16": ops._host().linear16}[kind]
    rows = x.numel() // K
    y = call(x, layer.weight, dtype, b)
    if kind == "4" and rows == 1:
        assert y is None                                       # (the row is laid down twice by the general code)
    else:
        assert y.shape == (*lead, N) and y.dtype == dtype and y.is_contiguous()
        assert torch.equal(y, want)
    assert torch.equal(layer(x), want)
    # layouts: rows of a wider tensor are read in place; what is not laid out for the kernels goes the general way
    x2 = x.reshape(-1, K)
    wide = torch.zeros((rows, K + 72), dtype=dtype, device="cuda")
    wide[:, :K] = x2
    odd = torch.zeros((rows, K + 1), dtype=dtype, device="cuda")
    odd[:, 1:] = x2
    for t, taken in ((wide[:, :K], not (kind == "4" and rows == 1)), (odd[:, 1:], False), (x2.t().contiguous().t(), rows == 1 and kind != "4")):
        if rows == 1 and t.stride(0) % 8:
            assert call(t, layer.weight, dtype, b) is None        # (one row at an odd pitch: refused by both)
            continue
        assert (call(t, layer.weight, dtype, b) is not None) == taken
        assert torch.equal(layer(t), want.reshape(-1, N))
    assert call(x.float(), layer.weight, dtype, b) is None and call(x, layer.weight, torch.float32, b) is None
    assert call(x[..., :K - 128], layer.weight, dtype, b) is None
    with pytest.raises(ValueError):
        layer(x[..., :K - 128])
    sub = x.as_subclass(type("Sub", (torch.Tensor,), {}))
    assert call(sub, layer.weight, dtype, b) is None


# every kernel that a layer call can end in, with and without whole 16-byte output rows (the W4 layer's K is the planes' half)
BIASED = [("2", 1, 4096, 4096, 128, "sym"), ("2", 1, 1001, 16384, 64, "asym"), ("2", 3, 33000, 512, 64, "sym"), ("2", 14, 24640, 1024, 128, "asym"),
          ("2", 16, 520, 14336, 256, "sym"), ("2", 24, 12288, 8192, 128, "sym"), ("2", 40, 28672, 4608, 64, "sym"), ("2", 80, 11009, 14336, 128, "asym"),
          ("2", 60, 11008, 4096, 128, "asym"), ("2", 200, 1000, 4096, 128, "sym"), ("2", 600, 4100, 1024, 256, "asym"), ("2", 1025, 14600, 256, 128, "sym"),
          ("2", 300, 4096, 8192, 128, "asym"), ("2", 520, 16640, 4096, 64, "sym"), ("2", 1025, 14601, 512, 128, "asym"),
          ("16", 1, 14336, 4096, 128, "sym"), ("16", 6, 1001, 9216, 64, "asym"), ("16", 300, 4096, 8192, 128, "sym"), ("16", 700, 11009, 2048, 128, "asym"),
          ("16", 1024, 14336, 1024, 128, "sym"), ("4", 1, 520, 2048, 128, "asym"), ("4", 20, 1001, 4096, 128, "sym"), ("4", 100, 1000, 4096, 64, "asym"),
          ("4", 1000, 14408, 256, 128, "sym")]


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["float16", "bfloat16"])
@pytest.mark.parametrize("kind,M,N,K,g,mode", BIASED)
def test_bias_in_the_kernels(gpu_ops, kind, M, N, K, g, mode, out):
    """Bit for bit the sum of two tensors, for values that round, vanish beside each other, overflow or are no numbers."""
    print(f"bias {kind} M={M} N={N} K={K} g={g} {mode} {out}", flush=True)
    dtype = getattr(torch, out)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    weight = torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16) * 0.02
    layer = LAYERS[kind].from_float(weight, g, mode, out_dtype=dtype)
    x = torch.randn((M, K), generator=gen, device="cuda").to(dtype)
    plain = layer(x)
    b = (torch.randn((N,), generator=gen, device="cuda") * 2.0 ** torch.randint(-12, 8, (N,), generator=gen, device="cuda")).to(dtype)
    b[:8] = torch.tensor([0.0, -0.0, float("inf"), float("-inf"), float("nan"), torch.finfo(dtype).max, torch.finfo(dtype).min, 1.0], dtype=dtype)
    b[8:16] = -plain[0, 8:16]
    want = plain + b
    layer.bias = b
    got = layer(x)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got.nan_to_num(0.0).view(torch.int16), want.nan_to_num(0.0).view(torch.int16))


@pytest.mark.gpu
def test_biases_that_the_kernels_do_not_add(gpu_ops):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    layer = gpu_ops.W2A8Linear.from_float(torch.randn((320, 512), generator=gen, device="cuda", dtype=torch.float16), 64, "sym")
    x = torch.randn((4, 512), generator=gen, device="cuda", dtype=torch.float16)
    plain = layer(x)
    b = torch.randn((400,), generator=gen, device="cuda", dtype=torch.float16)
    for bias in (b[1:321], b[:320].float(), torch.randn((640,), generator=gen, device="cuda", dtype=torch.float16)[::2], b[:1], b[0],
                 b[:320].bfloat16(), b[:320].expand(4, 320), torch.randn((4, 1), device="cuda", dtype=torch.float16)):
        layer.bias = bias
        got, want = layer(x), plain + bias
        assert got.dtype == want.dtype and torch.equal(got, want)
    # a derivative is asked of it
    p = torch.nn.Parameter(b[:320].clone())
    layer.bias = p
    y = layer(x)
    assert y.requires_grad and torch.equal(y, plain + p)
    y.sum().backward()
    assert torch.equal(p.grad, torch.full_like(p, 4.0))
    with torch.no_grad():
        assert not layer(x).requires_grad and torch.equal(layer(x), plain + p)
    import torch.autograd.forward_ad as fwd
    with fwd.dual_level(), torch.no_grad():
        layer.bias = None
        del layer.bias
        layer.bias = fwd.make_dual(b[:320].clone(), torch.ones_like(b[:320]))
        assert torch.equal(fwd.unpack_dual(layer(x)).tangent, torch.ones_like(plain))
    layer.bias = b[:300]
    with pytest.raises(RuntimeError):
        layer(x)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["2", "4", "16"])
def test_a_wider_bias_on_a_layer_of_one_channel(gpu_ops, monkeypatch, kind):
    """Token rows [M, 1] widen with the bias; of more (or fewer) dimensions the general code refuses it, and so does the layer."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    layer = LAYERS[kind].from_float(torch.randn((1, 256), generator=gen, device="cuda", dtype=torch.float16), 128, "sym")
    x = torch.randn((2, 3, 256), generator=gen, device="cuda", dtype=torch.float16)
    plain = layer(x)
    layer.bias = torch.randn((5,), generator=gen, device="cuda", dtype=torch.float16)
    assert torch.equal(layer(x[0]), plain[0] + layer.bias)
    for t in (x, x[0, 0]):
        with pytest.raises(RuntimeError):
            _without_native(monkeypatch, lambda: layer(t))
        with pytest.raises(RuntimeError):
            layer(t)
    layer.bias = layer.bias[:1]
    assert torch.equal(layer(x), plain + layer.bias)


@pytest.mark.gpu
def test_quantise_gemm_and_grouped(gpu_ops, monkeypatch):
    host = ops._host()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    for M, K, g, copies, sums in ((1, 4096, 128, 1, True), (7, 1088, 64, 2, True), (70, 512, 256, 1, False)):
        x = torch.randn((M, K), generator=gen, device="cuda", dtype=torch.float16)
        got, want = ops.quantize_act_int8(x, g, copies, sums), _without_native(monkeypatch, lambda: ops.quantize_act_int8(x, g, copies, sums))
        assert host.quantize(x, g, copies, sums) is not None
        assert torch.equal(got.q, want.q) and torch.equal(got.s_a, want.s_a) and got.group_size == want.group_size
        assert (got.rowsum is None) == (not sums) and got.q.shape == want.q.shape
        if sums:
            assert got.rowsum.shape == want.rowsum.shape and torch.equal(got.rowsum[:, :M], want.rowsum[:, :M])
    with pytest.raises(Exception, match="group_size"):
        ops.quantize_act_int8(x, 100)
    problems = []
    for M, N, K in ((1, 320, 4096), (17, 1000, 1024), (32, 64, 14336)):
        w = gpu_ops.W2A8Linear.from_float(torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16), 128, "sym").weight
        problems.append((ops.quantize_act_int8(torch.randn((M, K), generator=gen, device="cuda", dtype=torch.float16), 128), w))
    want = _without_native(monkeypatch, lambda: ops.w2a8_gemm_grouped(problems, torch.bfloat16))
    into = torch.empty_like(want[1])
    got = host.grouped([problems[0], (*problems[1], into), (*problems[2], None)], torch.bfloat16)
    assert got[1] is into and all(torch.equal(a, b) for a, b in zip(got, want))
    assert host.grouped([problems[0], (*problems[1], into)], torch.float16) is None          # an output of another type
    with pytest.raises(ValueError, match="out_dtype"):
        ops.w2a8_gemm_grouped([problems[0], (*problems[1], into)], torch.float16)
    for qa, w in problems + [(ops.quantize_act_int8(torch.randn((60, 1024), generator=gen, device="cuda", dtype=torch.float16), 128), problems[1][1])]:
        want = _without_native(monkeypatch, lambda: ops.w2a8_gemm(qa, w))
        assert torch.equal(host.gemm(qa, w, torch.float16), want)
    assert host.gemm(qa, problems[0][1], torch.float16) is None
    with pytest.raises(ValueError, match="does not match"):
        ops.w2a8_gemm(qa, problems[0][1])
    long = problems * 9                                        # more than one launch
    assert host.grouped(long, torch.float16) is None and len(ops.w2a8_gemm_grouped(long)) == 27


@pytest.mark.gpu
def test_each_stream_has_its_own_workspace_and_graphs_replay(gpu_ops):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    weight = torch.randn((320, 14336), generator=gen, device="cuda", dtype=torch.float16)
    layer = gpu_ops.W2A8Linear.from_float(weight, 128, "sym")
    layer16 = gpu_ops.W2A16Linear.from_float(weight, 128, "sym")
    xs = [torch.randn((m, 14336), generator=gen, device="cuda", dtype=torch.float16) for m in (1, 6, 70, 300)]
    want = [(layer(x), layer16(x)) for x in xs]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        side = [(layer(x), layer16(x)) for x in xs]
    stream.synchronize()
    assert len(layer.weight.workspaces) == 2
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        recorded = [(layer(x), layer16(x)) for x in xs]
    for _ in range(3):
        for pair in recorded:
            for y in pair:
                y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for pair, other, eager in zip(recorded, side, want):
            assert all(torch.equal(a, e) and torch.equal(b, e) for a, b, e in zip(pair, other, eager))
        layer(xs[1])
