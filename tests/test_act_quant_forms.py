"""Every form of the activation quantisers at the edges of its range: bit for bit the oracle's values (int8 rows), and digit
fragments that multiply out to what the int8 rows do."""
import numpy as np
import pytest
import torch

import parity_utils as pu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sums", [True, False])
@pytest.mark.parametrize("M,K,g,bf16", [
    (512, 2048, 64, False), (65, 2112, 64, True), (512, 4096, 128, False), (513, 4096, 128, True),     # 512 threads up to 512 rows
    (512, 4160, 64, False), (513, 4160, 64, False), (65, 8192, 256, True), (257, 8256, 64, False),     # 1024
    (130, 16384, 128, False), (513, 16384, 128, True), (513, 16448, 64, False), (70, 32768, 128, True),
    (600, 32768, 256, False), (66, 32832, 64, False),                                                  # ... and two passes
])
def test_int8_rows(gpu_ops, oracle, M, K, g, bf16, sums):
    print(f"act_quant M={M} K={K} g={g} bf16={bf16} sums={sums}", flush=True)
    gen = torch.Generator().manual_seed(M + K)
    x = torch.randn((M, K), generator=gen) * 3
    x[:, :: max(1, K // 7)] *= 30
    x[M // 2] = 0
    x = x.to(torch.bfloat16 if bf16 else torch.float16)
    bits = x.view(torch.int16).numpy().view(np.uint16)
    q, s_a, rs = oracle.c_act_quant(bits, g, is_bf16=True) if bf16 else oracle.c_act_quant(x.numpy(), g)
    qa = gpu_ops.quantize_act_int8(x.cuda(), g, rowsum=sums)
    np.testing.assert_array_equal(qa.q.cpu().numpy(), q)
    np.testing.assert_array_equal(qa.s_a.cpu().numpy(), s_a)
    if sums:
        want = torch.from_numpy(q).reshape(M, K // g, g).int().sum(2).t()
        assert torch.equal(qa.rowsum[:, :M].cpu(), want.to(torch.int32))


@pytest.mark.parametrize("out", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K,g,mode", [
    (256, 200, 11264, 128, "sym"),      # one row a workgroup
    (257, 200, 11264, 128, "asym"),     # two, the last workgroup with one
    (301, 128, 11328, 64, "sym"),       # one: two rows no longer fit beside another workgroup
    (259, 72, 64, 64, "asym"),          # two chunks
    (300, 72, 4160, 64, "sym"),         # an odd number of steps
    (260, 64, 32512, 128, "asym"),      # the longest row
])
def test_digit_fragments(gpu_ops, M, N, K, g, mode, out):
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    print(f"digit quantisation M={M} N={N} K={K} g={g} {mode} {out}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    dtype = getattr(torch, out)
    w = gpu_ops.W2A8Linear.from_float(torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16), g, mode).weight
    x = (torch.randn((M, K), generator=gen, device="cuda").abs() * 3).to(dtype)
    got, want = w2a8_linear_digits(x, w, dtype), gpu_ops.w2a8_gemm(gpu_ops.quantize_act_int8(x, g), w, dtype)
    # the same integers and scales: apart by a rounding of the outputs at most, wherever their fp32 sums were put together otherwise
    ulp = torch.from_numpy(pu.ulp_of(want.float().cpu().numpy(), out == "bfloat16")).cuda()
    held = x.float().abs().sum(1, keepdim=True) * w.s_r.float().max() * 3          # no running sum is larger
    assert bool(((got.float() - want.float()).abs() <= 1.01 * ulp + held * 2.0 ** -24 * (K // g)).all())
