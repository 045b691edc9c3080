"""The one-pass W4 kernel's 128-row tiles (csrc/gemm_tiled.hip: tiled_w4_tall): bit for bit what its 64-row tiles give, which
tests/test_w4a8.py holds to the oracle, at the edges of tiles and stages."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,N,K,g,mode", [
    (1000, 14408, 128, 64, "sym"),       # one stage; a last channel tile of one strip and a bit
    (897, 14336, 256, 128, "asym"),      # a last row tile of one row
    (1024, 14401, 384, 64, "asym"),      # three stages; 2-byte stores
    (960, 16384, 1152, 128, "sym"),      # nine stages; half a row tile
    (1536, 16384, 640, 128, "asym"),     # three rounds of workgroups
])
def test_same_bits_as_the_64_row_tiles(gpu_ops, M, N, K, g, mode, out):
    from slimkernels_amd.torch import w4 as tw4
    print(f"W4 tall tiles M={M} N={N} K={K} g={g} {mode} {out}", flush=True)
    dtype = getattr(torch, out)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + K)
    weight = torch.randn((N, K // g, g), generator=gen, device="cuda")
    if mode == "asym":                    # (shifted groups: every zero-point occurs)
        weight += torch.randn((N, K // g, 1), generator=gen, device="cuda") * 1.5
    w = tw4.W4A8Linear.from_float((weight * 0.02).half().reshape(N, K).contiguous(), g, mode).weight
    x = torch.randn((M, K), generator=gen, device="cuda").relu().half()
    tiles = [-(-N // 256) * -(-M // rows) for rows in (64, 128)]
    n64, n128 = (-(-t // 256) for t in tiles)
    assert n128 >= 2 and 41 * n128 < 24 * n64
    y = tw4.w4a8_gemm_one_pass(gpu_ops.quantize_act_int8(x, g), w, dtype, split_k=1)
    for lo in range(0, M, 192):           # too few tiles for 128 rows
        part = tw4.w4a8_gemm_one_pass(gpu_ops.quantize_act_int8(x[lo:lo + 192], g), w, dtype, split_k=1)
        assert torch.equal(part.view(torch.int16), y[lo:lo + 192].view(torch.int16)), lo
