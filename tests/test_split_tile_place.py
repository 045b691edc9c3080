"""Which tile and K split a workgroup of the split tiled kernels takes (split_tile_place in w2a8_common.h), checked on the
host: every (split, tile) pair gets one workgroup of the grid, and no CU gets more workgroups than with the pairs dealt out
evenly to the eight XCDs of 32 CUs."""
import os
import shutil
import subprocess

import pytest
import torch

from test_w2a16_plan import plan as w2a16_plan

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "slimkernels_amd", "csrc")

PROGRAM = r"""
#include "w2a8_common.h"
#include <cstdio>
#include <vector>
int main() {
    for (int tiles_n = 1; tiles_n <= 60; ++tiles_n)
        for (int tiles_m = 1; tiles_m <= 17; ++tiles_m)
            for (int splits = 1; splits <= 13; ++splits) {
                const int total = tiles_n * tiles_m, grid_x = (total + 7) / 8 * 8, grid = grid_x * splits;
                std::vector<int> seen(total * splits, 0), per_xcd(8, 0);
                int placed = 0;
                for (int wg = 0; wg < grid; ++wg) {
                    int tile = -1, split = -1;
                    if (!w2a8::split_tile_place(wg % grid_x, wg / grid_x, splits, tiles_n, tiles_m, tile, split)) continue;
                    if (tile < 0 || tile >= total || split < 0 || split >= splits || seen[split * total + tile]++) {
                        std::printf("%d x %d tiles, %d splits: wg %d -> %d %d\n", tiles_n, tiles_m, splits, wg, tile, split);
                        return 1;
                    }
                    ++placed;
                    ++per_xcd[wg & 7];
                }
                int hi = 0;
                for (int x : per_xcd) hi = x > hi ? x : hi;
                if (placed != total * splits || (hi + 31) / 32 > ((total * splits + 7) / 8 + 31) / 32) {
                    std::printf("%d x %d tiles, %d splits: placed %d, at most %d per XCD\n", tiles_n, tiles_m, splits, placed, hi);
                    return 1;
                }
            }
    std::printf("ok\n");
    return 0;
}
"""


needs_hipcc = pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"),
                                 reason="needs hipcc to compile the header for the host")


def _run(tmp_path, program):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    src = tmp_path / "place.hip"
    src.write_text(program)
    exe = tmp_path / "place"
    subprocess.run([hipcc, "--cuda-host-only", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True,
                   capture_output=True, timeout=300)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr


@needs_hipcc
def test_every_pair_placed_once_and_cus_level(tmp_path):
    _run(tmp_path, PROGRAM)


# a short last split: it may not count, and where it does not decide the grid is dealt out split by split
SHORT = r"""
#include "w2a8_common.h"
#include <cstdio>
#include <vector>
int main() {
    for (int splits = 2; splits <= 13; ++splits)
        for (int per = 2; per <= 40; per += 2)
            for (int last = 1; last <= per; ++last) {
                const int stages = per * (splits - 1) + last;
                if (w2a8::counted_splits(splits, stages, per) != (2 * last <= per ? splits - 1 : splits)) return 1;
            }
    for (int tiles_n = 1; tiles_n <= 60; ++tiles_n)
        for (int tiles_m = 1; tiles_m <= 17; ++tiles_m)
            for (int splits = 2; splits <= 13; ++splits) {
                const int total = tiles_n * tiles_m, grid_x = (total + 7) / 8 * 8;
                const bool even = w2a8::deal_evenly(total, splits, splits - 1);
                if (even != (w2a8::splits_uneven(total, splits) && (total * splits <= 256 || w2a8::splits_uneven(total, splits - 1)))) return 5;
                std::vector<int> seen(total * splits, 0);
                int placed = 0;
                for (int wg = 0; wg < grid_x * splits; ++wg) {
                    int tile = -1, split = -1;
                    if (!w2a8::split_tile_place(wg % grid_x, wg / grid_x, splits, tiles_n, tiles_m, tile, split, splits - 1)) continue;
                    if (tile < 0 || tile >= total || split < 0 || split >= splits || seen[split * total + tile]++) return 2;
                    if (!even && split != wg / grid_x) return 3;
                    ++placed;
                }
                if (placed != total * splits) return 4;
            }
    std::printf("ok\n");
    return 0;
}
"""


@needs_hipcc
def test_short_last_splits(tmp_path):
    _run(tmp_path, SHORT)


# the weight-only form deals out (split, channel tile) sets, their token tiles the members
SETS = r"""
#include "w2a8_common.h"
#include <cstdio>
#include <vector>
int main() {
    for (int tiles_n = 1; tiles_n <= 60; ++tiles_n)
        for (int tiles_m = 1; tiles_m <= 17; ++tiles_m)
            for (int splits = 2; splits <= 13; ++splits) {
                const int total = tiles_n * tiles_m, grid = w2a8::xcd_grid(tiles_n, tiles_m) * splits;
                std::vector<int> seen(total * splits, 0), per_xcd(8, 0);
                int placed = 0, hi = 0;
                for (int wg = 0; wg < grid; ++wg) {
                    int set = -1, m = -1;
                    if (!w2a8::xcd_place(wg, tiles_n * splits, tiles_m, set, m)) continue;
                    if (set < 0 || set >= tiles_n * splits || m < 0 || m >= tiles_m || seen[set * tiles_m + m]++) return 1;
                    ++placed;
                    ++per_xcd[wg & 7];
                }
                for (int x : per_xcd) hi = x > hi ? x : hi;
                if (placed != total * splits || (hi + 31) / 32 > ((total * splits + 7) / 8 + 31) / 32) return 2;
            }
    std::printf("ok\n");
    return 0;
}
"""


@needs_hipcc
def test_every_set_placed_once(tmp_path):
    _run(tmp_path, SETS)


def _uneven(total, splits):
    """splits_uneven"""
    return -(-(-(-total // 8) * splits) // 32) > -(-(-(-total * splits // 8)) // 32)


def _tiles(M, N, rows=64):
    return -(-N // 256) * -(-M // rows)


def _splits(stages, asked):
    per = -(-stages // asked)
    return -(-stages // per)


def _close(y, ref):
    """Split sums against others: fp32 in another order, both rounded to fp16, 2^-11 of a value at most, 3e-4 in the norm."""
    assert torch.isfinite(y).all() and (y.double() - ref.double()).norm() <= 3e-4 * ref.double().norm()


EVEN = [
    (430, 1500, 4608, 128, "sym", 6),     # 6 x 7 tiles
    (430, 1500, 4608, 64, "asym", 6),
    (190, 3500, 4608, 128, "asym", 6),    # 14 x 3: the token tiles of a channel tile together
    (190, 3500, 4608, 64, "sym", 6),
    (385, 1537, 4480, 128, "asym", 5),    # 7 x 7, one row and one channel in the last of each; 2-byte stores
    (257, 4160, 7680, 256, "asym", 6),    # a group of 256: splits of equal length
]


@pytest.mark.gpu
@pytest.mark.parametrize("bits,M,N,K,g,mode,split", [(bits, *case) for case in EVEN for bits in (2, 4) if (bits, case[3]) != (4, 256)])
def test_int8_pairs_dealt_out_evenly(gpu_ops, bits, M, N, K, g, mode, split):
    """The int8 tiled kernels of 2-bit and of 4-bit weights where (split, tile) pairs are dealt out evenly: a tile's splits meet from
    different XCDs.  Against the unsplit call, and bit for bit on a second run (the splits are added in their order)."""
    from slimkernels_amd.torch import w4 as tw4
    stages = K // (256 if g == 256 else 128)
    assert _uneven(_tiles(M, N), _splits(stages, split))
    print(f"even dealing W{bits} M={M} N={N} K={K} g={g} {mode} split={split}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N + bits)
    weight = torch.randn((N, K // g, g), generator=gen, device="cuda")
    if mode == "asym":                    # (shifted groups: every zero-point occurs)
        weight += torch.randn((N, K // g, 1), generator=gen, device="cuda") * 1.5
    layer = (tw4.W4A8Linear if bits == 4 else gpu_ops.W2A8Linear).from_float((weight * 0.02).half().reshape(N, K).contiguous(), g, mode)
    x = torch.randn((M, K), generator=gen, device="cuda").half()
    qa = gpu_ops.quantize_act_int8(x, g)

    def run(n):
        if bits == 4:
            return tw4.w4a8_gemm_one_pass(qa, layer.weight, torch.float16, split_k=n)
        return gpu_ops.w2a8_gemm(qa, layer.weight, torch.float16, kernel="tiled", split_k=n)
    y = run(split)
    _close(y, run(1))
    assert torch.equal(run(split), y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g,mode,split,form", [
    (617, 2322, 4096, 128, "sym", 5, (128, 5, 1)),     # 10 x 5 tiles of 128 rows
    (231, 5127, 4608, 128, "asym", 6, (128, 6, 1)),    # 21 x 2; scalar partial sums
    (275, 4997, 4096, 64, "asym", 5, (64, 5, 1)),      # 20 x 5 of 64 rows
    (417, 1680, 6144, 128, "sym", 5, (64, 5, 2)),      # 7 x 7, two K halves in a workgroup
    (113, 5248, 6144, 256, "asym", 6, (64, 6, 2)),     # 21 x 2
])
def test_weight_only_sets_dealt_out_evenly(gpu_ops, M, N, K, g, mode, split, form):
    assert w2a16_plan(M, N, K, g, split) == form and _uneven(_tiles(M, N, form[0]), form[1])
    print(f"even dealing W2A16 M={M} N={N} K={K} g={g} {mode} split={split}", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N)
    w = gpu_ops.W2A8Linear.from_float(torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16) * 0.02, g, mode).weight
    x = torch.randn((M, K), generator=gen, device="cuda").half()
    y = gpu_ops.w2a16_gemm(x, w, split_k=split)
    _close(y, gpu_ops.w2a16_gemm(x, w, split_k=1))
    assert torch.equal(gpu_ops.w2a16_gemm(x, w, split_k=split), y)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,g,mode", [
    (657, 3424, 23040, 128, "sym"),     # digit form: 14 x 6 tiles, an odd one per XCD and split
    (652, 1000, 4160, 64, "asym"),      # more than four token tiles, odd steps
    (130, 1100, 6144, 128, "sym"),      # three token tiles of one channel tile on a queue
    (64, 1500, 9216, 128, "asym"),      # one token tile
    (257, 4160, 7936, 256, "asym"),     # 17 x 5 tiles in six splits, the last a sixth as long as the others
    (422, 1344, 6656, 256, "asym"),     # ... dealt out evenly all the same, one workgroup a CU
    (340, 3352, 8192, 256, "sym"),      # the digit form with such a last split
])
def test_split_calls(gpu_ops, M, N, K, g, mode):
    """The split tiled kernels (int8, digits, weight-only) on grids whose tiles are no multiple of eight, against the unsplit
    calls: the sums differ in their fp32 order and both are rounded to fp16, 2^-11 of a value at most, 3e-4 in the norm."""
    from slimkernels_amd.torch.ops import w2a8_linear_digits
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + N)
    w = gpu_ops.W2A8Linear.from_float(torch.randn((N, K), generator=gen, device="cuda", dtype=torch.float16) * 0.02, g, mode).weight
    x = torch.randn((M, K), generator=gen, device="cuda").half()
    qa = gpu_ops.quantize_act_int8(x, g)

    def close(y, ref):
        assert (y.double() - ref.double()).norm() <= 3e-4 * ref.double().norm()
    plain = gpu_ops.w2a8_gemm(qa, w, torch.float16, kernel="tiled", split_k=1)
    for split in (3, 6):
        close(gpu_ops.w2a8_gemm(qa, w, torch.float16, kernel="tiled", split_k=split), plain)
    close(w2a8_linear_digits(x, w), plain)
    if K % 128 == 0:
        plain = gpu_ops.w2a16_gemm(x, w, split_k=1)
        for split in (3, 6):
            close(gpu_ops.w2a16_gemm(x, w, split_k=split), plain)
