"""Which tile and K split a workgroup of the split tiled kernels takes (split_tile_place in w2a8_common.h), checked on the
host: every (split, tile) pair gets one workgroup of the grid, and no CU gets more workgroups than with the pairs dealt out
evenly to the eight XCDs of 32 CUs."""
import os
import shutil
import subprocess

import pytest
import torch

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
