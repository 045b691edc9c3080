// Host-side entry points of the digit form of the W2A8 path (gemm_mx.hip): activation quantisation into digit
// fragments and the tiled GEMM on the block-scaled matrix cores.  As the other launchers: no validation, enqueue only.
#pragma once
#include "w2a8_common.h"

namespace w2a8 {

namespace mx {
constexpr int kFragRows = 32;        // token rows of a fragment
constexpr int kFragBytes = 2560;     // 32 rows x 64 elements: 1024 bytes of fp4 digits, 1536 of fp6 digits
constexpr int kStageSteps = 2;       // 64-element steps per pipeline stage
constexpr int kStripsPerWg = 4;      // a wave each
constexpr int kMaxK = 32512;         // the quantising kernel holds a row in 64 KiB of LDS (and 1024 threads' registers)
}  // namespace mx

struct MxParams {
    const uint8_t* frag;    // activation digits: [row block][steps rounded up to even][2560]
    const float* cs;        // [K / (64 or 128)][M] centring sums: -centre / 16 * the sum of q over the elements of a drain
    const float* s_a;       // [M]
    const uint32_t* w_r;    // repacked codes
    const uint16_t* s_r;    // [G][strips][16][4] fp16 bits
    const uint8_t* zp_r;    // [G][strips][16][4] or nullptr
    void* out;              // [M][ldo] fp16 / bf16 bits
    const uint16_t* bias;   // [N] in the output's type, added to the rounded outputs, or nullptr
    float* ws_partial;      // split-K partial tiles
    unsigned* ws_counter;   // arrival counters (the quantising kernel zeroes them)
    int ldo, M, N, K, G, steps, strips, zp_const;
    int group_shift;        // 1 with groups of 256 (two stages share a scale), else 0
    int split;              // K splits (grid.y)
    int stages_per_split;
};

inline int mx_row_blocks(int M) { return (M + mx::kFragRows - 1) / mx::kFragRows; }
__host__ __device__ inline int mx_padded_steps(int K) { return (K / kStepK + 1) / 2 * 2; }
// what a launch looks like: row blocks per workgroup tile (2 or 4), tiles, K splits and stages per split
struct MxPlan { int rb, tiles, split, stages_per_split; };
MxPlan mx_plan(int M, int N, int K, int group_size);
float mx_predicted_time(int M, int N, int K, int group_size, int per_group_zp, int rb, int split);

// centre: the zero-point the group sums start from (the layer's, or 2 where it has one per group); counters: n_counters
// words to be zeroed
hipError_t launch_mx_quant(const void* x, int ldx, bool x_bf16, int M, int K, int group_size, int centre, uint8_t* frag, float* cs,
                           float* s_a, unsigned* counters, int n_counters, hipStream_t stream);
hipError_t launch_mx_gemm(const MxParams& p, int rb, int gs, bool out_bf16, hipStream_t stream);

}  // namespace w2a8
