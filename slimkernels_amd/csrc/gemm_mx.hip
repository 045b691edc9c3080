// The digit form of the W2A8 GEMM for gfx950: int8 activations times 2-bit weights on the block-scaled matrix cores
// (v_mfma_f32_32x32x64_f8f6f4) for many token rows, exact.
//
// Why not the int8 matrix cores (tiled_bodies.h): there every accumulator costs a conversion and an fma per scale
// group, and that and the unpacking hold the matrix cores to 0.53 of their rate in the main loop.  The fp4 / fp6 forms of
// the f8f6f4 instruction run at twice the int8 rate, so an activation may cost two of them: q in -127..127 is split
// exactly into two digits,
//     q = 32 * a4 + 8 * a6,   a4 = fp4 (e2m1) nearest to q / 32,   a6 = fp6 (e2m3) of the rest, |rest| <= 16,
// and a code c in 0..3 IS the fp4 number c / 2 once its two bits lie at the bottom of a nibble.  Products are
// multiples of 1/16 and the group sums of q * c stay below 2^18, so the fp32 accumulators hold them exactly: the drain is
// one fma per element and group instead of two instructions, and a packed weight dword becomes operands in 6
// instructions per 16 codes.
//
// The zero-point is in the accumulators from the start: the first matrix instruction of a group takes -zp * sum q / 16 of
// its rows as the addend (the quantising kernel writes it, one fp32 per row and group), a multiple of 1/16 like the
// products, so what is folded is the exact sum of q * (code - zp) and the running sums go through the oracle's values, bit
// for bit where K is not split.  (Taken off the running sums in one piece in front of the loop instead, the offset
// is about a hundred times the result on activations whose mean is not zero, and up to 2.3 % of the fp16 outputs rounded
// the other way.)  Per-group zero-points: centred on 2 in that way, what is missing of two groups at a time goes onto the
// running sums as a matrix product (groups of 128: two stages' at a time).  The addends cost LDS reads (16 or 32 of 16
// bytes a wave and stage of 128 rows) and no vector instruction, and the pass over the groups in front of the loop is gone.
//
// Measured: 38 cycles per 32x32x64 instruction with the 4 drain fmas of groups of 128 beside it, 49 with the 8 of
// groups of 64 (32 alone) in a probe; on random operands the faster matrix instructions run into the power limit
// (4096 x 14336 x 4096: 448 thousand cycles at 2.07 GHz against the int8 kernel's 556 at 2.43).  Layer calls with their
// quantisation in one run on one card, us: the int8 path / this kernel with the offset in front of the loop / this kernel:
// 4096 x 14336 x 4096 244 / 241 / 237, with per-group zero-points 276 / 263 / 257; 2048 x 28672 x 8192 in groups of 64
// 575 / 515 / 512, with per-group zero-points 726 / 629 / 583; 1024 x 14336 x 4096 80 / 74 / 72.  What is left over the
// matrix cores' own time is the vector instructions beside them (186 per 32 of them), prologue and epilogue of a tile, and the
// half-empty last round of tiles.
//
// Activation fragments (written by mx_quant_kernel): one of 2560 bytes per 32 rows x 64 elements, in operand order.
// Lane l holds row l & 31, elements 32 * (l >> 5) .. + 31: 16 bytes of fp4 digits at 16 * l, the first 16 bytes of its
// fp6 digits at 1024 + 16 * l, the other 8 at 2048 + 8 * l.  Slot j of the 32 is element 8 * (j / 8) + (j % 8) / 2 +
// 4 * (j % 2): the order in which the weight dwords of the streaming layout come apart into nibbles.
#include <algorithm>

#include "mx_launch.h"
#include "w2a8_launch.h"

namespace w2a8 {

namespace {

using namespace mx;
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v6i __attribute__((ext_vector_type(6)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

constexpr int kFp6 = 2, kFp4 = 4;          // operand formats of the f8f6f4 instructions
constexpr int kScaleOne = 127, kScale4 = 129;   // 2^(x - 127)

// ---- activations: per-token quantisation straight into digit fragments.  R rows per workgroup, 32 elements per thread (an
// fp6 conversion takes 32), R neighbouring lanes on the same elements of R rows: their pieces of a fragment are 16 * R bytes in
// one run, where one row's pieces are 16 bytes at a time, 2560 apart (the times stand at mx_quant_plan).  The rows are read
// once, whole cache lines at a time: a thread's 64 bytes are four lines' worth of address work per lane otherwise, so they turn
// through LDS: piece i of a thread's four lies at i * pitch + its chunk.  With pitch = 4 and a row = 16 / R modulo 16 pieces the 16
// lanes of a write's and of a read's phase fall into all banks.  The quotients are those of act_quant_keep_kernel, bit for
// bit.  32 consecutive rows go to one XCD, so that the pieces of a fragment meet in one L2.
template <bool BF16, int R>
__global__ __launch_bounds__(1024) void mx_quant_kernel(const uint16_t* __restrict__ x, int ldx, int M, int K, int group_size,
                                                        uint8_t* __restrict__ frag, float* __restrict__ cs, float centre,
                                                        float* __restrict__ s_a, unsigned* __restrict__ counters, int n_counters,
                                                        int pitch, int row_pieces) {
    __shared__ float red[16][R];
    const int xcd = blockIdx.x & 7, kth = blockIdx.x >> 3;
    constexpr int kSets = 32 / R;   // workgroups of 32 rows
    const int m0 = M >= 256 ? ((kth / kSets) * 8 + xcd) * 32 + kth % kSets * R : (int)blockIdx.x * R;
    if (m0 >= M) return;   // (uniform: the grid is rounded up to whole sets of rows)
    const int tid = threadIdx.x;
    if (m0 == 0)   // the arrival counters of a split GEMM behind this launch
        for (int i = tid; i < n_counters; i += (int)blockDim.x) counters[i] = 0u;
    const int r = tid % R, c = tid / R, m = m0 + r;
    const bool on = c * 32 < K && m < M;
    extern __shared__ __attribute__((aligned(16))) v4u row[];
    const int threads = (int)blockDim.x, pieces = K / 8;
    const auto widen = [](uint32_t w, float& a, float& b) {
        a = BF16 ? __uint_as_float(w << 16) : half_bits_to_float((uint16_t)(w & 0xffffu));
        b = BF16 ? __uint_as_float(w & 0xffff0000u) : half_bits_to_float((uint16_t)(w >> 16));
    };
    {
        // (threads / R >= K / 32: four rounds of threads / R pieces cover a row, the R rows one after the other)
        v4u raw[4];
        const int per = threads / R, lr = tid / per, lp = tid % per;   // the row and the piece this thread loads
        const v4u* src = reinterpret_cast<const v4u*>(x + (size_t)min(m0 + lr, M - 1) * ldx);
#pragma unroll
        for (int i = 0; i < 4; ++i) raw[i] = i * per + lp < pieces ? src[i * per + lp] : v4u{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = i * per + lp;
            if (p < pieces) row[lr * row_pieces + (p & 3) * pitch + (p >> 2)] = raw[i];
        }
    }
    __syncthreads();
    float f[32];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const v4u raw = on ? row[r * row_pieces + i * pitch + c] : v4u{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            widen(raw[k], f[8 * i + 2 * k], f[8 * i + 2 * k + 1]);
            amax = fmaxf(amax, fmaxf(fabsf(f[8 * i + 2 * k]), fabsf(f[8 * i + 2 * k + 1])));
        }
    }
#pragma unroll
    for (int off = 32; off >= R; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    const int waves = threads >> 6;
    if ((tid & 63) < R) red[tid >> 6][r] = amax;
    __syncthreads();
    amax = red[0][r];
    for (int w = 1; w < waves; ++w) amax = fmaxf(amax, red[w][r]);
    const float s = fmaxf(amax, 1e-9f) / 127.0f;
    if (c == 0 && m < M) s_a[m] = s;
    const float inv_s = 1.0f / s;

    float sumf = 0.0f;   // (whole numbers below 2^24: exact)
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        f[i] = fminf(fmaxf(rne_quotient(f[i], s, inv_s), -127.0f), 127.0f);
        sumf += f[i];
    }
    v4u hi;
    v16f lo_even, lo_odd;   // the rests in slot order: the conversion takes its two inputs alternately
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        uint32_t w = 0;
#define SLIMK_MX_PAIR(B)                                                                                       \
        w = (uint32_t)__builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, f[8 * d + B], f[8 * d + 4 + B], 32.0f, B);
        SLIMK_MX_PAIR(0) SLIMK_MX_PAIR(1) SLIMK_MX_PAIR(2) SLIMK_MX_PAIR(3)
#undef SLIMK_MX_PAIR
#define SLIMK_MX_REST(B)                                                                                       \
        {                                                                                                      \
            const v2f back = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 32.0f, B);                            \
            lo_even[4 * d + B] = f[8 * d + B] - back[0];                                                       \
            lo_odd[4 * d + B] = f[8 * d + 4 + B] - back[1];                                                    \
        }
        SLIMK_MX_REST(0) SLIMK_MX_REST(1) SLIMK_MX_REST(2) SLIMK_MX_REST(3)
#undef SLIMK_MX_REST
        hi[d] = w;
    }
    const v6i lo = __builtin_bit_cast(v6i, __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(lo_even, lo_odd, 8.0f));
    if (on) {
        const int steps2 = mx_padded_steps(K);
        uint8_t* dst = frag + ((size_t)(m >> 5) * steps2 + (c >> 1)) * kFragBytes;
        const int fl = (c & 1) * 32 + (m & 31);
        *reinterpret_cast<v4u*>(dst + fl * 16) = hi;
        *reinterpret_cast<v4i*>(dst + 1024 + fl * 16) = v4i{lo[0], lo[1], lo[2], lo[3]};
        *reinterpret_cast<v2i*>(dst + 2048 + fl * 8) = v2i{lo[4], lo[5]};
    }
    const int tpd = group_size == 64 ? 2 : 4;   // threads of a row per drain of the GEMM (all of a drain's are on or off)
    for (int off = 1; off < tpd; off <<= 1) sumf += __shfl_xor(sumf, off * R, 64);
    if (on && c % tpd == 0) cs[(size_t)(c / tpd) * M + m] = sumf * centre;
}

__device__ __forceinline__ v16f mfma_hi(v4i a, v4i b, v16f c) {   // 4 * a4 * c/2
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i{a[0], a[1], a[2], a[3], 0, 0, 0, 0}, v8i{b[0], b[1], b[2], b[3], 0, 0, 0, 0},
                                                           c, kFp4, kFp4, 0, kScale4, 0, kScaleOne);
}
__device__ __forceinline__ v16f mfma_lo(v4i a, v2i a2, v4i b, v16f c) {   // a6 * c/2
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v8i{a[0], a[1], a[2], a[3], a2[0], a2[1], 0, 0},
                                                           v8i{b[0], b[1], b[2], b[3], 0, 0, 0, 0}, c, kFp6, kFp4, 0, 0, 0, 0);
}

// The four raw dwords of a lane (16 elements of its quad x 4 channels) as the operands of the unit's two blocks of 32
// channels.  Two dwords' nibbles are interleaved first (a nibble then holds two channels' codes of one element), the
// masks leave one channel's code at the bottom of each nibble, and the row swap hands each half-wave both quads'
// elements of its own channel: block nb's lane l holds channel nb * 32 + (l & 31), elements 32 * (l >> 5) .. + 31.
__device__ __forceinline__ void unpack_unit(const v4i& raw, v4i (&b)[2]) {
    const v4u r = __builtin_bit_cast(v4u, raw);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t x = (r[2 * h] & 0x0f0f0f0fu) | ((r[2 * h + 1] << 4) & 0xf0f0f0f0u);
        uint32_t y = ((r[2 * h] >> 4) & 0x0f0f0f0fu) | (r[2 * h + 1] & 0xf0f0f0f0u);
        asm("" : "+v"(x), "+v"(y));   // (keeps the masks below from being folded back into the two merges: 6 more instructions)
        const v2u lo = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane16_swap(x & 0x33333333u, (x >> 2) & 0x33333333u, false, false));
        // (field 3 is stored with its high bit flipped)
        const v2u hi = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane16_swap(y & 0x33333333u, ((y >> 2) & 0x33333333u) ^ 0x22222222u, false, false));
        b[0][h] = (int)lo[0];
        b[0][2 + h] = (int)lo[1];
        b[1][h] = (int)hi[0];
        b[1][2 + h] = (int)hi[1];
    }
}

// Workgroup = 4 waves side by side along the channels (a strip of 64 each) x RB blocks of 32 token rows; per stage of
// 128 elements the activation fragments come into a three-slot LDS ring (LDS-direct, two stages ahead, shared by the
// waves), the wave's own weight units and scales into two wave-private slots (a wave moves a stage's units to registers
// before it asks for the units two stages on).
// BIAS: p.bias is added to the rounded outputs (whole 16-byte output rows only; instantiations of their own, as in tiled_bodies.h)
// GS = 64-element steps per drain: 1 (groups of 64) or 2 (128; groups of 256 drain twice with the same scale).
template <int RB, int GS, bool SPLIT, bool ZP, int WGS, typename OutT, bool BIAS>
__device__ __forceinline__ void mx_body(const MxParams& p) {
    constexpr int kABytes = RB * kStageSteps * kFragBytes;       // 20 or 10 KiB
    constexpr int kALoads = (kABytes / 1024 + 3) / 4;            // LDS-direct loads of 1 KiB per wave and stage: 5 or 3
    constexpr int kASlot = kABytes;
    constexpr int kSpare = kALoads * 4 * 1024 > kABytes ? 1024 : 0;   // RB = 2: where the two surplus loads land
    constexpr int kWBytes = kStripsPerWg * kStageSteps * kUnitBytes;
    constexpr int kSBytes = kStripsPerWg * 256;
    constexpr int kGroups = kStageSteps / GS;                    // drains of a block per stage
    constexpr int kCBytes = RB * kGroups * kFragRows * 4;
    constexpr int kCSlots = ZP && GS == 2 ? 3 : 2;              // (3: the zero-point correction takes two stages' sums)
    constexpr int kLds = 3 * kASlot + 2 * (kWBytes + kSBytes) + kCSlots * kCBytes + kSpare;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
    constexpr int kBM = RB * kFragRows;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    // tile order as in tiled_bodies.h: channel tiles that divide by eight go to the XCDs in bands, token tile major
    const int tiles_n = (p.strips + kStripsPerWg - 1) / kStripsPerWg, tiles_m = (p.M + kBM - 1) / kBM;
    const int total = tiles_m * tiles_n, per_xcd = (total + 7) / 8;
    const int xcd = (int)(blockIdx.x & 7), local = (int)(blockIdx.x >> 3);
    int tile, split_idx = 0;
    if (SPLIT) {
        const int counted = p.group_shift ? counted_splits((int)gridDim.y, (p.steps + 1) / 2, p.stages_per_split) : 0;
        if (!split_tile_place((int)blockIdx.x, (int)blockIdx.y, (int)gridDim.y, tiles_n, tiles_m, tile, split_idx, counted)) return;
        tile = __builtin_amdgcn_readfirstlane(tile);
        split_idx = __builtin_amdgcn_readfirstlane(split_idx);
    } else if (tiles_n % 8 == 0) {
        const int band = tiles_n / 8;
        tile = (local / band) * tiles_n + xcd * band + local % band;
    } else if (tiles_m >= 2 && tiles_m <= 4) {
        int n_tile, m_tile_i;
        if (!xcd_place((int)blockIdx.x, tiles_n, tiles_m, n_tile, m_tile_i)) return;
        tile = m_tile_i * tiles_n + n_tile;
    } else {
        tile = xcd * per_xcd + local;
    }
    if (!SPLIT && (local >= per_xcd || tile >= total)) return;
    const int m_tile = (tile / tiles_n) * kBM;
    const int strip_raw = (tile % tiles_n) * kStripsPerWg + wave;
    const int strip = min(strip_raw, p.strips - 1);   // a surplus wave recomputes the last strip and stores nothing
    const bool strip_ok = strip_raw < p.strips;

    const int steps2 = (p.steps + 1) / 2 * 2;
    const int all_stages = steps2 / 2;
    const int stage0 = SPLIT ? split_idx * p.stages_per_split : 0;
    const int n_stages = SPLIT ? min(p.stages_per_split, all_stages - stage0) : all_stages;

    const int row_blocks = (p.M + kFragRows - 1) / kFragRows;
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.frag), 0, (int)((size_t)row_blocks * steps2 * kFragBytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(p.w_r), 0, (int)min(weight_bytes(p.strips, p.steps), (size_t)0x7fffffff), 0x00020000);
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.s_r), 0, (int)min((size_t)p.strips * p.G * 128, (size_t)0x7fffffff), 0x00020000);
    const int drains = p.steps / GS;                       // of the whole reduction
    const __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.cs), 0, (int)((size_t)p.M * drains * 4), 0x00020000);

    // activations: chunk c = wave + 4 i of 1 KiB; a row block's two fragments of a stage are 5 chunks in one piece
    // (all of it the wave's, below 2 GiB: in scalar registers beside the lane's 16 bytes.  Said outright: with offsets that the
    // compiler computed in vector registers each load was a loop over their values.  A row block past the last repeats it)
    uint32_t a_off[kALoads];
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
        const int c = min(wave + 4 * i, kABytes / 1024 - 1), rb = c / 5;
        a_off[i] = (uint32_t)__builtin_amdgcn_readfirstlane(min(m_tile / kFragRows + rb, row_blocks - 1) * (steps2 * kFragBytes) + c % 5 * 1024);
    }
    const uint32_t run_pitch = (uint32_t)p.strips * (kRunSteps * kUnitBytes), strip_off = (uint32_t)strip * (kRunSteps * kUnitBytes);
    const uint32_t s_pitch = (uint32_t)p.strips * 128;     // bytes between groups
    const uint32_t s_voff = (GS == 1 ? half * s_pitch : 0u) + (lane & 31) * 4;
    uint8_t* const a_lds = lds;
    uint8_t* const w_lds = lds + 3 * kASlot + wave * (kStageSteps * kUnitBytes);
    uint8_t* const s_lds = lds + 3 * kASlot + 2 * kWBytes + wave * 256;
    uint8_t* const c_lds = lds + 3 * kASlot + 2 * (kWBytes + kSBytes);
    // centring sums: a stage's RB x kGroups pieces of 32 rows, two pieces a load (waves past the last one repeat an earlier
    // wave's load); drains past the end of K read as zero
    const int c_piece = wave % (kCBytes / 256) * 2 + half, c_rb = c_piece / kGroups, c_gi = c_piece % kGroups;
    const uint32_t c_off = ((uint32_t)c_gi * (uint32_t)p.M + (uint32_t)(m_tile + c_rb * kFragRows + col)) * 4u;

#define SLIMK_LDS_PTR(ptr) ((__attribute__((address_space(3))) void*)(ptr))
    auto fetch_a = [&](int stage, int slot) {
#pragma unroll
        for (int i = 0; i < kALoads; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, SLIMK_LDS_PTR(a_lds + (wave + 4 * i < kABytes / 1024 ? slot * kASlot + (wave + 4 * i) * 1024 : kLds - 1024)),
                                                     16, lane * 16, a_off[i] + (uint32_t)((stage0 + stage) * (kStageSteps * kFragBytes)), 0, 0);
    };
    auto fetch_w = [&](int stage, int slot) {
        const int st = (stage0 + stage) * kStageSteps;
        const uint32_t off = (uint32_t)(st / kRunSteps) * run_pitch + (uint32_t)(st % kRunSteps) * kUnitBytes + strip_off;
#pragma unroll
        for (int s = 0; s < kStageSteps; ++s)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, SLIMK_LDS_PTR(w_lds + slot * kWBytes + s * kUnitBytes), 16, lane * 16,
                                                     off + s * kUnitBytes, 0, 0);
        const int g = GS == 1 ? st : (stage0 + stage) >> p.group_shift;   // (past the last group: reads as zero)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, SLIMK_LDS_PTR(s_lds + slot * kSBytes), 4, s_voff,
                                                 g * s_pitch + (uint32_t)strip * 128, 0, 0);
    };
    auto fetch_c = [&](int stage, int slot) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(c_rsrc, SLIMK_LDS_PTR(c_lds + slot * kCBytes + wave % (kCBytes / 256) * 256), 4, c_off,
                                                 (uint32_t)((stage0 + stage) * kGroups) * (uint32_t)p.M * 4u, 0, 0);
    };
    constexpr int kLoads = kALoads + kStageSteps + 1;      // a wave's requests for activations, weights and scales per stage

    float t[RB][2][16];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int j = 0; j < 16; ++j) t[rb][nb][j] = 0.0f;

    fetch_c(0, 0);
    fetch_a(0, 0);
    fetch_w(0, 0);
    fetch_a(min(1, n_stages - 1), 1);
    fetch_w(min(1, n_stages - 1), 1);

    const int sub = (lane >> 4) & 1, c16 = lane & 15;      // channel nb * 32 + col = sub-block 2 nb + sub, column c16

    // ---- main loop.  A unit of work is (row block, drain of the stage, channel block): its instructions start from the
    // rows' centring sums and go into accumulator set u & 1 while the other set is folded into the running sums; the last
    // unit of a stage is folded at the top of the next.
    constexpr int kUnits = RB * 2 * kGroups;
    // Two workgroups on a CU (256 registers a lane): both channel blocks of a row block start from one copy of its centring
    // sums, and the next stage's raw weights are read ahead.  Three (168): each unit's sums are read into its accumulators
    // as soon as these are folded, the raw weights at the top of their stage.
    constexpr bool kShare = WGS == 2, kAhead = WGS == 2;
    v16f acc[2];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[0][j] = acc[1][j] = 0.0f;
    float sc_prev = 0.0f;
    const __amdgpu_buffer_rsrc_t z_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(ZP ? p.zp_r : reinterpret_cast<const uint8_t*>(p.s_r)), 0,
        (int)min((size_t)p.strips * p.G * 64, (size_t)0x7fffffff), 0x00020000);
    float sc_last[2] = {0.0f, 0.0f};                       // ZP, GS = 2: the scales of the stage before
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    int slot = 0, wslot = 0, cslot = 0;
    v4i raw[kStageSteps];
    uint16_t sraw[kGroups][2];
    auto read_w = [&](int ws) {                            // the wave's units and scales of a stage, LDS -> registers
        const uint8_t* w_st = w_lds + ws * kWBytes + lane * 16;
        const uint8_t* s_st = s_lds + ws * kSBytes + (c16 * 4 + sub) * 2;
#pragma unroll
        for (int s = 0; s < kStageSteps; ++s) raw[s] = *reinterpret_cast<const v4i*>(w_st + s * kUnitBytes);
#pragma unroll
        for (int gi = 0; gi < kGroups; ++gi)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) sraw[gi][nb] = *reinterpret_cast<const uint16_t*>(s_st + gi * 128 + nb * 4);
    };
    if (kAhead) {
        read_w(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    for (int stage = 0; stage < n_stages; ++stage) {
        const uint8_t* a_st = a_lds + slot * kASlot + lane * 16;
        const uint8_t* a_st8 = a_lds + slot * kASlot + 2048 + lane * 8;
        struct Frag { v4i hi, lo; v2i lo2; };
        Frag aq[kStageSteps];                              // a row block's two fragments, refilled behind their last use
        auto load_hi = [&](int rb, int st) { aq[st].hi = *reinterpret_cast<const v4i*>(a_st + (2 * rb + st) * kFragBytes); };
        auto load_lo = [&](int rb, int st) {
            aq[st].lo = *reinterpret_cast<const v4i*>(a_st + (2 * rb + st) * kFragBytes + 1024);
            // (volatile: two of these merged into one read would land outside the operands they belong to)
            aq[st].lo2 = *(const volatile __attribute__((address_space(3))) v2i*)(a_st8 + (2 * rb + st) * kFragBytes);
        };
        // the centring sums of the lane's 16 accumulator rows: the first addend of the units of (row block, drain) rc
        v16f start;
        auto load_start = [&](int rc, v16f& to) {
            const v4f* c_st = reinterpret_cast<const v4f*>(c_lds + cslot * kCBytes + rc * (kFragRows * 4) + half * 16);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v4f v = c_st[2 * i];
#pragma unroll
                for (int j = 0; j < 4; ++j) to[4 * i + j] = v[j];
            }
        };
        if (!kAhead) read_w(wslot);
        load_start(0, kShare ? start : acc[0]);
#pragma unroll
        for (int st = 0; st < kStageSteps; ++st) {
            load_hi(0, st);
            load_lo(0, st);
        }
        // The centring sums one stage on go where the stage before had them: every wave is past its reads.  They are asked
        // for first, so that the wait for all but the requests below covers them.  The rest two stages on: every wave is
        // past its reads of that activation slot, this wave past those of its weight slot.
        uint32_t z_zp = 0u;   // ZP: the zero-points of a drain (half 0: GS = 1 the stage's first, GS = 2 that of the stage before)
        if constexpr (ZP) {
            const int d = GS == 1 ? 2 * (stage0 + stage) + half : max(stage0 + stage - 1 + half, 0);
            z_zp = __builtin_amdgcn_raw_buffer_load_b32(z_rsrc, (((uint32_t)(d >> p.group_shift) * (uint32_t)p.strips + strip) * 16 + c16) * 4, 0, 0);
        }
        const int cnext = cslot == kCSlots - 1 ? 0 : cslot + 1;
        fetch_c(min(stage + 1, n_stages - 1), cnext);
        fetch_a(min(stage + 2, n_stages - 1), slot == 0 ? 2 : slot - 1);
        if (!kAhead) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        fetch_w(min(stage + 2, n_stages - 1), wslot);
        float sc[kGroups][2];
#pragma unroll
        for (int gi = 0; gi < kGroups; ++gi)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) sc[gi][nb] = half_bits_to_float(sraw[gi][nb]) * 16.0f;
        v4i b[kStageSteps][2];
#pragma unroll
        for (int s = 0; s < kStageSteps; ++s) unpack_unit(raw[s], b[s]);

#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            const int rb = u / (2 * kGroups), gi = (u / 2) % kGroups, nb = u % 2;
            const int pu = (u + kUnits - 1) % kUnits;
            const int prb = pu / (2 * kGroups), pgi = (pu / 2) % kGroups, pnb = pu % 2;
            const float scale = u == 0 ? sc_prev : sc[pgi][pnb];
            if (u == kUnits - 2 * kGroups) {
                // everything but this stage's own requests has landed: the next stage's weights are this wave's alone
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
                if (kAhead) read_w(wslot ^ 1);
            }
            // The previous unit is folded beside all but the first of this unit's instructions: its last result is not
            // there yet when that one issues.
            constexpr int kMfmas = 2 * GS;
#pragma unroll
            for (int i = 0; i < kMfmas; ++i) {
                const int st = gi * GS + i / 2;
                const Frag& a = aq[st];
                const v16f c = i == 0 && kShare ? start : acc[u & 1];
                acc[u & 1] = i % 2 == 0 ? mfma_hi(a.hi, b[st][nb], c) : mfma_lo(a.lo, a.lo2, b[st][nb], c);
                if (kShare && i == 0 && nb == 1 && u + 1 < kUnits) load_start(u / 2 + 1, start);
                if (rb + 1 < RB && nb == 1) {
                    if (i % 2 == 0) load_hi(rb + 1, st);
                    else load_lo(rb + 1, st);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (i > 0) {
#pragma unroll
                    for (int j = 16 * (i - 1) / (kMfmas - 1); j < 16 * i / (kMfmas - 1); ++j)
                        t[prb][pnb][j] = __builtin_fmaf(acc[(u & 1) ^ 1][j], scale, t[prb][pnb][j]);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (!kShare && i == kMfmas - 1 && u + 1 < kUnits) {
                    load_start((u + 1) / 2, acc[(u & 1) ^ 1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        sc_prev = sc[kGroups - 1][1];
        if constexpr (ZP) {
            // Per-group zero-points: (2 - zp) * scale * rowsum of two drains at a time, a half-wave supplying a drain, as a
            // matrix product onto the running sums.  The row sum (15 bits) comes apart into two bf16 numbers, 8 * (zp - 2) *
            // scale (19 bits) into three, exactly, and their six products are exact in fp32: half the matrix core's time
            // of v_mfma_f32_32x32x2_f32 and no vector load in flight beside the requests
            // (4096 x 14336 x 4096 278 -> 263 us).
            // (groups of 128: an odd number of stages ends with its last one alone, which half 1 supplies)
            if (GS == 1 || (stage & 1) || stage == n_stages - 1) {
                const bool on = GS == 1 || half == 1 || (stage & 1);
                const uint8_t* const c_st = GS == 1 ? c_lds + cslot * kCBytes + half * (kFragRows * 4)
                                                    : c_lds + (half == 1 || !(stage & 1) ? cslot : cslot == 0 ? kCSlots - 1 : cslot - 1) * kCBytes;
                const auto upper = [](float v) { return __float_as_uint(v) & 0xffff0000u; };
                v4u zb[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float scale0 = GS == 1 ? sc[0][i] : sc_last[i], scale1 = sc[kGroups - 1][i];   // (16 times the scales)
                    const float scale = half == 1 ? scale1 : scale0;
                    float z = on ? ((float)((z_zp >> (8 * (2 * i + sub))) & 0xffu) - 2.0f) * 0.5f * scale : 0.0f;
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const uint32_t u = upper(z);
                        zb[i][d] = u | (u >> 16);
                        z -= __uint_as_float(u);
                    }
                    zb[i][3] = 0u;
                }
#pragma unroll
                for (int rb = RB - 1; rb >= 0; --rb) {
                    const float sum = *reinterpret_cast<const float*>(c_st + rb * (kGroups * kFragRows * 4) + col * 4);
                    const uint32_t u = upper(sum);
                    const uint32_t pair = (u >> 16) | upper(sum - __uint_as_float(u));
                    const v4u za = {pair, pair, pair, 0u};
#pragma unroll
                    for (int i = 1; i >= 0; --i) {
                        v16f c;
#pragma unroll
                        for (int j = 0; j < 16; ++j) c[j] = t[rb][i][j];
                        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, za), __builtin_bit_cast(v8b, zb[i]), c, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 16; ++j) t[rb][i][j] = c[j];
                    }
                }
            }
            if (GS == 2) {
                sc_last[0] = sc[0][0];
                sc_last[1] = sc[0][1];
            }
        }
        // (the wave's requests for the next stage landed above) meet the other waves
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        slot = slot == 2 ? 0 : slot + 1;
        wslot ^= 1;
        cslot = cnext;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j)
        t[RB - 1][1][j] = __builtin_fmaf(acc[(kUnits - 1) & 1][j], sc_prev, t[RB - 1][1][j]);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");   // the last (repeated) requests have landed: LDS is free

    uint16_t* out = reinterpret_cast<uint16_t*>(p.out);
    if (SPLIT) {
        // publish the partial sums, the last workgroup of the tile adds them up in split order: as in tiled_bodies.h
        // (write-through 16-byte stores, each followed by the idle cycles its data registers need before reuse)
        constexpr int kTileBytes = kBM * 256 * 4;
        constexpr int kCoherent = 17;  // sc0 | sc1
        const int n_split = (int)gridDim.y;
        const __amdgpu_buffer_rsrc_t ws_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            p.ws_partial, 0, (int)((size_t)n_split * total * kTileBytes), 0x00020000);
        const uint32_t ws_lane = (uint32_t)wave * (RB * 2 * 4 * 1024) + lane * 16;
        const uint32_t ws_tile = (uint32_t)tile * kTileBytes, ws_pitch = (uint32_t)total * kTileBytes;
        uint32_t ws_off[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            ws_off[rb] = ws_lane + rb * 8192 + (uint32_t)split_idx * ws_pitch + ws_tile;
            asm volatile("" : "+v"(ws_off[rb]));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float* tv = &t[rb][i / 4][(i % 4) * 4];
                const v4f v = {tv[0], tv[1], tv[2], tv[3]};
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), ws_rsrc, ws_off[rb] + i * 1024, 0, kCoherent);
                asm volatile("s_nop 1" ::: "memory");
            }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        if (tid == 0) {
            const unsigned prev = __hip_atomic_fetch_add(p.ws_counter + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *reinterpret_cast<uint32_t*>(lds) = (prev == (unsigned)(n_split - 1));
        }
        __syncthreads();
        const bool last = *reinterpret_cast<uint32_t*>(lds) != 0;
        if (!last) return;
        __syncthreads();   // (the verdict is read before the output staging overwrites it)
        constexpr int kChunk = 2;   // row blocks whose fragments are in flight together
#pragma unroll
        for (int rb0 = 0; rb0 < RB; rb0 += kChunk) {
#pragma unroll
            for (int rb = 0; rb < kChunk; ++rb)
#pragma unroll
                for (int j = 0; j < 32; ++j) t[rb0 + rb][j / 16][j % 16] = 0.0f;
            for (int sp = 0; sp < n_split; ++sp) {
                v4f v[kChunk][8];
#pragma unroll
                for (int rb = 0; rb < kChunk; ++rb)
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        v[rb][i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                            ws_rsrc, ws_lane + (rb0 + rb) * 8192 + i * 1024, sp * ws_pitch + ws_tile, kCoherent));
#pragma unroll
                for (int rb = 0; rb < kChunk; ++rb)
#pragma unroll
                    for (int j = 0; j < 32; ++j) t[rb0 + rb][j / 16][j % 16] += v[rb][j / 4][j % 4];
            }
        }
        if (tid == 0) __hip_atomic_store(p.ws_counter + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---- epilogue: out = cast(t * s_a[m]); lane (col, half), element j: row (j & 3) + 8 * (j >> 2) + 4 * half
    if (!strip_ok) return;
    const bool wide = (p.N & 7) == 0 && (p.ldo & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    constexpr int kPitch = 72;   // floats: the half-waves' rows (4 apart) fall into different halves of the banks
    static_assert(32 * kPitch * 4 * kStripsPerWg <= kLds, "output staging exceeds the stage buffers");
    float* stage_out = reinterpret_cast<float*>(lds) + wave * (32 * kPitch);
    // the token scales, four rows a load, all in flight together (rows past M: zero, or what the scratch holds behind them)
    const __amdgpu_buffer_rsrc_t sa_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.s_a), 0, (p.M + 3) / 4 * 16, 0x00020000);
    out8 bias8 = {0, 0, 0, 0};
    if constexpr (BIAS) bias8 = *reinterpret_cast<const out8*>(p.bias + min(strip * kStripN + (lane & 7) * 8, p.N - 8));
    v4f sa4[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            sa4[rb][i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(sa_rsrc, (m_tile + rb * 32 + i * 8 + 4 * half) * 4, 0, 0));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        float sa[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) sa[j] = sa4[rb][j >> 2][j & 3];
        if (wide) {
            // 8 channels = one 16-byte store per lane: the values turn through the wave's corner of LDS
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    stage_out[((j & 3) + 8 * (j >> 2) + 4 * half) * kPitch + nb * 32 + col] = t[rb][nb][j] * sa[j];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = i * 8 + (lane >> 3), cg = lane & 7;
                const v4f lo = *reinterpret_cast<const v4f*>(stage_out + row * kPitch + cg * 8);
                const v4f hi = *reinterpret_cast<const v4f*>(stage_out + row * kPitch + cg * 8 + 4);
                v4u v;
                v.x = (uint32_t)OutT::cast(lo.x) | ((uint32_t)OutT::cast(lo.y) << 16);
                v.y = (uint32_t)OutT::cast(lo.z) | ((uint32_t)OutT::cast(lo.w) << 16);
                v.z = (uint32_t)OutT::cast(hi.x) | ((uint32_t)OutT::cast(hi.y) << 16);
                v.w = (uint32_t)OutT::cast(hi.z) | ((uint32_t)OutT::cast(hi.w) << 16);
                if constexpr (BIAS) v = add_bias8<OutT>(v, bias8);
                const int m = m_tile + rb * 32 + row, n = strip * kStripN + cg * 8;
                if (m < p.M && n < p.N) *reinterpret_cast<v4u*>(out + (size_t)m * p.ldo + n) = v;
            }
        } else {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int m = m_tile + rb * 32 + (j & 3) + 8 * (j >> 2) + 4 * half, n = strip * kStripN + nb * 32 + col;
                    if (m < p.M && n < p.N) out[(size_t)m * p.ldo + n] = OutT::cast(t[rb][nb][j] * sa[j]);
                }
        }
    }
}

// 128-row tiles: two workgroups per CU (80 KiB of LDS and 256 registers each); 64-row tiles two or three
template <int RB, int GS, bool SPLIT, bool ZP, int WGS, typename OutT, bool BIAS>
__global__ __launch_bounds__(256, WGS) void mx_gemm_kernel(const MxParams p) {
    mx_body<RB, GS, SPLIT, ZP, WGS, OutT, BIAS>(p);
}

template <int RB, int GS, int WGS>
void launch_rb_gs(const MxParams& p, bool out_bf16, dim3 grid, hipStream_t stream) {
    const dim3 block(256);
    const bool biased = p.bias != nullptr && output_rows_whole(p.out, p.ldo, p.N);
#define SLIMK_MX_LAUNCH_OUT(SPLITV, ZPV, OUT)                                                                  \
    do {                                                                                                       \
        if (biased) mx_gemm_kernel<RB, GS, SPLITV, ZPV, WGS, OUT, true><<<grid, block, 0, stream>>>(p);        \
        else mx_gemm_kernel<RB, GS, SPLITV, ZPV, WGS, OUT, false><<<grid, block, 0, stream>>>(p);              \
    } while (0)
#define SLIMK_MX_LAUNCH(SPLITV, ZPV)                                  \
    do {                                                              \
        if (out_bf16) SLIMK_MX_LAUNCH_OUT(SPLITV, ZPV, OutBF16);      \
        else SLIMK_MX_LAUNCH_OUT(SPLITV, ZPV, OutF16);                \
    } while (0)
    const bool zp = p.zp_r != nullptr;
    if (p.split > 1) {
        if (zp) SLIMK_MX_LAUNCH(true, true);
        else SLIMK_MX_LAUNCH(true, false);
    } else {
        if (zp) SLIMK_MX_LAUNCH(false, true);
        else SLIMK_MX_LAUNCH(false, false);
    }
#undef SLIMK_MX_LAUNCH
#undef SLIMK_MX_LAUNCH_OUT
}

}  // namespace

// The predicted time of a layer call in this form (us, quantisation included): start-up, quantisation, the round trip of
// the partial sums, and stages per workgroup times what one, two or more workgroups of a CU take for a stage together, more
// of it in groups of 64 (twice the drains) and with per-group zero-points.  Least squares on the logarithm over 3482 timed
// plans of drawn shapes and of thirteen decoder matrices (2048..28672 channels, K = 2048..28672, groups of 64 and 128,
// 96..2048 rows, symmetric and per-group zero-points): 5.9 % rms, 5.7 % on 2690 plans of other shapes.
float mx_predicted_time(int M, int N, int K, int group_size, int per_group_zp, int rb, int split) {
    const int stages = mx_padded_steps(K) / 2, per = (stages + split - 1) / split;
    const int tiles = ((N + 255) / 256) * ((M + rb * kFragRows - 1) / (rb * kFragRows));
    const int n = (tiles * split + 255) / 256;
    float each = rb == 2 ? (n == 1 ? 0.596f : n == 2 ? 0.857f : 0.4234f * (float)n)
                         : (n == 1 ? 0.977f : n == 2 ? 1.463f : 0.757f * (float)n);
    if (group_size == 64) each *= 1.257f;
    if (per_group_zp) each *= group_size == 64 ? 1.145f : 1.129f;
    const float sums = split > 1 ? 0.0886e-6f * 8.0f * (float)split * (float)M * (float)N : 0.0f;
    return 13.7f + 1.119e-6f * (float)M * (float)K + sums + ((float)per + 2.87f) * each;
}

// 128-row tiles where they fill the chip; otherwise the tile height and K split with the smallest predicted time
// (1024 x 14336 x 4096: 448 128-row tiles unsplit 74 us, 64-row tiles 94; 512 x 8192 x 28672: 128-row tiles in four splits
// 142 us, unsplit 243, 64-row tiles 150..233).
MxPlan mx_plan(int M, int N, int K, int group_size) {
    const int tiles_n = ((N + kStripN - 1) / kStripN + kStripsPerWg - 1) / kStripsPerWg;
    const int stages = mx_padded_steps(K) / 2;
    MxPlan plan{4, tiles_n * ((M + 127) / 128), 1, stages};
    if (plan.tiles >= 2 * 256) return plan;
    int best_split = 1;
    float best = 1e30f;
    for (int rb = 2; rb <= 4; rb += 2) {
        const int tiles = tiles_n * ((M + rb * kFragRows - 1) / (rb * kFragRows));
        for (int split : {1, 2, 3, 4, 6, 8}) {
            if (split > 1 && (stages / split < 6 || tiles * split > 1100)) break;
            const float time = mx_predicted_time(M, N, K, group_size, 0, rb, split);
            if (time < best) {
                best = time;
                best_split = split;
                plan.rb = rb;
                plan.tiles = tiles;
            }
        }
    }
    int per = (stages + best_split - 1) / best_split;
    if (group_size == 256) per = (per + 1) / 2 * 2;   // (a split owns whole groups)
    plan.stages_per_split = per;
    plan.split = (stages + per - 1) / per;
    return plan;
}

// How the quantising kernel's workgroups hold their rows in LDS (in pieces of 16 bytes), and how many rows they have.
namespace {
struct MxQuantPlan { int rows, pitch, row_pieces; };
constexpr int kMxQuantLds = 65536 - 256;   // beside the waves' maxima
MxQuantPlan mx_quant_layout(int K, int rows) {
    const int chunks = K / 32, pitch = (chunks + 27) / 16 * 16 - 12;   // 4 modulo 16
    const MxQuantPlan plan{rows, pitch, 4 * pitch + 16 / rows};
    if (rows == 1 && plan.row_pieces * 16 > kMxQuantLds) return {1, chunks, 4 * chunks};   // (the longest rows: without the padding)
    return plan;
}
}  // namespace
// Two rows where there are more than 256 of them and two fit, with other workgroups beside them on the CU: 4096 x 4096 17.6 ->
// 14.6 us, 2048 x 8192 17.9 -> 15.7, 1024 x 11008 15.1 -> 11.3; up to 256 rows one (256 x 6144 5.4 against 5.9), 2048 x 14336 27.9
// against 29.0.  Four rows: level (4096 x 4096 15.4, 2048 x 8192 15.6).
static MxQuantPlan mx_quant_plan(int M, int K) { return mx_quant_layout(K, M > 256 && K <= 11264 ? 2 : 1); }

hipError_t launch_mx_quant(const void* x, int ldx, bool x_bf16, int M, int K, int group_size, int centre, uint8_t* frag, float* cs,
                           float* s_a, unsigned* counters, int n_counters, hipStream_t stream) {
    const float f = -(float)centre / 16.0f;   // (the accumulators hold sums of q * code / 16)
    const MxQuantPlan plan = mx_quant_plan(M, K);
    const int rows = plan.rows;
    const dim3 grid((unsigned)(M >= 256 ? (M + 255) / 256 * (256 / rows) : (M + rows - 1) / rows));
    const dim3 block((unsigned)((K / 32 * rows + 63) / 64 * 64));
    const size_t lds = (size_t)rows * plan.row_pieces * 16;
#define SLIMK_MX_QUANT(R)                                                                                                            \
    do {                                                                                                                             \
        if (x_bf16) mx_quant_kernel<true, R><<<grid, block, lds, stream>>>((const uint16_t*)x, ldx, M, K, group_size, frag, cs, f, s_a, counters, n_counters, plan.pitch, plan.row_pieces); \
        else mx_quant_kernel<false, R><<<grid, block, lds, stream>>>((const uint16_t*)x, ldx, M, K, group_size, frag, cs, f, s_a, counters, n_counters, plan.pitch, plan.row_pieces);       \
    } while (0)
    if (rows == 2) SLIMK_MX_QUANT(2);
    else SLIMK_MX_QUANT(1);
#undef SLIMK_MX_QUANT
    return hipGetLastError();
}

hipError_t launch_mx_gemm(const MxParams& p, int rb, int gs, bool out_bf16, hipStream_t stream) {
    const int bm = rb * kFragRows;
    const int tiles = ((p.strips + kStripsPerWg - 1) / kStripsPerWg) * ((p.M + bm - 1) / bm);
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)p.split);
    if (rb == 4) {
        if (gs == 1) launch_rb_gs<4, 1, 2>(p, out_bf16, grid, stream);
        else launch_rb_gs<4, 2, 2>(p, out_bf16, grid, stream);
    } else if (tiles * p.split <= 2 * 256) {
        if (gs == 1) launch_rb_gs<2, 1, 2>(p, out_bf16, grid, stream);
        else launch_rb_gs<2, 2, 2>(p, out_bf16, grid, stream);
    } else {
        if (gs == 1) launch_rb_gs<2, 1, 3>(p, out_bf16, grid, stream);
        else launch_rb_gs<2, 2, 3>(p, out_bf16, grid, stream);
    }
    return hipGetLastError();
}

}  // namespace w2a8
