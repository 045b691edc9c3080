// Weight-only W2 GEMM for gfx950, many token rows: fp16 / bf16 activations times 2-bit weights on the fp16 / bf16
// matrix cores (v_mfma_f32_32x32x16), tiles through LDS.  The few-rows kernel (gemm_w2a16.hip) takes 16 rows per
// workgroup and unpacks the weights again for each of them; here an unpacked operand serves 64 or 128 rows.
//
// Workgroup = 4 waves side by side along the channels (a strip of 64 each) x RB blocks of 32 token rows, stages of 64
// reduction elements.  Activations come LDS-direct from the row-major matrix, each lane at the address of its operand
// (1 KiB per 32 rows x 16 elements, lane-major: every fragment read is one conflict-free ds_read_b128), two stages
// ahead through a ring of three; the wave's weight unit, scales and zero-points take the same road into wave-private
// places of the ring.
//
// The operand is exactly code - zp, for either type: a byte of four codes is the selector of two v_perm_b32 that look
// up the high and low bytes of the four possible values, two more put the bytes together (6 instructions per 4
// codes; fp16 with a uniform zero-point needs no low bytes).  Before the look-up a row swap hands each half-wave the
// codes of its own channel.  The stage's fp32 sums are folded into the running sums with the group's scale (one fma
// per element and 64 elements, whatever the group size).
#include <algorithm>

#include "w2a8_launch.h"

namespace w2a8 {

namespace {

typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

constexpr int kStripsPerWg = 4;

template <bool XBF>
__device__ __forceinline__ v16f mfma16(v4u a, v4u b, v16f c) {
    if constexpr (XBF) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// the high and the low bytes of (0, 1, 2, 3) - z in the activations' type, byte c for code c (z <= 255: exact)
struct CodeTable { uint32_t hi, lo; };
template <bool XBF>
__device__ __forceinline__ CodeTable code_table(int z) {
    uint32_t v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float f = (float)(c - z);
        v[c] = XBF ? __float_as_uint(f) >> 16 : (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
    }
    const uint32_t v01 = v[0] | (v[1] << 16), v23 = v[2] | (v[3] << 16);
    return {__builtin_amdgcn_perm(v23, v01, 0x07050301u), __builtin_amdgcn_perm(v23, v01, 0x06040200u)};
}

// KP = 2: eight waves, the second four on the second half of the workgroup's steps in a ring of their own; the halves
// meet in LDS (half the partial sums of a split launch with as many waves on a CU).
// BIAS: p.bias is added to the rounded outputs, on whole 16-byte output rows only (instantiations of their own: the branch for it
// cost unsplit calls without one 1 to 4 %, in graphs 535 x 10024 x 4096 in asymmetric groups of 256 74.1 -> 77.3 us).
template <int RB, int KP, bool ZP, bool PARTIAL, typename OutT, bool XBF, bool BIAS>
__device__ __forceinline__ void w2a16_tiled_body(const W2A16Params& p, const int steps_per_split, const int group_shift) {
    constexpr int kBM = RB * 32;
    constexpr int kASlot = RB * 4096, kWSlot = kStripsPerWg * kUnitBytes, kSSlot = kStripsPerWg * 256;
    constexpr int kSlot = kASlot + kWSlot + kSSlot * (ZP ? 2 : 1);
    constexpr int kLds = 3 * kSlot;   // a ring
    constexpr int kPitch = 72;   // floats of an output staging row
    static_assert(32 * kPitch * 4 * kStripsPerWg <= kLds, "output staging exceeds the stage buffers");
    __shared__ __attribute__((aligned(16))) uint8_t lds_all[KP * kLds];

    const int tid = threadIdx.x, lane = tid & 63;
    const int kh = KP == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & (kStripsPerWg - 1);
    uint8_t* const lds = lds_all + kh * kLds;
    const int col = lane & 31, half = lane >> 5, c16 = lane & 15, sub = (lane >> 4) & 1;
    const uint16_t* const bias = BIAS ? early_bias(p.bias) : nullptr;
    // token tiles of a channel tile next to each other on one XCD: they read the same weights
    const int tiles_n = (p.strips + kStripsPerWg - 1) / kStripsPerWg, tiles_m = (p.M + kBM - 1) / kBM;
    // ((split, channel tile) pairs dealt out together where split by split is uneven: 360 x 1584 x 11264 43.5 -> 28.1 us, 505 x
    // 5360 x 11520 119 -> 84.  The partial sums meet in a second launch: no split has to share an XCD with another.)
    int n_tile, m_tile_i, split_idx = PARTIAL ? (int)blockIdx.y : 0;
    if (PARTIAL && splits_uneven(tiles_n * tiles_m, (int)gridDim.y)) {
        int set;
        if (!xcd_place((int)(blockIdx.y * gridDim.x + blockIdx.x), tiles_n * (int)gridDim.y, tiles_m, set, m_tile_i)) return;
        split_idx = __builtin_amdgcn_readfirstlane(set / tiles_n);
        n_tile = __builtin_amdgcn_readfirstlane(set % tiles_n);
    } else if (!xcd_place((int)blockIdx.x, tiles_n, tiles_m, n_tile, m_tile_i)) {
        return;
    }
    const int m_tile = m_tile_i * kBM;
    const int strip_raw = n_tile * kStripsPerWg + wave;
    const int strip = min(strip_raw, p.strips - 1);   // a surplus wave recomputes the last strip and stores nothing
    const bool strip_ok = strip_raw < p.strips;
    // (KP = 2: an even number of steps in every split, so that the halves meet at the same barriers; no split is empty)
    const int wg_step0 = PARTIAL ? split_idx * steps_per_split : 0;
    const int wg_steps = PARTIAL ? min(steps_per_split, p.steps - wg_step0) : p.steps;
    const int n_steps = wg_steps / KP, step0 = wg_step0 + kh * n_steps;

    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.x), 0, (int)min(((size_t)(p.M - 1) * p.ldx + p.K) * 2, (size_t)0x7fffffff), 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(p.w_r), 0, (int)min(weight_bytes(p.strips, p.steps), (size_t)0x7fffffff), 0x00020000);
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.s_r), 0, (int)min((size_t)p.strips * p.G * 128, (size_t)0x7fffffff), 0x00020000);
    const __amdgpu_buffer_rsrc_t z_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(ZP ? p.zp_r : reinterpret_cast<const uint8_t*>(p.s_r)), 0,
        (int)min((size_t)p.strips * p.G * 64, (size_t)0x7fffffff), 0x00020000);

    // Wave w fetches piece w of every row block: elements (2 * half + (w >> 1)) * 16 + (w & 1) * 8 .. + 7 of the step
    // (the elements a half-wave's weight codes hold after the row swap).  Rows past M read as zero: their offset lies
    // past the buffer.
    uint32_t x_off[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int row = m_tile + rb * 32 + col;
        x_off[rb] = row < p.M ? (uint32_t)row * (uint32_t)p.ldx * 2u + ((2 * half + (wave >> 1)) * 16 + (wave & 1) * 8) * 2u : 0x80000000u;
    }
    const uint32_t run_pitch = (uint32_t)p.strips * (kRunSteps * kUnitBytes), strip_off = (uint32_t)strip * (kRunSteps * kUnitBytes);
#define SLIMK_LDS_PTR(ptr) ((__attribute__((address_space(3))) void*)(ptr))
    auto fetch = [&](int step, int slot) {
        uint8_t* const base = lds + slot * kSlot;
        const int st = step0 + step, g = st >> group_shift;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, SLIMK_LDS_PTR(base + (rb * 4 + wave) * 1024), 16, x_off[rb], st * (kStepK * 2), 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, SLIMK_LDS_PTR(base + kASlot + wave * kUnitBytes), 16, lane * 16,
                                                 (uint32_t)(st / kRunSteps) * run_pitch + (uint32_t)(st % kRunSteps) * kUnitBytes + strip_off, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, SLIMK_LDS_PTR(base + kASlot + kWSlot + wave * 256), 4, (lane & 31) * 4,
                                                 ((uint32_t)g * p.strips + strip) * 128u, 0, 0);
        if constexpr (ZP)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(z_rsrc, SLIMK_LDS_PTR(base + kASlot + kWSlot + kSSlot + wave * 256), 4, (lane & 15) * 4,
                                                     ((uint32_t)g * p.strips + strip) * 64u, 0, 0);
    };
#undef SLIMK_LDS_PTR
    constexpr int kLoads = RB + 2 + (ZP ? 1 : 0);   // LDS-direct loads of a wave per stage

    v4i raw;
    uint16_t sraw[2];
    uint32_t zraw = 0;
    auto read_w = [&](int slot) {   // the wave's unit, scales and zero-points of a stage, LDS -> registers
        const uint8_t* base = lds + slot * kSlot + kASlot;
        raw = *reinterpret_cast<const v4i*>(base + wave * kUnitBytes + lane * 16);
        const uint8_t* s = base + kWSlot + wave * 256 + (c16 * 4 + sub) * 2;
        sraw[0] = *reinterpret_cast<const uint16_t*>(s);
        sraw[1] = *reinterpret_cast<const uint16_t*>(s + 4);
        if constexpr (ZP) zraw = *reinterpret_cast<const uint32_t*>(base + kWSlot + kSSlot + wave * 256 + c16 * 4);
    };
    const CodeTable uniform = code_table<XBF>(p.zp_const);

    float t[RB][2][16];
    v16f acc[2];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[0][j] = acc[1][j] = 0.0f;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int j = 0; j < 32; ++j) t[rb][j / 16][j % 16] = 0.0f;
    float sc_prev = 0.0f;

    fetch(0, 0);
    fetch(min(1, n_steps - 1), 1);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kLoads) : "memory");
    read_w(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

    int slot = 0;
    for (int step = 0; step < n_steps; ++step) {
        const int next = slot == 2 ? 0 : slot + 1;
        const uint8_t* const a_st = lds + slot * kSlot + lane * 16;
        // fragments of a row block: two sets of registers, or (64-row tiles, three waves per SIMD) one whose pieces are
        // refilled behind their last use
        constexpr int kSets = RB == 4 ? 2 : 1;
        v4u aq[kSets][4];
        auto load_a = [&](int rb, int c) { aq[rb % kSets][c] = *reinterpret_cast<const v4u*>(a_st + (rb * 4 + c) * 1024); };
#pragma unroll
        for (int c = 0; c < 4; ++c) load_a(0, c);
        fetch(min(step + 2, n_steps - 1), slot == 0 ? 2 : slot - 1);   // (every wave is past its reads of that slot)
        const float sc[2] = {half_bits_to_float(sraw[0]), half_bits_to_float(sraw[1])};

        // b[nb][c]: piece c = 2 * odd + h of the channels nb * 32 + col
        v4u b[2][4];
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const CodeTable tab = ZP ? code_table<XBF>((zraw >> (8 * (2 * nb + sub))) & 0xffu) : uniform;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t w = (uint32_t)raw[i];
                const uint32_t s0 = (w >> (4 * nb)) & 0x03030303u;
                const uint32_t s1 = nb == 0 ? (w >> 2) & 0x03030303u : ((w >> 6) & 0x03030303u) ^ 0x02020202u;   // (field 3 is stored flipped)
                const v2u sel = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane16_swap(s0, s1, false, false));
#pragma unroll
                for (int odd = 0; odd < 2; ++odd) {
                    const uint32_t hi = __builtin_amdgcn_perm(0u, tab.hi, sel[odd]);
                    uint32_t lo01, lo23;
                    if constexpr (!XBF && !ZP) {   // (|code - zp| <= 3: the low bytes are zero)
                        lo01 = __builtin_amdgcn_perm(0u, hi, 0x010c000cu);
                        lo23 = __builtin_amdgcn_perm(0u, hi, 0x030c020cu);
                    } else {
                        const uint32_t lo = __builtin_amdgcn_perm(0u, tab.lo, sel[odd]);
                        lo01 = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
                        lo23 = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
                    }
                    b[nb][odd * 2 + i / 2][(i % 2) * 2] = lo01;
                    b[nb][odd * 2 + i / 2][(i % 2) * 2 + 1] = lo23;
                }
            }
        }

        // A unit of work is (row block, channel block): its four instructions go into accumulator set u & 1 while the
        // other set is folded into the running sums (not beside the first: its last result is not there yet)
        constexpr int kUnits = RB * 2;
#pragma unroll
        for (int u = 0; u < kUnits; ++u) {
            const int rb = u / 2, nb = u % 2, prb = ((u + kUnits - 1) % kUnits) / 2, pnb = nb ^ 1;
            const float scale = u == 0 ? sc_prev : sc[pnb];
            if (nb == 0) {
                if (rb + 1 < RB) {
                    if (kSets == 2)
#pragma unroll
                        for (int c = 0; c < 4; ++c) load_a(rb + 1, c);
                } else {
                    // everything but this stage's own requests has landed: the next stage's weights are this wave's alone
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads) : "memory");
                    read_w(next);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                v16f zero;
#pragma unroll
                for (int j = 0; j < 16; ++j) zero[j] = 0.0f;
                acc[u & 1] = mfma16<XBF>(aq[rb % kSets][c], b[nb][c], c == 0 ? zero : acc[u & 1]);
                if (kSets == 1 && nb == 1 && rb + 1 < RB) load_a(rb + 1, c);
                __builtin_amdgcn_sched_barrier(0);
                if (c > 0) {
#pragma unroll
                    for (int j = 16 * (c - 1) / 3; j < 16 * c / 3; ++j)
                        t[prb][pnb][j] = __builtin_fmaf(acc[(u & 1) ^ 1][j], scale, t[prb][pnb][j]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        sc_prev = sc[1];
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (this wave's requests for the next stage landed above)
        slot = next;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) t[RB - 1][1][j] = __builtin_fmaf(acc[1][j], sc_prev, t[RB - 1][1][j]);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");   // the last (repeated) requests have landed: LDS is free
    if constexpr (KP == 2) {   // the second half's running sums, lane-linear, into the first half's
        constexpr int kSums = RB * 8 * 1024;   // bytes of a wave
        static_assert(kStripsPerWg * kSums <= KP * kLds, "the halves' exchange exceeds the rings");
        v4f* const meet = reinterpret_cast<v4f*>(lds_all + wave * kSums) + lane;
        if (kh == 1) {
#pragma unroll
            for (int i = 0; i < RB * 8; ++i) {
                const float* tv = &t[i / 8][(i / 4) % 2][(i % 4) * 4];
                meet[i * 64] = v4f{tv[0], tv[1], tv[2], tv[3]};
            }
        }
        __syncthreads();
        if (kh == 0) {
#pragma unroll
            for (int i = 0; i < RB * 8; ++i) {
                const v4f v = meet[i * 64];
#pragma unroll
                for (int j = 0; j < 4; ++j) t[i / 8][(i / 4) % 2][(i % 4) * 4 + j] += v[j];
            }
        }
        __syncthreads();       // (the output staging goes over the same memory)
        if (kh == 1) return;
    }
    if (!strip_ok) return;

    if constexpr (PARTIAL) {   // fp32 partial sums [split][M][N]: 128 bytes of a row per half-wave and store
        float* ws = p.ws + (size_t)split_idx * p.M * p.N;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int m = m_tile + rb * 32 + (j & 3) + 8 * (j >> 2) + 4 * half, n = strip * kStripN + nb * 32 + col;
                    if (m < p.M && n < p.N) ws[(size_t)m * p.N + n] = t[rb][nb][j];
                }
        return;
    }
    uint16_t* out = reinterpret_cast<uint16_t*>(p.out);
    const bool wide = (p.N & 7) == 0 && (p.ldo & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    float* stage_out = reinterpret_cast<float*>(lds) + wave * (32 * kPitch);
    out8 bias8 = {0, 0, 0, 0};
    if constexpr (BIAS) bias8 = *reinterpret_cast<const out8*>(bias + min(strip * kStripN + (lane & 7) * 8, p.N - 8));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        if (wide) {
            // 8 channels = one 16-byte store per lane: the values turn through the wave's corner of LDS
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    stage_out[((j & 3) + 8 * (j >> 2) + 4 * half) * kPitch + nb * 32 + col] = t[rb][nb][j];
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
                    if (m < p.M && n < p.N) out[(size_t)m * p.ldo + n] = OutT::cast(t[rb][nb][j]);
                }
        }
    }
}

// (four-wave workgroups: two of 128 or three of 64 rows per CU; eight-wave ones, 64 rows only: one)
template <int RB, int KP, bool ZP, bool PARTIAL, typename OutT, bool XBF, bool BIAS>
__global__ __launch_bounds__(KP * 256, RB == 4 || KP == 2 ? 2 : 3) void w2a16_tiled_kernel(const W2A16Params p, const int steps_per_split, const int group_shift) {
    w2a16_tiled_body<RB, KP, ZP, PARTIAL, OutT, XBF, BIAS>(p, steps_per_split, group_shift);
}

template <int RB, int KP, bool ZP, bool XBF>
void launch_rb(const W2A16Params& p, bool out_bf16, dim3 grid, int sps, int shift, hipStream_t stream) {
    const dim3 block(KP * 256);
    if (p.split > 1) {   // (the sums' launch adds the bias)
        w2a16_tiled_kernel<RB, KP, ZP, true, OutF16, XBF, false><<<grid, block, 0, stream>>>(p, sps, shift);
    } else if (p.bias) {
        if (out_bf16) w2a16_tiled_kernel<RB, KP, ZP, false, OutBF16, XBF, true><<<grid, block, 0, stream>>>(p, sps, shift);
        else w2a16_tiled_kernel<RB, KP, ZP, false, OutF16, XBF, true><<<grid, block, 0, stream>>>(p, sps, shift);
    } else {
        if (out_bf16) w2a16_tiled_kernel<RB, KP, ZP, false, OutBF16, XBF, false><<<grid, block, 0, stream>>>(p, sps, shift);
        else w2a16_tiled_kernel<RB, KP, ZP, false, OutF16, XBF, false><<<grid, block, 0, stream>>>(p, sps, shift);
    }
}

}  // namespace

// K is a multiple of 128, an even number of steps, dealt out to the splits in pairs.  Where rounding up to whole pairs
// would leave the last splits empty (146 pairs in 16 splits: ten each, the sixteenth would start past the end) there are
// only as many as have work.
static int pairs_per_split(int steps, int split) { return (steps / 2 + split - 1) / split; }
static int splits_with_work(int steps, int split) {
    const int per = pairs_per_split(steps, split);
    return (steps / 2 + per - 1) / per;
}

// rb: row blocks of 32 per workgroup tile (2 or 4); halves: K parts inside a workgroup (1, or 2 with rb = 2).  With
// p.split > 1, one of splits_with_work, the partial sums go to p.ws.
hipError_t launch_w2a16_tiled(const W2A16Params& p, int rb, int halves, int gs, bool out_bf16, hipStream_t stream) {
    const int tiles_n = (p.strips + kStripsPerWg - 1) / kStripsPerWg, tiles_m = (p.M + rb * 32 - 1) / (rb * 32);
    const dim3 grid((unsigned)xcd_grid(tiles_n, tiles_m), (unsigned)p.split);
    const int sps = pairs_per_split(p.steps, p.split) * 2, shift = gs == 1 ? 0 : (gs == 2 ? 1 : 2);
    const bool zp = p.zp_r != nullptr;
#define SLIMK_W2A16_TILED(RBV, KPV)                                                              \
    do {                                                                                         \
        if (zp) {                                                                                \
            if (p.x_bf16) launch_rb<RBV, KPV, true, true>(p, out_bf16, grid, sps, shift, stream);   \
            else launch_rb<RBV, KPV, true, false>(p, out_bf16, grid, sps, shift, stream);        \
        } else {                                                                                 \
            if (p.x_bf16) launch_rb<RBV, KPV, false, true>(p, out_bf16, grid, sps, shift, stream);  \
            else launch_rb<RBV, KPV, false, false>(p, out_bf16, grid, sps, shift, stream);       \
        }                                                                                        \
    } while (0)
    if (rb == 4) SLIMK_W2A16_TILED(4, 1);
    else if (halves == 2) SLIMK_W2A16_TILED(2, 2);
    else SLIMK_W2A16_TILED(2, 1);
#undef SLIMK_W2A16_TILED
    return hipGetLastError();
}

// Which kernel, which tile height and how many K splits: the smallest predicted time.  The few-rows kernel runs 16 rows
// x one strip per workgroup, 0.02 us for each and 4096 reduction elements.  A 64-row workgroup of this kernel takes
// 0.65 us a step alone on a CU, two side by side 1.0, three and more 0.47 each (128-row ones 0.97, 1.7 and 0.85 each),
// an eight-wave one with two K halves 1.03 for a step of both and 2 us for their meeting: ahead while one round of them
// covers the problem, as it needs half the splits (300 x 4096 x 14336: three splits of two halves 51.6 us, six splits
// 55.0 on the same card; 768 x 5120 x 5120 unsplit 47.9, in two splits 56.2; in two rounds it loses, 400 x 2048 x 20480 in six
// 67.5 against 64.9).  A split writes and reads its partial sums at about 5 TB/s, plus the second launch.  Within 6 % of the measured times
// of fourteen shapes (64..1024 rows, 1024..28672 channels, K = 4096..14336) at one to eight splits: 300 x 4096 x 14336 80 -> 49 us,
// 128 x 14336 x 4096 39 -> 31, 1024 x 14336 x 4096 275 -> 115, 100 x 28672 x 8192 132 -> 74; 64 x 4096 x 4096 stays with
// the few-rows kernel (8.4 against 13 us).
W2A16Plan w2a16_plan(int M, int strips, int steps, int gs, int split) {
    W2A16Plan plan{0, split > 0 ? split : w2a16_few_rows_split(M, strips, steps, gs), 1};
    if (M <= 32) return plan;
    const float few_rows = 3.5f + 0.02f * (float)strips * (float)((M + 15) / 16) * (float)steps / 64.0f;
    const int tiles_n = (strips + kStripsPerWg - 1) / kStripsPerWg;
    const int cap = std::max(1, steps / (gs > 2 ? gs : 2) / 4);   // (what an explicit request is held to)
    float best = 0.93f * few_rows;   // (in hand: 120 x 13224 x 2560, predicted level, ran 26.9 -> 29.0 us)
    for (int rb = 2; rb <= 4; rb += 2) {
        const int tiles = tiles_n * ((M + rb * 32 - 1) / (rb * 32));
        for (int s : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (split > 0) s = split;
            if (s > cap && split <= 0) break;
            s = splits_with_work(steps, s);
            const int wgs = (tiles * s + 255) / 256;
            const float each = rb == 2 ? (wgs == 1 ? 0.65f : wgs == 2 ? 1.0f : 0.47f * (float)wgs)
                                       : (wgs == 1 ? 0.97f : wgs == 2 ? 1.7f : 0.85f * (float)wgs);
            const float sums = s > 1 ? 3.0f + (float)s * (float)M * (float)strips * (64.0f * 8.0f / 5e6f) : 0.0f;
            const float time = 2.5f + (float)((steps + s - 1) / s) * each + sums;
            const float halves = rb == 2 && tiles * s <= 256 ? 4.5f + (float)((steps / 2 + s - 1) / s) * 1.03f + sums : 1e30f;
            if (std::min(time, halves) < best) {
                best = std::min(time, halves);
                plan = {rb, s, halves < time ? 2 : 1};
            }
            if (split > 0) break;
        }
    }
    return plan;
}

}  // namespace w2a8
