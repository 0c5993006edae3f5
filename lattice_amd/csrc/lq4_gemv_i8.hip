// Decode GEMV for up to eight activation rows on the integer matrix cores:
//   y[b, n] = sum_k W[n, k] * x[b, k],  b < batch <= 8.
//
// Instruction.  v_mfma_i32_16x16x32_i8 multiplies a 16 x 32 by a 32 x 16 matrix of signed bytes into 16 x 16 32-bit
// sums.  K = 32 is exactly one Q4 block, so one instruction forms the integer dot products of one block of 16 weight
// rows with 16 activation columns, and the block's scale and bias are applied to its result in f32 afterwards.
//   B operand (32 x 16): the weights.  Lane l supplies column n = l % 16 (a weight row), k = 8 * (l / 16) .. + 7:
//     the eight nibbles of payload dword l / 16 of that row's block, spread into bytes by two masks.
//   A operand (16 x 32): the activations, staged as fixed point scaled per block (x = xs * q) and cut into signed byte
//     digits; either way they fill the operand.  Five to eight activation rows: two digits each (q = 256 hi + lo, xs = the
//     block's largest magnitude / 32639), operand row m = 2 b + digit.  Up to four rows ("wide"): four digits each (28 bits
//     and sign, xs a power of two), m = 4 b + digit.
//   D (16 x 16): lane l receives column n = l % 16, rows m = 4 (l / 16) .. + 3, i.e. for ITS weight row both digits
//     of activation rows 2 (l / 16) and 2 (l / 16) + 1 (wide: the four digits of row l / 16).  256 hi + lo is one
//     integer multiply-add, and
//       y[b, n] += (scale_n * xs_b) * (256 hi + lo) + bias_n * (xs_b * sum of the block's fixed-point x)
//     needs the block header of the lane's own row only, and every lane owns two outputs of its row from the first block to
//     the last.  The bias terms of four blocks are one v_mfma_f32_16x16x4_f32 (sums x biases, K = the four blocks): lane group
//     g reads the header of the g-th of the four blocks, its bias is that instruction's operand as it stands, and the scales
//     reach the other groups by three lane swaps.  The xs of a chunk's eight blocks lie one a lane, each row of sixteen lanes
//     holding those of its two activation rows, and are broadcast by the multiplication that uses them.
// Per instruction (16 rows x 32 weights = 320 bytes of weights): 13 vector operations, three to spread the nibbles among them,
// and 10 bytes a lane from LDS.  (With the header and both rows' xs and sums read for every block it was 23 operations and
// 32 bytes: 1.2 us a unit of 2.5 KB a wave, 0.4 of them the LDS.)
//
// Memory.  A unit is 16 rows x 8 blocks (2.5 KB): 160 pieces of 16 bytes, which the load unit puts into the wave's own part of
// LDS, up to four units ahead, so that a workgroup's share of the matrix is on its way while the activations are staged.
// (Each lane with blocks of its own, 160 contiguous bytes a row, was four times the address work, one unit ahead, and a
// rewrite into LDS.)  No barrier: what a wave multiplies it has brought itself.
//
// Work split.  One workgroup a CU takes tiles of 16 rows (tile = blockIdx, then += gridDim); its waves split K in chunks
// of 8 blocks and add their partial sums through LDS in wave order.  Each wave stages the activations of its own
// chunks only, once for all tiles of the workgroup; with one tile at a time it multiplies nothing else.
//
// Where the time goes (12288 x 2048 at eight rows, 8.7 -> 6.9 us; 2048 x 2048 5.5 -> 4.3): 0.6 us until the activations are asked
// for, 1 until they arrive, 0.8 to stage them, then 0.7 to 1 a round of units and 0.6 for the meeting; the weights have arrived
// by then.  A launch is a single pass through its code, so the order of the code (activations first) and its length count.
//
// LoRA.  The factor t = A . x of the adapter (of every view's adapter) is either in memory when the launch starts
// (lora.t / mv.t), or computed by the launch itself (lora.slots set): the first lora.rank workgroups are producers,
// one per row of A (the views' A stacked), each forming that row's dot products with the batch's activation rows
// and publishing them as {value, tag of the launch} words; the other workgroups pick them up into LDS when their first
// tile is multiplied, by which time the producers, who have nothing else to do, are done.  The launcher adds the
// producers only where CUs are idle beside the others (workgroups + producers <= CUs: a matrix of 2560 rows occupies 160; see plan_i8).  A value
// that has not arrived after the poll limit is computed by the wave that misses it, in the producers' order of
// summation (same bits), and counted in sync[2].
//
// Precision.  The weights enter exactly, the integer sums are exact.  Five to eight rows: an activation is rounded to a
// multiple of its block's largest magnitude / 32639 (step 3e-5 of the block maximum, against 5e-4 of the element for the
// f16 rounding of the 4x4x4 kernel and of the reference's tiled kernel, shaders/gemm_q4_tiled.metal:45-48).  Up to four rows
// it is cut off below 2^-27 .. 2^-28 of the block's largest magnitude: an f32 value of at least a 16th of that, and an f16
// value of at least a 2^-16th, enters exactly, so they track an f32 GEMV as the reference's gemm_q4 does.  (Two rows are
// served by pairs of f16 values elsewhere, 22 bits of each element.  Three digits, 22 bits and sign below the block's maximum,
// kept fewer of elements far below it.  2560 x 4096, rms of the activations' rounding alone, pairs / three digits / four: N(0,1)
// 4.4e-8 / 1.7e-7 / 2e-9, one channel in 64 a hundred times larger 4.3e-8 / 3.8e-7 / 1.6e-8; of the results against f64 6.5e-6 / 2.2e-7 /
// 1.5e-7 and 1.5e-5 / 4.1e-7 / 1.5e-7.  The fourth digit is free in the instruction; staging it costs 2048 x 2048 3.86 -> 3.98 us.)  Any finite f32 activation is in range (the scale is per block); a block whose largest
// magnitude is below 2^-100 counts as zero; an infinite or NaN activation makes the outputs of its row NaN.
#include "lq4_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace lq4 {

namespace {

typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int kBpw = 8;            // blocks per wave chunk
constexpr int kStageBytes = 16 * kBpw * kBlockBytes;  // a unit in LDS: 16 rows x 160 bytes, one behind the other
constexpr int kStageDwords = kStageBytes / 4, kRowDwords = kBpw * kBlockBytes / 4;
constexpr uint32_t kMaxStages = 4;  // units a wave has in flight
constexpr uint32_t kMeet = 4;       // rounds of tiles between two meetings of a workgroup's waves
constexpr size_t kLdsBytes = 160 * 1024;
constexpr int kXqBytes = 512;      // per block: [4 k groups][16 operand rows] x 8 bytes
constexpr int kXfBytes = 64;       // per block: [4 lane groups][xs of rows 2g, 2g + 1, then their sums] f32

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Memory -> LDS, 16 or 4 bytes a lane: lane l's bytes land at LDS byte address `lds` + 16 l (or + 4 l).  `base` and `lds` are
// wave-uniform.  By hand, like the loads of the activations: the compiler would make every LDS access wait for the former, and
// count the latter without them.  The compiler knows of no hazard either: a vector load may read a scalar register five wait
// states after a vector instruction wrote it (v_readlane, where the compiler keeps scalars in a vector register), so each brings
// its own.  m0 cannot be named as written: it is reserved, and set by the compiler in front of whatever of its own reads it.
// load16's register is filled only when a wait has passed: tests/test_isa.py looks for anything that touches it before.
__device__ __forceinline__ void dma16(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void dma4(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ f32x4 load16(const void* base, uint32_t off) {
    f32x4 r;
    asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %1, %2" : "=v"(r) : "v"(off), "s"(base) : "memory");
    return r;
}
// Until at most `units` units (three loads each, or more) are outstanding.
__device__ __forceinline__ void wait_units(uint32_t units) {
    if (units == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (units == 1) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
    else if (units == 2) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else if (units == 3) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p));
}

__device__ __forceinline__ float as_f32(uint32_t u) { return __builtin_bit_cast(float, u); }
__device__ __forceinline__ uint32_t as_u32(float f) { return __builtin_bit_cast(uint32_t, f); }

typedef float float4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float f16_lo(uint32_t h) { return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h & 0xFFFFu))); }
__device__ __forceinline__ float f16_hi(uint32_t h) { return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h >> 16))); }
// Lane N of the lane's row of sixteen.
template <int N>
__device__ __forceinline__ float of_row_lane(float v) {
    return as_f32(static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(as_u32(v)), 0x150 + N, 0xF, 0xF, true)));
}
// out[i] = v of row i of the wave's four rows of sixteen, in every row.
__device__ __forceinline__ void rows_apart(float v, float (&out)[4]) {
    const auto halves = __builtin_amdgcn_permlane32_swap(as_u32(v), as_u32(v), false, false);
    const auto lo = __builtin_amdgcn_permlane16_swap(halves[0], halves[0], false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(halves[1], halves[1], false, false);
    out[0] = as_f32(lo[0]);
    out[1] = as_f32(lo[1]);
    out[2] = as_f32(hi[0]);
    out[3] = as_f32(hi[1]);
}

// A lane's part of the dot product of row j of A with an activation row: eight values from 512 to 512, four such steps requested at
// once (one after the other, 2048 weights were four round trips to memory, and the producers the last
// to be ready: q, k and v of 2048 + 2 x 512 rows at eight rows, rank 16 on two of them, four layers 29.2 us, 22.9 so).
__device__ __forceinline__ float a_row_dot(const void* a, int a_is_f16, uint32_t j, uint32_t k, const float* __restrict__ x, int lane) {
    constexpr int kAhead = 4;
    float p = 0.0f;
    for (uint32_t k0 = 0; k0 < k; k0 += kAhead * 512) {
        f32x4 xv[kAhead][2], av[kAhead][2];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const uint32_t kk = k0 + i * 512 + lane * 8, at = kk < k ? kk : 0;
            const f32x4* xp = reinterpret_cast<const f32x4*>(x + at);
            xv[i][0] = xp[0];
            xv[i][1] = xp[1];
            const size_t ai = static_cast<size_t>(j) * k + at;
            const f32x4* ap = reinterpret_cast<const f32x4*>(a_is_f16 ? static_cast<const char*>(a) + ai * 2 : static_cast<const char*>(a) + ai * 4);
            av[i][0] = ap[0];
            av[i][1] = ap[a_is_f16 ? 0 : 1];
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (a_is_f16) {
                typedef _Float16 half8 __attribute__((ext_vector_type(8)));
                const half8 h = __builtin_bit_cast(half8, av[i][0]);
                av[i][0] = f32x4{static_cast<float>(h[0]), static_cast<float>(h[1]), static_cast<float>(h[2]), static_cast<float>(h[3])};
                av[i][1] = f32x4{static_cast<float>(h[4]), static_cast<float>(h[5]), static_cast<float>(h[6]), static_cast<float>(h[7])};
            }
            if (k0 + i * 512 + lane * 8 < k) {
#pragma unroll
                for (int e = 0; e < 8; ++e) p = fmaf(av[i][e / 4][e % 4], xv[i][e / 4][e % 4], p);
            }
        }
    }
    return p;
}

// WIDE: up to four activation rows at four digits; else up to eight at two.
// CW x TW waves: CW waves split the chunks of one tile, TW tiles are worked on side by side.
// MULTI: the rows are those of several matrices stacked one under the other (MultiViews: view v = rows [begin[v],
// begin[v + 1]), every view a whole number of 16-row tiles), each with its own output [batch, rows of the view] and its
// own LoRA factors; w, y, y_stride and lora are then unused.
// LORA: with adapters (on any view).  Four layers of eight rows, which have none, took 142 us with this code in their way, 134
// without.
template <int CW, int TW, bool WIDE, bool MULTI, bool LORA>
__global__ __launch_bounds__(64 * CW * TW) void gemv_q4_i8(const uint8_t* __restrict__ w, uint32_t n, uint32_t k,
                                                           const float* __restrict__ x, uint32_t x_stride,
                                                           uint32_t batch, float* __restrict__ y, uint32_t y_stride,
                                                           uint32_t stages, LoraEpilogue lora, MultiViews mv) {
    constexpr int WAVES = CW * TW;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // ---- producers of the LoRA factors (see the head of the file): workgroup p < prod owns stacked row p of A ----
    const uint32_t prod = LORA && lora.slots ? lora.rank : 0;  // (several views: lora.rank is the ranks of all views together)
    auto a_row_of = [&](uint32_t p, const void*& a, int& a_is_f16, uint32_t& j) {
        a = lora.a;
        a_is_f16 = lora.b_is_f16;
        j = p;
        if constexpr (MULTI) {
            uint32_t v = 0;
#pragma unroll
            for (int i = 1; i < kMaxViews; ++i) v += (static_cast<uint32_t>(i) < mv.count && p >= mv.t_off[i]) ? 1u : 0u;
            a = mv.a[v];
            a_is_f16 = mv.b_is_f16[v];
            j = p - mv.t_off[v];
        }
    };
    if (blockIdx.x < prod) {
        const void* a;
        int a_is_f16;
        uint32_t j;
        a_row_of(blockIdx.x, a, a_is_f16, j);
        // a wave per activation row: no barrier, nothing through LDS, one cross-lane sum before the word goes out
        for (uint32_t b = wave; b < batch; b += WAVES) {
            const float total = wave_sum(a_row_dot(a, a_is_f16, j, k, x + static_cast<size_t>(b) * x_stride, lane));
            const unsigned long long word = (static_cast<unsigned long long>(launch_tag()) << 32) | as_u32(total);
            if (lane == 0) __hip_atomic_store(&lora.slots[blockIdx.x * 8 + b], word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    const uint32_t wg = blockIdx.x - prod, n_wg = gridDim.x - prod;  // this workgroup among those that stream weights
    const uint32_t tw = TW == 1 ? 0 : wave / CW, cw = TW == 1 ? wave : wave % CW;
    const uint32_t nb = k / kBlockWeights;
    const size_t row_bytes = static_cast<size_t>(nb) * kBlockBytes;
    // LDS: [whole chunks] activation digits | [whole chunks] activation scales and sums | [WAVES][stages] units |
    // [kMeet][WAVES][64][2] partial sums | [8][64] LoRA factors
    const uint32_t chunks = (nb + kBpw - 1) / kBpw;
    uint8_t* const xq = smem;
    uint8_t* const xf = xq + chunks * (kBpw * kXqBytes);
    uint32_t* const ring = reinterpret_cast<uint32_t*>(xf + chunks * (kBpw * kXfBytes)) + wave * stages * kStageDwords;
    float* const part = reinterpret_cast<float*>(xf + chunks * (kBpw * kXfBytes)) + WAVES * stages * kStageDwords;
    float* const t_lds = part + kMeet * WAVES * 64 * 2;  // [8 activation rows][kMaxLoraRank]: the factors picked up from the producers

    const uint32_t my_chunks = cw < chunks ? (chunks - cw + CW - 1) / CW : 0;  // chunk c * CW + cw

    // ---- stage the activations: the waves of column cw (one: TW = 1) its chunks ----
    // A lane's task: eight values of one activation row, a k group of a block.  64 lanes = four k groups x kRows rows x kTaskBlocks
    // blocks, so a chunk is kTasks of them, of which wave tw takes tw, tw + TW, ..
    constexpr uint32_t kRows = WIDE ? 4 : 8;      // activation rows the operand holds
    constexpr int kTaskBlocks = 16 / kRows, kTasks = kBpw / kTaskBlocks, kMyTasks = kTasks > TW ? kTasks / TW : 1;
    // q = rint(x / xs) with xs = block maximum / kQScale: |q| stays below kQScale + 2 whatever the rounding of the
    // reciprocal, both digits within -128..127.  (Wide: below.)
    constexpr float kQScale = 32639.0f;
    const uint32_t kg = lane & 3, xb = (static_cast<uint32_t>(lane) >> 2) & (kRows - 1), xblk = static_cast<uint32_t>(lane) / (4 * kRows);
    auto task_block = [&](uint32_t c, int i) { return (c * CW + cw) * kBpw + (tw + i * TW) * kTaskBlocks + xblk; };
    // rows and blocks that do not exist re-read an existing one
    const uint32_t x_lane = ((xb < batch ? xb : 0) * x_stride + kg * 8) * 4;
    auto x_off = [&](uint32_t c, int i) {
        const uint32_t blk = task_block(c, i);
        return x_lane + (blk < nb ? blk : nb - 1) * (kBlockWeights * 4);
    };
    auto quad_max = [](uint32_t v) {
        v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xB1, 0xF, 0xF, false)));
        return max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4E, 0xF, 0xF, false)));
    };
    auto quad_sum = [](auto v) {
        auto of = [](auto w, auto ctrl) {
            return __builtin_bit_cast(decltype(w), __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, w), decltype(ctrl)::value, 0xF, 0xF, false));
        };
        v += of(v, std::integral_constant<int, 0xB1>{});
        return v + of(v, std::integral_constant<int, 0x4E>{});
    };
    auto stage_chunk = [&](uint32_t c, auto xv_of) {
        float my_xs = 0.0f, my_sum = 0.0f;  // k group i's lane: of the wave's i-th task
        uint8_t* const dst = xq + task_block(c, 0) * kXqBytes + kg * 128 + (WIDE ? 4 : 2) * xb * 8;
#pragma unroll
        for (int i = 0; i < kMyTasks; ++i) {
            f32x4 xa, xc;
            xv_of(i, xa, xc);
            const float v[8] = {xa.x, xa.y, xa.z, xa.w, xc.x, xc.y, xc.z, xc.w};
            // largest magnitude as a bit pattern: infinities and NaNs come out on top of every finite value
            uint32_t abits = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) abits = max(abits, as_u32(v[j]) & 0x7FFFFFFFu);
            abits = quad_max(abits);
            const bool none = abits < 0x0D800000u || task_block(c, i) >= nb;  // below 2^-100, or past the end of the row: counts for nothing
            constexpr int kDigits = WIDE ? 4 : 2;
            uint32_t dg[kDigits][2];
            float xs, sum;  // sum: of the block's q, in units of xs
            if constexpr (WIDE) {
                // q = x * 2^(154 - e), truncated, with e = the maximum's exponent field (27 and more): |q| < 2^28, so that eight
                // of them add up in 32 bits.  xs is what 2^16 of q stand for, so that it is no denormal.
                const uint32_t e = abits >> 23;
                const float inv = none ? 0.0f : as_f32((281u - e) << 23);
                xs = none ? 0.0f : abits >= 0x7F800000u ? as_f32(0x7FC00000u) : as_f32((e - 11u) << 23);
                int lane_sum = 0;
                // Byte i of q + 0x80808080, less 128, is digit i (-128..127) of q.  u: those of element {0, 2, 4, 6}[p] (h = 0) or
                // {1, 3, 5, 7}[p], as the two masks lay out a payload dword's nibbles; a digit's four go into one dword.
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t u[4];
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const int q = static_cast<int>(v[2 * p + h] * inv);
                        lane_sum += q;
                        u[p] = (static_cast<uint32_t>(q) + 0x80808080u) ^ 0x80808080u;
                    }
                    const uint32_t a0 = __builtin_amdgcn_perm(u[1], u[0], 0x05010400u), a1 = __builtin_amdgcn_perm(u[3], u[2], 0x05010400u);
                    const uint32_t b0 = __builtin_amdgcn_perm(u[1], u[0], 0x07030602u), b1 = __builtin_amdgcn_perm(u[3], u[2], 0x07030602u);
                    dg[0][h] = __builtin_amdgcn_perm(a1, a0, 0x05040100u);
                    dg[1][h] = __builtin_amdgcn_perm(a1, a0, 0x07060302u);
                    dg[2][h] = __builtin_amdgcn_perm(b1, b0, 0x05040100u);
                    dg[3][h] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
                }
                sum = quad_sum(static_cast<float>(lane_sum) * (1.0f / 65536.0f));
            } else {
                const float xs_any = as_f32(abits) * (1.0f / kQScale), inv_any = __builtin_amdgcn_rcpf(xs_any);
                const float inv = none ? 0.0f : inv_any;
                // (an infinite or NaN activation: the row's outputs become NaN)
                xs = none ? 0.0f : abits >= 0x7F800000u ? as_f32(0x7FC00000u) : xs_any;
                // 1.5 * 2^23 + q as a float has q in its low 23 bits in two's complement: bits = 0x4B400000 + q
                uint32_t qb[8], sum_bits = 0;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    qb[j] = as_u32(fmaf(v[j], inv, 12582912.0f));
                    sum_bits += qb[j];
                }
                sum = static_cast<float>(quad_sum(static_cast<int>(sum_bits - 8u * 0x4B400000u)));
                // Digits -128..127 from the lowest up: byte 0 of q, byte 1 of q + 0x80.  Byte p of an operand word pair = element
                // {0, 2, 4, 6, 1, 3, 5, 7}[p] of the k group: the order in which the two masks lay out a payload dword's nibbles.
                typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
                const u16x2 up = {0x80, 0x80};
#pragma unroll
                for (int h = 0; h < 2; ++h) {  // (two 16-bit q side by side)
                    const uint32_t p0 = __builtin_amdgcn_perm(qb[2 + h], qb[h], 0x05040100u), p1 = __builtin_amdgcn_perm(qb[6 + h], qb[4 + h], 0x05040100u);
                    const uint32_t h0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, p0) + up);
                    const uint32_t h1 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, p1) + up);
                    dg[0][h] = __builtin_amdgcn_perm(p1, p0, 0x06040200u);
                    dg[1][h] = __builtin_amdgcn_perm(h1, h0, 0x07050301u);
                }
            }
            my_xs = kg == static_cast<uint32_t>(i) ? xs : my_xs;
            my_sum = kg == static_cast<uint32_t>(i) ? sum : my_sum;
            // operand row of (b, digit): the highest digit first
            uint4* const to = reinterpret_cast<uint4*>(dst + i * (TW * kTaskBlocks * kXqBytes));
#pragma unroll
            for (int t = 0; t < kDigits; t += 2) to[t / 2] = make_uint4(dg[kDigits - 1 - t][0], dg[kDigits - 1 - t][1], dg[kDigits - 2 - t][0], dg[kDigits - 2 - t][1]);
        }
        if (kg < static_cast<uint32_t>(kMyTasks)) {
            // of a chunk: [row pair g][2 block + row of the pair] xs (wide: [row][2 block]), then [block][row] xs * sum
            const uint32_t blk = task_block(c, kg), j = blk % kBpw;
            float* f = reinterpret_cast<float*>(xf + (blk - j) * kXfBytes);
            f[WIDE ? 16 * xb + 2 * j : 16 * (xb >> 1) + 2 * j + (xb & 1)] = my_xs;
            f[64 + 8 * j + xb] = my_xs * my_sum;
        }
    };

    // The values of a wave's first chunks are requested before any weight (loads are answered in the order a CU
    // issued them: behind the weights the staging would wait for these), all at once.
    const bool stages_rows = tw < kTasks && my_chunks;  // uniform (more tiles side by side than tasks, or more waves than chunks: not all)
    constexpr int kAhead = TW < 4 ? 2 * TW : 8;  // chunks
    // (out of the way of the usual case, whose code then lies together: one chunk a wave with one tile at a time)
    auto has_chunk = [&](int c) { return c == 0 || (TW == 1 ? __builtin_expect(static_cast<uint32_t>(c) < my_chunks, 0) : static_cast<uint32_t>(c) < my_chunks); };
    f32x4 xv[kAhead][kMyTasks][2];
#pragma unroll
    for (int c = 0; c < kAhead; ++c) {
        if (has_chunk(c)) {  // uniform
#pragma unroll
            for (int i = 0; i < kMyTasks; ++i) {
                const uint32_t at = x_off(c, i);
                xv[c][i][0] = load16(x, at);
                xv[c][i][1] = load16(x, at + 16);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);  // nothing below is scheduled above these loads

    const uint32_t n_tiles = (n + 15) / 16;
    // tiles of the workgroup: blockIdx + j * gridDim; of this wave: j = tw, tw + TW, ...; a round = TW tiles
    const uint32_t wg_tiles = wg < n_tiles ? (n_tiles - wg + n_wg - 1) / n_wg : 0;
    const uint32_t rounds = (wg_tiles + TW - 1) / TW;
    const uint32_t my_tiles = tw < wg_tiles ? (wg_tiles - tw + TW - 1) / TW : 0;
    const uint32_t units = my_tiles * my_chunks;  // unit u = (my tile u / my_chunks, my chunk u % my_chunks)
    auto first_row = [&](uint32_t t) { return (wg + (t * TW + tw) * n_wg) * 16; };
    // MULTI: the view that holds stacked row `row` (uniform: called with a tile's first row)
    auto view_of = [&](uint32_t row) {
        uint32_t v = 0;
        if constexpr (MULTI) {
#pragma unroll
            for (int i = 1; i < kMaxViews; ++i) v += (static_cast<uint32_t>(i) < mv.count && row >= mv.begin[i]) ? 1u : 0u;
        }
        return v;
    };

    auto r_of = [](int l) { return static_cast<uint32_t>(l & 15); };  // the weight row of the tile a lane's outputs belong to
    // A unit is 160 pieces of 16 bytes, ten a row: lane l brings pieces l, l + 64 and (half the lanes) l + 128.
    const uint32_t row32 = static_cast<uint32_t>(row_bytes);
    auto piece_off = [&](uint32_t i) { return i / 10 * row32 + i % 10 * 16; };
    const uint32_t off0 = piece_off(lane), off1 = piece_off(lane + 64), off2 = piece_off((lane & 31) + 128);
    auto load_unit = [&](uint32_t u, uint32_t stage) {
        const uint32_t t = u / my_chunks, c = u - t * my_chunks;
        const uint32_t row0 = first_row(t);
        const uint8_t* wv = w;
        uint32_t row_base = 0, row_end = n;
        if constexpr (MULTI) {
            const uint32_t v = view_of(row0);
            wv = mv.w[v];
            row_base = mv.begin[v];
            row_end = mv.begin[v + 1];
        }
        const uint32_t at = (c * CW + cw) * (kBpw * kBlockBytes);  // of the chunk in a row
        const uint8_t* const base = wv + (row0 - row_base) * row_bytes + at;
        const uint32_t to = lds_address(ring + stage * kStageDwords);
        const uint32_t rows = row_end - row0;  // of the tile and behind it
        if (__builtin_expect(rows >= 16 && rows * row_bytes >= 15 * row_bytes + at + kBpw * kBlockBytes, 1)) {  // uniform
            dma16(to, base, off0);
            dma16(to + 1024, base, off1);
            if (lane < 32) dma16(to + 2048, base, off2);
        } else {
            // the matrix ends inside the unit: dword by dword, rows and bytes past the end read the last ones
            const uint32_t last = rows * row32 - at - 4;
#pragma unroll 1
            for (int i = 0; i < kStageDwords / 64; ++i) {
                const uint32_t e = i * 64 + lane, r = e / kRowDwords, off = (r < rows ? r : rows - 1) * row32 + e % kRowDwords * 4;
                dma4(to + i * 256, base, off < last ? off : last);
            }
        }
    };

    // The LoRA factor B of the wave's first tile (its first sixteen ranks, f16 in eights) is requested before
    // anything else and used in that tile's epilogue: requested there, its whole latency stood between the last
    // matrix instruction and the store, and a workgroup of these launches has one tile or two.
    struct alignas(16) H8 { _Float16 v[8]; };
    f32x4 b_pre[2];
    bool use_pre = false;
    if (LORA && cw == 0 && my_tiles) {  // uniform
        const uint32_t row0 = first_row(0);
        const void* bq = lora.b;
        uint32_t rank = lora.rank, row_end = n, row_base = 0;
        int b16 = lora.b_is_f16;
        if constexpr (MULTI) {
            const uint32_t v = view_of(row0);
            bq = mv.b[v];
            rank = mv.rank[v];
            b16 = mv.b_is_f16[v];
            row_end = mv.begin[v + 1];
            row_base = mv.begin[v];
        }
        if (rank && b16 && rank % 8 == 0) {
            use_pre = true;
            const uint32_t row = (row0 + r_of(lane) < row_end ? row0 + r_of(lane) : row_end - 1) - row_base;
            b_pre[0] = load16(bq, row * rank * 2);
            b_pre[1] = load16(bq, row * rank * 2 + (rank >= 16 ? 16 : 0));
        }
    }
    const uint32_t first_units = units < stages ? units : stages;
    for (uint32_t i = 0; i < first_units; ++i) load_unit(i, i);
    __builtin_amdgcn_sched_barrier(0);  // nothing below is scheduled above these loads
    wait_units(first_units);
#pragma unroll
    for (int c = 0; c < kAhead; ++c)
#pragma unroll
        for (int i = 0; i < kMyTasks; ++i) asm volatile("" : "+v"(xv[c][i][0]), "+v"(xv[c][i][1]));
    if constexpr (LORA) asm volatile("" : "+v"(b_pre[0]), "+v"(b_pre[1]));
    if (stages_rows) {
#pragma unroll
        for (int c = 0; c < kAhead; ++c) {
            if (has_chunk(c)) stage_chunk(c, [&](int i, f32x4& a, f32x4& b) {
                a = xv[c][i][0];
                b = xv[c][i][1];
            });
        }
#pragma unroll 1
        for (uint32_t c = kAhead; c < my_chunks; ++c)  // (behind the weights)
            stage_chunk(c, [&](int i, f32x4& a, f32x4& b) {
                const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const uint8_t*>(x) + x_off(c, i));
                a = p[0];
                b = p[1];
            });
    }
    if constexpr (TW > 1) __syncthreads();
    else asm volatile("" ::: "memory");  // (one tile at a time: a wave multiplies what it staged itself)
    // The LoRA factors of the producers: item i = (stacked row of A i / 8, activation row i % 8), 64 items a wave.  Picked up once, when
    // the wave's first tile is multiplied, in front of the barrier of its partial sums, behind which the factors are read: the
    // producers need some 2.5 us, and the product has begun after 3 (picked up before it, the four layers of a_row_dot's comment
    // took 31.5 us, 28.4 behind it).
    auto pick_up = [&] {
        const uint32_t tag = launch_tag();
        const unsigned long long none = static_cast<unsigned long long>(tag) << 32;  // lanes without an item: as if published
        for (uint32_t i0 = wave * 64; i0 < prod * 8; i0 += 64 * WAVES) {  // uniform
            const uint32_t i = i0 + lane;
            const bool mine = i < prod * 8 && (i & 7) < batch;
            // first through the caches (the usual case: the producers are done, one fetch per XCD), then past them
            unsigned long long v = none;
            if (lora.spin_limit) {
                if (mine) v = *static_cast<const volatile unsigned long long*>(&lora.slots[i]);
                for (uint32_t spin = 0; spin < lora.spin_limit && !__all(static_cast<uint32_t>(v >> 32) == tag); ++spin) {
                    __builtin_amdgcn_s_sleep(4);
                    if (mine) v = __hip_atomic_load(&lora.slots[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            } else if (mine) {
                v = 0;  // (no polling at all: every item is computed here)
            }
            float val = as_f32(static_cast<uint32_t>(v));
            uint64_t missing = __ballot(static_cast<uint32_t>(v >> 32) != tag);
            while (missing) {  // uniform: the wave computes the item itself, in the producers' order of summation
                const uint32_t fl = static_cast<uint32_t>(__builtin_ctzll(missing));
                missing &= missing - 1;
                const uint32_t item = i0 + fl;
                const void* a;
                int a_is_f16;
                uint32_t j;
                a_row_of(item >> 3, a, a_is_f16, j);
                const float* xr = x + static_cast<size_t>(item & 7) * x_stride;
                const float total = wave_sum(a_row_dot(a, a_is_f16, j, k, xr, lane));
                if (static_cast<uint32_t>(lane) == fl) val = total;
                if (lane == 0) __hip_atomic_fetch_add(&lora.sync[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (i < prod * 8) t_lds[(i & 7) * kMaxLoraRank + (i >> 3)] = mine ? val : 0.0f;
        }
    };

    // ---- the product ----
    const uint32_t r = lane & 15, g = lane >> 4;  // operand mapping: weight row r of the tile, k group / row pair g
    float acc0 = 0.0f, acc1 = 0.0f;
    auto multiply = [&](uint32_t u, uint32_t c, uint32_t stage) {
        const uint32_t behind = units - 1 - u;
        wait_units(behind < stages - 1 ? behind : stages - 1);
        const uint32_t blk0 = (c * CW + cw) * kBpw;
        uint32_t* const unit = ring + stage * kStageDwords;
        if (__builtin_expect(blk0 + kBpw > nb, 0)) {  // uniform: blocks past the end of the row; their headers become zero (and their activations are)
            for (uint32_t i = lane; i < 16 * kBpw; i += 64)
                if (blk0 + i % kBpw >= nb) unit[i / kBpw * kRowDwords + i % kBpw * 5] = 0;
        }
        const uint32_t *head = unit + r * kRowDwords, *data = head + 1 + g;
        const uint8_t* xqp = xq + blk0 * kXqBytes + lane * 8;
        const float* xfp = reinterpret_cast<const float*>(xf + blk0 * kXfBytes);
        const float xs = xfp[lane];
        // four blocks at a time, straight-line: their LDS reads, then their four matrix instructions back to back,
        // then their results
        auto four = [&](auto j0c) {
            constexpr int j0 = decltype(j0c)::value;
            // lane group g: the header of block j0 + g, and of that block the sums of activation row b(r): operands of the matrix
            // instruction that adds up bias * sum over the four blocks; its results land as those of the integer ones do
            const uint32_t hd = head[5 * (j0 + g)];
            const float sx = xfp[64 + 8 * (j0 + g) + (WIDE ? r >> 2 : 2 * (r >> 2) + (r & 1))];
            uint32_t qd[4];
            long aop[4];
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                qd[jj] = data[5 * (j0 + jj)];
                aop[jj] = *reinterpret_cast<const long*>(xqp + (j0 + jj) * kXqBytes);
            }
            float sc[4];
            rows_apart(f16_lo(hd), sc);
            // The products are added to the bias terms of their own four blocks, with which they cancel to a large part (two sums
            // that meet at the end lose what the result would have kept: 2048 x 2048 at three rows, rms error 2.9e-7).
            float4v acc = __builtin_amdgcn_mfma_f32_16x16x4f32(sx, f16_hi(hd), float4v{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            int4v d[4];
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) {
                const uint32_t even = qd[jj] & 0x0F0F0F0Fu, odd = (qd[jj] >> 4) & 0x0F0F0F0Fu;
                const long bop = static_cast<long>((static_cast<uint64_t>(odd) << 32) | even);
                const int4v zero = {0, 0, 0, 0};
                d[jj] = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop[jj], bop, zero, 0, 0, 0);
            }
            auto one = [&](auto jc) {
                constexpr int jj = decltype(jc)::value, j = j0 + jj;
                const float s0 = of_row_lane<2 * j>(xs) * sc[jj];
                if constexpr (WIDE) {
                    // the sums of the two digits above and of the two below are exact in f32: one rounding in their add
                    acc.x = fmaf(s0, fmaf(static_cast<float>(d[jj].z * 256 + d[jj].w), 1.0f / 65536.0f, static_cast<float>(d[jj].x * 256 + d[jj].y)), acc.x);
                } else {
                    const float s1 = of_row_lane<2 * j + 1>(xs) * sc[jj];
                    acc.x = fmaf(s0, static_cast<float>(d[jj].x * 256 + d[jj].y), acc.x);
                    acc.y = fmaf(s1, static_cast<float>(d[jj].z * 256 + d[jj].w), acc.y);
                }
            };
            one(std::integral_constant<int, 0>{});
            one(std::integral_constant<int, 1>{});
            one(std::integral_constant<int, 2>{});
            one(std::integral_constant<int, 3>{});
            acc0 += acc.x;
            acc1 += acc.y;
        };
        four(std::integral_constant<int, 0>{});
        four(std::integral_constant<int, 4>{});
        asm volatile("" : "+v"(acc0), "+v"(acc1));  // (sunk below the branch, the broadcasts are instructions of their own)
        if (u + stages < units) {  // uniform; the unit's LDS reads are done
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            load_unit(u + stages, stage);
        }
    };
    // The sums of round t's tile and what belongs to them, to memory.
    auto finish = [&](uint32_t t) {
        const uint32_t row = first_row(t) + r;
        const float* const mine = part + (t % kMeet) * (WAVES * 64 * 2) + (tw * CW * 64 + lane) * 2;
        float acc0 = 0.0f, acc1 = 0.0f;
#pragma unroll
        for (int v = 0; v < CW; ++v) {
            const float2 pv = *reinterpret_cast<const float2*>(mine + v * (64 * 2));
            acc0 += pv.x;
            acc1 += pv.y;
        }
        {
            if (row < n) {
                const uint32_t b0 = WIDE ? g : 2 * g, b1 = WIDE ? batch : 2 * g + 1;  // (wide: one row a lane)
                // this row's adapter and output: the launch's, or (several views) those of the tile's view
                LoraEpilogue lo = lora;
                float* yv = y;
                uint32_t ys = y_stride, lrow = row;
                if constexpr (MULTI) {
                    const uint32_t v = view_of(first_row(t));
                    lo.b = mv.b[v];
                    lo.t = mv.t[v];
                    lo.rank = mv.rank[v];
                    lo.b_is_f16 = mv.b_is_f16[v];
                    lo.scale = mv.scale[v];
                    yv = mv.y[v];
                    ys = mv.begin[v + 1] - mv.begin[v];
                    lrow = row - mv.begin[v];
                }
                // t of activation rows b0 and b1, `t0[i]` = factor i: from memory, or (producers) from LDS
                auto delta = [&](auto* t0, auto* t1) {
                    float l0 = 0.0f, l1 = 0.0f;
                    if (lo.b_is_f16 && lo.rank % 8 == 0) {
                        // eight factors a step: one 16-byte load of B[row, i..i+7] (the first two steps of the wave's
                        // first tile: requested at the start of the kernel) and four of t
                        const _Float16* brow = static_cast<const _Float16*>(lo.b) + static_cast<size_t>(lrow) * lo.rank;
                        auto eight = [&](const H8& bq, uint32_t i) {
                            const float4 ta = *reinterpret_cast<const float4*>(t0 + i), tb = *reinterpret_cast<const float4*>(t0 + i + 4);
                            const float4 ua = *reinterpret_cast<const float4*>(t1 + i), ub = *reinterpret_cast<const float4*>(t1 + i + 4);
                            const float tv[8] = {ta.x, ta.y, ta.z, ta.w, tb.x, tb.y, tb.z, tb.w};
                            const float uv[8] = {ua.x, ua.y, ua.z, ua.w, ub.x, ub.y, ub.z, ub.w};
#pragma unroll
                            for (int jj = 0; jj < 8; ++jj) {
                                const float bv = static_cast<float>(bq.v[jj]);
                                l0 = fmaf(bv, tv[jj], l0);
                                l1 = fmaf(bv, uv[jj], l1);
                            }
                        };
                        uint32_t i = 0;
                        if (use_pre && t == 0) {  // uniform
                            eight(__builtin_bit_cast(H8, b_pre[0]), 0);
                            if (lo.rank >= 16) eight(__builtin_bit_cast(H8, b_pre[1]), 8);
                            i = lo.rank >= 16 ? 16 : 8;
                        }
                        for (; i < lo.rank; i += 8) eight(*reinterpret_cast<const H8*>(brow + i), i);
                    } else {
                        for (uint32_t i = 0; i < lo.rank; ++i) {
                            const size_t bi = static_cast<size_t>(lrow) * lo.rank + i;
                            const float bv = lo.b_is_f16 ? static_cast<float>(static_cast<const _Float16*>(lo.b)[bi])
                                                         : static_cast<const float*>(lo.b)[bi];
                            l0 = fmaf(bv, t0[i], l0);
                            l1 = fmaf(bv, t1[i], l1);
                        }
                    }
                    acc0 = fmaf(lo.scale, l0, acc0);
                    acc1 = fmaf(lo.scale, l1, acc1);
                };
                if (LORA && lo.rank) {
                    const uint32_t c0 = b0 < batch ? b0 : 0, c1 = b1 < batch ? b1 : 0;
                    if (prod) {
                        uint32_t off = 0;
                        if constexpr (MULTI) off = mv.t_off[view_of(first_row(t))];
                        delta(t_lds + c0 * kMaxLoraRank + off, t_lds + c1 * kMaxLoraRank + off);
                    } else {
                        delta(lo.t + c0 * lo.rank, lo.t + c1 * lo.rank);
                    }
                }
                if (b0 < batch) yv[static_cast<size_t>(b0) * ys + lrow] = acc0;
                if (b1 < batch) yv[static_cast<size_t>(b1) * ys + lrow] = acc1;
            }
        }
    };

    // The waves meet every kMeet rounds (once, where a workgroup has that many tiles or fewer): in between each goes at its own
    // pace, so that one reads LDS while another computes.  (With a meeting a round the four layers of a_row_dot's comment took 28.4 us, 24.9 so.)
    // (with adapters: what finish and pick_up load is waited for at their end, in a form that the compiler sees.  Left to it, it assumes
    // such loads pending on the registers that every unit of the product uses, and empties the ring in front of each: with rank 16
    // 10240 x 4096 at eight rows 15.5 -> 14.2 us, 12288 x 4096 16.4 -> 14.7, 5120 x 5120 12.1 -> 11.1.)
    // (Not behind the last tiles, where only their stores are left: 2048 x 2048 at four rows 4.66 -> 4.58, at eight 5.03 -> 4.98.)
    auto settle = [] {
        if constexpr (LORA) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    };
    for (uint32_t t = 0, u = 0, stage = 0; t < rounds; ++t) {
        if (t < my_tiles) {  // uniform in the wave
            acc0 = 0.0f;
            acc1 = 0.0f;
            for (uint32_t c = 0; c < my_chunks; ++c, ++u) {
                multiply(u, c, stage);
                stage = stage + 1 == stages ? 0 : stage + 1;
            }
            *reinterpret_cast<float2*>(part + ((t % kMeet) * WAVES + wave) * (64 * 2) + lane * 2) = make_float2(acc0, acc1);
        }
        if (prod && t == 0) {  // uniform
            pick_up();
            settle();
        }
        if ((t + 1) % kMeet == 0 || t + 1 == rounds) {
            __syncthreads();
            for (uint32_t q = t - t % kMeet + cw; q <= t && q < my_tiles; q += CW) finish(q);
            if (t + 1 < rounds) {
                settle();
                __syncthreads();
            }
        }
    }
}

struct I8Plan {
    uint32_t cw, tw, grid, stages;
    size_t lds;
};

}  // namespace

// At least two 16-row tiles per CU, of rows of up to 2816 weights.
bool gemv_i8_many_short_rows(uint32_t n, uint32_t k, uint32_t cu_count) {
    return (n + 15) / 16 >= 2 * cu_count && k >= 1024 && k <= 2816;
}

namespace {

struct I8Split {
    uint32_t cw, tw, steps;  // columns of chunks, tiles side by side, units a wave is left with
};
uint32_t steps_i8(uint32_t n_tiles, uint32_t chunks, uint32_t cu_count, uint32_t cw, uint32_t tw) {
    return ((n_tiles + tw - 1) / tw + cu_count - 1) / cu_count * ((chunks + cw - 1) / cw);
}
I8Split split_i8(uint32_t n_tiles, uint32_t chunks, uint32_t cu_count, bool wide) {
    // Up to a tile a CU: as many waves as split its chunks, up to eight.  With more, eight waves as 8, 4, 2 or 1 columns of chunks
    // beside 1, 2, 4 or 8 tiles, whichever leaves a wave the fewest units (12288 x 2560 is 5 as 2 x 4, 6 else; 8 x 1 has
    // the shorter staging, so it is taken where it is no worse).  One column only of short rows, which four of the waves stage (up to four
    // activation rows: two): us as 2 x 4 / 1 x 8 at five rows 32768 x 1280 11.3 / 10.0, x 1792 13.1 / 12.0, x 2304 15.8 / 15.2, x 2816 17.7 / 18.3,
    // at three rows 10.1 / 9.7, 12.5 / 12.1, 14.4 / 15.2.
    I8Split best{chunks >= 8 ? 8u : chunks >= 4 ? 4u : chunks >= 2 ? 2u : 1u, 1, 0};
    auto steps = [&](uint32_t cw, uint32_t tw) { return steps_i8(n_tiles, chunks, cu_count, cw, tw); };
    best.steps = steps(best.cw, best.tw);
    if (n_tiles <= cu_count || chunks < 2) return best;
    best.steps = ~0u;
    for (uint32_t cw = 8; cw >= (chunks <= (wide ? 7u : 9u) ? 1u : 2u); cw /= 2)
        if (cw < 2 * chunks && steps(cw, 8 / cw) < best.steps) best = I8Split{cw, 8 / cw, steps(cw, 8 / cw)};
    return best;
}

// producers: workgroups of the launch that compute LoRA factors.  Where they find no idle CU beside the usual split, but do beside
// more tiles in a workgroup at up to two steps more, that one: the launch for the factors which they save takes three (rank 16, eight
// rows, us with that launch / so / plain: 5120 x 4096 12.5 / 10.2 / 9.0, 4096 x 2048 7.7 / 6.4 / 4.5, 12288 x 2048 10.8 / 9.9 / 7.2, 4096 x 2560 8.3 / 7.9 /
// 5.3, 4096 x 4096 10.3 / 9.7 / 7.0).  Up to four rows from a tile for every CU on (rank 16, three and four rows, with that launch / so: 5120 x
// 4096 10.6 / 8.6, 4096 x 2048 6.9 / 5.9, 12288 x 2048 9.5 / 8.5); 4000 x 2048, 7.0 / 5.9, keeps the launch, as tests/test_gpu_parity.py has it.
bool plan_i8(uint32_t n, uint32_t k, uint32_t batch, uint32_t cu_count, I8Plan* out, uint32_t producers = 0) {
    if (k == 0 || k % kBlockWeights || n == 0 || batch == 0 || batch > 8) return false;
    const uint32_t nb = k / kBlockWeights;
    const uint32_t chunks = (nb + kBpw - 1) / kBpw;
    const uint32_t n_tiles = (n + 15) / 16;
    I8Plan p;
    I8Split split = split_i8(n_tiles, chunks, cu_count, batch <= 4);
    auto fits = [&](const I8Split& s) { return std::min((n_tiles + s.tw - 1) / s.tw, cu_count) + producers <= cu_count; };
    if (producers && (batch > 4 || n_tiles >= cu_count) && split.cw * split.tw == 8 && !fits(split)) {
        const uint32_t usual = split.steps;
        for (uint32_t tw = 2 * split.tw; tw <= 4; tw *= 2) {
            const I8Split s{8 / tw, tw, steps_i8(n_tiles, chunks, cu_count, 8 / tw, tw)};
            if (!fits(s) || s.steps > usual + 2) continue;
            split = s;
            break;
        }
    }
    p.cw = split.cw;
    p.tw = split.tw;
    auto bytes = [&](uint32_t stages) {
        const uint32_t waves = p.cw * p.tw;
        return static_cast<size_t>(chunks) * kBpw * (kXqBytes + kXfBytes) + static_cast<size_t>(waves) * (stages * kStageBytes + kMeet * 64 * 2 * 4) + 8 * kMaxLoraRank * 4;
    };
    while (bytes(1) > kLdsBytes) {
        if (p.tw > 1) p.tw /= 2;
        else if (p.cw > 1) p.cw /= 2;
        else return false;
    }
    const uint32_t groups = (n_tiles + p.tw - 1) / p.tw;  // rounds of tiles in all
    p.grid = groups <= cu_count ? groups : cu_count;
    const uint32_t units = (groups + p.grid - 1) / p.grid * ((chunks + p.cw - 1) / p.cw);  // most of a wave
    p.stages = units < kMaxStages ? units : kMaxStages;
    while (bytes(p.stages) > kLdsBytes) --p.stages;
    p.lds = bytes(p.stages);
    *out = p;
    return true;
}

template <int CW, int TW, bool WIDE, bool MULTI, bool LORA>
void launch_i8(const I8Plan& p, const uint8_t* w, uint32_t n, uint32_t k, const float* x, uint32_t x_stride,
               uint32_t batch, float* y, uint32_t y_stride, const LoraEpilogue& lora, const MultiViews& mv,
               hipStream_t stream) {
    static LdsCapOnce lds_cap;
    constexpr auto kernel = gemv_q4_i8<CW, TW, WIDE, MULTI, LORA>;
    lds_cap.raise(reinterpret_cast<const void*>(kernel), kLdsBytes);
    const uint32_t producers = lora.slots ? lora.rank : 0;
    launch_kernel(kernel, dim3(producers + p.grid), dim3(64 * CW * TW), p.lds, stream, w, n,
                       k, x, x_stride, batch, y, y_stride, p.stages, lora, mv);
}

template <bool WIDE, bool MULTI, bool LORA>
void launch_i8_shape(const I8Plan& p, const uint8_t* w, uint32_t n, uint32_t k, const float* x, uint32_t x_stride,
                     uint32_t batch, float* y, uint32_t y_stride, const LoraEpilogue& lora, const MultiViews& mv,
                     hipStream_t stream) {
#define LQ4_I8(CW_, TW_)                \
    if (p.cw == CW_ && p.tw == TW_)     \
    return launch_i8<CW_, TW_, WIDE, MULTI, LORA>(p, w, n, k, x, x_stride, batch, y, y_stride, lora, mv, stream)
    LQ4_I8(8, 1); LQ4_I8(4, 2); LQ4_I8(2, 4); LQ4_I8(1, 8); LQ4_I8(4, 1); LQ4_I8(2, 2); LQ4_I8(2, 1); LQ4_I8(1, 1);
#undef LQ4_I8
}

template <bool MULTI>
void launch_i8_rows(const I8Plan& p, const uint8_t* w, uint32_t n, uint32_t k, const float* x, uint32_t x_stride,
                    uint32_t batch, float* y, uint32_t y_stride, const LoraEpilogue& lora, const MultiViews& mv, bool with_lora,
                    hipStream_t stream) {
    auto go = [&](auto wide) {
        constexpr bool W = decltype(wide)::value;
        if (with_lora) launch_i8_shape<W, MULTI, true>(p, w, n, k, x, x_stride, batch, y, y_stride, lora, mv, stream);
        else launch_i8_shape<W, MULTI, false>(p, w, n, k, x, x_stride, batch, y, y_stride, lora, mv, stream);
    };
    if (batch <= 4) go(std::true_type{});
    else go(std::false_type{});
}

}  // namespace

// The eight waves of every CU have a unit in more than `percent` of their steps.
bool gemv_i8_busier_than(uint32_t percent, uint32_t n, uint32_t k, uint32_t batch, uint32_t cu_count) {
    const uint32_t n_tiles = (n + 15) / 16, chunks = (k / kBlockWeights + kBpw - 1) / kBpw;
    return static_cast<uint64_t>(n_tiles) * chunks * 100 > 8ull * percent * cu_count * split_i8(n_tiles, chunks, cu_count, batch <= 4).steps;
}

bool gemv_i8_serves(uint32_t n, uint32_t k, uint32_t batch, uint32_t cu_count) {
    I8Plan p;
    return plan_i8(n, k, batch, cu_count, &p);
}

void launch_gemv_i8(const uint8_t* w, uint32_t n, uint32_t k, const float* x, uint32_t x_stride, uint32_t batch,
                    float* y, uint32_t y_stride, const LoraEpilogue& lora, uint32_t cu_count, hipStream_t stream) {
    I8Plan p;
    if (!plan_i8(n, k, batch, cu_count, &p, lora.slots ? lora.rank : 0)) return;  // the caller asked gemv_i8_serves first
    const MultiViews none{};
    launch_i8_rows<false>(p, w, n, k, x, x_stride, batch, y, y_stride, lora, none, lora.rank != 0, stream);
}

// The launch can carry `rank_total` producer workgroups for the LoRA factors when they find idle CUs beside the
// workgroups that stream weights (one workgroup runs per CU), the slots (rank_total x 8) and the LDS hold them, and a
// 16-byte row of A can be loaded (K a multiple of 8 elements is given: K is a multiple of 32).
bool gemv_i8_lora_in_launch(uint32_t n, uint32_t k, uint32_t batch, uint32_t rank_total, uint32_t cu_count) {
    I8Plan p;
    return rank_total != 0 && rank_total <= static_cast<uint32_t>(kMaxLoraRank) && plan_i8(n, k, batch, cu_count, &p, rank_total) &&
           p.grid + rank_total <= cu_count;
}

// The stacked launch serves views that are whole numbers of 16-row tiles.
bool gemv_i8_multi_serves(const MultiViews& mv, uint32_t k, uint32_t batch, uint32_t cu_count) {
    if (mv.count == 0 || mv.count > static_cast<uint32_t>(kMaxViews)) return false;
    for (uint32_t v = 0; v < mv.count; ++v)
        if ((mv.begin[v + 1] - mv.begin[v]) % 16) return false;
    I8Plan p;
    return plan_i8(mv.begin[mv.count], k, batch, cu_count, &p);
}

void launch_gemv_i8_multi(const MultiViews& mv, uint32_t k, const float* x, uint32_t x_stride, uint32_t batch,
                          uint32_t cu_count, const LoraEpilogue* in_launch, hipStream_t stream) {
    const uint32_t n = mv.begin[mv.count];
    I8Plan p;
    if (!plan_i8(n, k, batch, cu_count, &p, in_launch ? in_launch->rank : 0)) return;  // the caller asked gemv_i8_multi_serves first
    const LoraEpilogue hand = in_launch ? *in_launch : LoraEpilogue{};  // rank = the views' ranks together, slots, sync
    bool with_lora = false;
    for (uint32_t v = 0; v < mv.count; ++v) with_lora |= mv.rank[v] != 0;
    launch_i8_rows<true>(p, nullptr, n, k, x, x_stride, batch, nullptr, 0, hand, mv, with_lora, stream);
}

}  // namespace lq4
