// Expert passes of the MoE path for many tokens: a grouped GEMM over native Q4 blocks on the f16 matrix cores, as exact
// as the one-token kernels.
//
// The grouped GEMV (lq4_moe_i8.hip) serves four (token, slot) pairs per pass over an expert's rows: right while experts
// have two or three tokens each and the weights' bytes are what is paid for.  With dozens of tokens per expert it reads
// (and unpacks) every block a dozen times; 512 tokens of top 8 among 64 experts took 345 us in the two passes.
// Here a workgroup owns 512 weight rows x up to 64 pairs of one expert and reads its blocks once.
//
// Arithmetic.  A Q4 weight is n * d + b with a nibble n and f16 scale and bias per 32 weights; rounding it to f16, as
// the dense prefill does, is not exact enough here.  So the matrix cores multiply nibbles, not weights: the 32 nibbles of a
// block are f16 operands, an activation is the sum of two f16 values hi + lo after scaling its row by a power of two to a
// largest magnitude in [2^14, 2^15) (22 bits of every element, and every element to 2^-39 of the row's largest), and
// v_mfma_f32_32x32x16_f16 forms D = sum n * (hi + lo) over exactly one block in four instructions.  Then
// acc += d * D in f32, one fma per output: with the weight row in the lane (32x32 D layout: column = lane % 32), d is one
// register.  The bias term sum_b bias[b] * (sum of x over block b) is a product with K = number of blocks and goes through
// the matrix cores too, with the blocks' sums as hi + lo.  1-3e-7 of the largest output against the f64 oracle.
// The nibbles have to be normal numbers: masked out of the dword as they stand they are exact f16 subnormals (n * 2^-24) and
// cost four operations less per dword, but the matrix unit then aligns its products by the subnormals' exponent and keeps
// ten bits less of them (1e-5 of the largest output).
//
// What bounds it: issue.  512 tokens of top 8 among 64 experts (hidden 2048, inter 512, shared expert), gate/up pass 67 us,
// down pass 42 (median of 60 launches).  Counters, gate/up / down: 1.50 / 0.75 M matrix instructions of 32 clocks keep the
// matrix cores busy for 23 / 11 us of that; 7.9 / 8.6 vector and 0.80 / 0.86 LDS instructions go with each of them, and the
// waves spend 36 / 34 % of their cycles ready but waiting for the issue port and 30 / 33 % on a counter.  In a step of two
// tiles it is 64 matrix instructions, 256 fma, 144 operations that turn nibbles into f16 and about 30 others, so every one
// of them is placed by hand, and whatever could be left to memory instructions is: weights and activations go straight
// into LDS.
//
// Loads.  Each lane fetching the 20-byte blocks of its own row, as the dense kernels do, was half of the time at first: 16
// bytes each at a 1280-byte stride cost the address unit a clock per lane and load, whatever the cache held.  Now five
// neighbouring lanes fetch the 80 bytes of a row's step, straight into LDS.
//
// Measured, whole layer in one call (us, before -> here): 512 tokens 411 -> 147, 256 tokens 224 -> 130, 128 tokens 131 -> 121;
// 96 tokens 106 -> 111 and 64 tokens 86 -> 120, which stay with the grouped GEMV (moe_takes_gemm has the line).
#include <utility>

#include "lq4_internal.hpp"

namespace lq4 {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4u __attribute__((aligned(4)));

constexpr int kStepBlocks = 4;       // blocks of a row per step; steps come in pairs
constexpr int kTilePairs = 64;       // pairs per workgroup, two matrix tiles of 32
constexpr int kWaves = 8;            // 64 weight rows each
constexpr int kThreads = 64 * kWaves;
constexpr int kWgRows = 64 * kWaves;
constexpr uint32_t kMaxExperts = 1024;
constexpr uint32_t kMaxPairs = 4096;  // (token, slot) pairs of one call, the C ABI's limit

// LDS: two images of a step's activations, [block][part hi/lo][32-pair tile][32 pairs][4 dwords] of 16-byte units; per wave two
// images of its weights, [64 rows] of 80 bytes as they lie in memory; the block sums of a pair of steps, [64 pairs][part][8].
constexpr int kXBytes = kStepBlocks * 2 * 2 * 2048;
constexpr int kWBytes = 64 * kStepBlocks * kBlockBytes;
constexpr int kSumBytes = kTilePairs * 32;
constexpr int kLdsBytes = 2 * kXBytes + kWaves * 2 * kWBytes + kSumBytes;
// A pair's four units would put a wave's operand reads (one unit of 32 neighbouring pairs, 64 bytes apart) on a quarter of
// the banks: unit j of pair t is kept at place j ^ twist(t), which differs over any eight (or sixteen) neighbours that
// share a bank otherwise.
__host__ __device__ inline uint32_t twist(uint32_t t) { return ((t >> 1) & 2u) | (((t >> 1) ^ (t >> 3)) & 1u); }

// Packed activation row: block slots padded to whole pairs of steps, 128 bytes each ([part][dword] units of eight f16), then per
// 8 slots 32 bytes of block sums ([part] of eight f16).  Slot = block, except that the last, partial step of a row of nb blocks
// holds the row's last four (its weights are read as the row's last 80 bytes, so that no load leaves the row), those of the
// step before as zeros.
__host__ __device__ inline uint32_t padded_blocks(uint32_t nb) { return (nb + 2 * kStepBlocks - 1) / (2 * kStepBlocks) * (2 * kStepBlocks); }
__host__ __device__ inline uint32_t record_bytes(uint32_t nb) { return padded_blocks(nb) * (128 + 4); }

__device__ __forceinline__ float silu(float v) {
    const float den = 1.0f + expf(-v);
    float r = __builtin_amdgcn_rcpf(den);
    r = fmaf(fmaf(-den, r, 1.0f), r, r);  // one Newton step: the quotient to an ulp, at a third of a division
    return den < INFINITY ? v * r : v * 0.0f;
}

// ---- activations -> packed rows ---------------------------------------------------------------------------------
struct PackJob {
    const float* x;     // [rows, k] dense
    uint8_t* out;       // [rows] records
    float* factor;      // [rows]: 2^5 / row scale (what an accumulated sum is multiplied with), NaN for a row with one
    uint32_t rows, k;
};

// One workgroup per row of job a, then of job b.  A thread converts eight neighbouring values at a time.
__global__ __launch_bounds__(256) void moe_pack_kernel(PackJob a, PackJob b) {
    __shared__ uint32_t s_max[4];
    const bool second = blockIdx.x >= a.rows;
    const float* __restrict__ x = second ? b.x : a.x;
    const uint32_t row = second ? blockIdx.x - a.rows : blockIdx.x, k = second ? b.k : a.k;
    const uint32_t nb = k / kBlockWeights, nbp = padded_blocks(nb), rec = record_bytes(nb);
    const uint32_t tid = threadIdx.x;
    const float4* __restrict__ xr = reinterpret_cast<const float4*>(x + static_cast<size_t>(row) * k);
    uint8_t* const out = (second ? b.out : a.out) + static_cast<size_t>(row) * rec;
    const uint32_t units = nb * 4;  // eight values each
    uint32_t mx = 0;                // largest magnitude as bits: infinities and NaNs come out on top
    float4 keep[2];
    for (uint32_t u = tid; u < units; u += 256) {
        const float4 lo = xr[2 * u], hi = xr[2 * u + 1];
        if (u == tid) {
            keep[0] = lo;
            keep[1] = hi;
        }
        const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = max(mx, __builtin_bit_cast(uint32_t, v[i]) & 0x7FFFFFFFu);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) mx = max(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), d, 64)));
    if ((tid & 63) == 0) s_max[tid >> 6] = mx;
    __syncthreads();
    mx = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
    // scale = 2^(14 - exponent): the largest magnitude lands in [2^14, 2^15).  A row below 2^-100 counts as zero.
    const bool finite = mx < 0x7F800000u, live = finite && mx >= 0x0D800000u;
    const uint32_t ebits = mx >> 23;  // 27 .. 254 when live
    const float scale = live ? __builtin_bit_cast(float, (268u - ebits) << 23) : 0.0f;
    if (tid == 0)
        (second ? b.factor : a.factor)[row] = live ? __builtin_bit_cast(float, (ebits - 9u) << 23)
                                                   : finite ? 0.0f : __builtin_bit_cast(float, 0x7FC00000u);
    const uint32_t whole = nb / kStepBlocks * kStepBlocks, gap = (kStepBlocks - nb % kStepBlocks) % kStepBlocks;
    for (uint32_t u = tid; u < nbp * 4; u += 256) {  // (whole quads of lanes share a block)
        const uint32_t slot = u >> 2, j = u & 3;
        const uint32_t blk = slot < whole ? slot : slot - gap;  // (wraps below `whole + gap`: no block)
        float v[8];
        if (live && blk < nb && (slot < whole || slot >= whole + gap)) {
            const uint32_t i = 4 * blk + j;
            const float4 lo = i == tid ? keep[0] : xr[2 * i], hi = i == tid ? keep[1] : xr[2 * i + 1];
            v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = 0.0f;
        }
        float sum = 0.0f;
        half8 ph, pl;
        // operand order: nibbles 0 4 | 1 5 | 2 6 | 3 7
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int src = (i >> 1) + 4 * (i & 1);
            const float xs = v[src] * scale;
            sum += xs;
            ph[i] = static_cast<_Float16>(xs);
            pl[i] = static_cast<_Float16>(xs - static_cast<float>(ph[i]));
        }
        *reinterpret_cast<half8*>(out + slot * 128 + j * 16) = ph;
        *reinterpret_cast<half8*>(out + slot * 128 + 64 + j * 16) = pl;
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        if (j == 0) {
            sum *= 0.03125f;  // |sum| <= 2^20 before
            const _Float16 sh = static_cast<_Float16>(sum), sl = static_cast<_Float16>(sum - static_cast<float>(sh));
            uint8_t* const so = out + nbp * 128 + slot / 8 * 32 + slot % 8 * 2;
            *reinterpret_cast<_Float16*>(so) = sh;
            *reinterpret_cast<_Float16*>(so + 16) = sl;
        }
    }
}

// ---- grouping -----------------------------------------------------------------------------------------------------
// order: the pair indices of every expert next to each other, in the order in which the waves arrive (it differs from run to
// run; moe_gemm_tile sums every pair alike wherever it lies, so the results do not), and the list of workgroup tiles {expert,
// first place in order, pairs}.  `extra` > 0: expert `experts` with every token once (the shared expert; its places are token
// numbers).  Entries up to tile_bound that no tile needs get 0 pairs.
__global__ __launch_bounds__(1024) void moe_tiles_kernel(const int32_t* __restrict__ ids, uint32_t tokens, uint32_t slots,
                                                         uint32_t top_k, uint32_t experts, uint32_t extra,
                                                         uint32_t tile_bound, int32_t* __restrict__ order,
                                                         int4* __restrict__ tiles) {
    __shared__ int32_t s_cnt[kMaxExperts], s_off[kMaxExperts];
    __shared__ int32_t s_sum[2][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    s_cnt[tid] = 0;
    __syncthreads();
    const uint32_t pairs = tokens * top_k;
    int32_t e[kMaxPairs / 1024], place[kMaxPairs / 1024];
#pragma unroll
    for (uint32_t i = 0; i < kMaxPairs / 1024; ++i) {
        const uint32_t p = tid + i * 1024;
        e[i] = -1;
        if (p < pairs) {
            const int32_t id = ids[p / top_k * slots + p % top_k];
            if (id >= 0 && id < static_cast<int32_t>(experts)) e[i] = id;
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < kMaxPairs / 1024; ++i) place[i] = e[i] >= 0 ? atomicAdd(&s_cnt[e[i]], 1) : 0;
    __syncthreads();
    // a thread per expert: its pairs and its tiles, scanned together
    const int32_t c = tid < experts ? s_cnt[tid] : 0;
    const int32_t nt = (c + kTilePairs - 1) / kTilePairs;
    int32_t v[2] = {c, nt};
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int32_t up = __shfl_up(v[q], d, 64);
            if (static_cast<int>(lane) >= d) v[q] += up;
        }
    }
    if (lane == 63) {
        s_sum[0][wave] = v[0];
        s_sum[1][wave] = v[1];
    }
    __syncthreads();
    int32_t before[2] = {0, 0}, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
#pragma unroll
        for (int q = 0; q < 2; ++q) before[q] += w < wave ? s_sum[q][w] : 0;
        total += s_sum[1][w];
    }
    const int32_t off = before[0] + v[0] - c;
    s_off[tid] = off;
    // The tiles in sequence (the shared expert's first, then expert by expert) are cut into eight runs, one per XCD: entry i is
    // taken by XCD i % 8, so the tiles of one expert mostly meet in one L2.
    const int32_t xt = (static_cast<int32_t>(extra) + kTilePairs - 1) / kTilePairs, all = xt + total, per = (all + 7) / 8;
    auto put = [&](int32_t k, int32_t ex, int32_t first, int32_t n) {
        const int32_t at = k % per * 8 + k / per;
        if (at < static_cast<int32_t>(tile_bound)) tiles[at] = make_int4(ex, first, n, 0);
    };
    const int32_t first_tile = xt + before[1] + v[1] - nt;
    for (int32_t i = 0; i < nt; ++i)
        put(first_tile + i, static_cast<int32_t>(tid), off + i * kTilePairs, min(kTilePairs, c - i * kTilePairs));
    for (int32_t i = static_cast<int32_t>(tid); i < xt; i += 1024)
        put(i, static_cast<int32_t>(experts), i * kTilePairs, min(kTilePairs, static_cast<int32_t>(extra) - i * kTilePairs));
    for (int32_t i = static_cast<int32_t>(tid); i < static_cast<int32_t>(tile_bound); i += 1024)  // entries of no tile
        if (all == 0 || i % 8 * per + i / 8 >= all || i / 8 >= per) tiles[i] = make_int4(0, 0, 0, 0);
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kMaxPairs / 1024; ++i) {
        const uint32_t p = tid + i * 1024;
        if (e[i] >= 0) order[s_off[e[i]] + place[i]] = static_cast<int32_t>(p / top_k * slots + p % top_k);
    }
}

// ---- the expert passes ----------------------------------------------------------------------------------------------
// One set of tensors: the routed experts', or the shared expert's own.
struct MoeSide {
    const uint8_t* w;       // expert-major rows
    const uint8_t* x;       // packed activation rows
    const float* factor;    // their factors
    float* out;
    uint32_t nb;            // blocks per row
    uint32_t out_rows;      // outputs per pair: I (gate/up, weight rows I + I) or H (down)
};
struct MoeGemmArgs {
    MoeSide routed, shared;
    const int4* tiles;
    const int32_t* order;
    uint32_t slots;         // routing slots per token (pair = token * slots + slot)
    uint32_t experts;       // tile expert `experts` = the shared one
    uint32_t groups, per_group;  // workgroups per tile, and the chunks of kWgRows weight rows that each of them takes in turn
};

// The eight nibbles of a dword as f16, order 0 4 | 1 5 | 2 6 | 3 7, in nine steps of one instruction each (they are spread
// over the shadows of matrix instructions): under the exponent of 1024 a nibble counts ones or, four bits up, sixteens.
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
struct NibbleTmp {
    uint32_t t[4], u;
};
__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t magic) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(magic));
    return r;
}
__device__ __forceinline__ void nibble_op(int op, uint32_t q, uint32_t magic, NibbleTmp& n, u32x4& out) {
    const half2v m1024 = {static_cast<_Float16>(-1024.0f), static_cast<_Float16>(-1024.0f)};
    const half2v m64 = {static_cast<_Float16>(-64.0f), static_cast<_Float16>(-64.0f)};
    const half2v inv16 = {static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
    auto f16 = [](uint32_t v) { return __builtin_bit_cast(half2v, v); };
    switch (op) {
        case 0: n.t[0] = and_or(q, 0x000F000Fu, magic); break;
        case 1: n.t[1] = and_or(q, 0x00F000F0u, magic); break;
        case 2: n.u = q >> 8; break;
        case 3: n.t[2] = and_or(n.u, 0x000F000Fu, magic); break;
        case 4: n.t[3] = and_or(n.u, 0x00F000F0u, magic); break;
        case 5: out.x = __builtin_bit_cast(uint32_t, f16(n.t[0]) + m1024); break;
        case 6: out.y = __builtin_bit_cast(uint32_t, f16(n.t[1]) * inv16 + m64); break;
        case 7: out.z = __builtin_bit_cast(uint32_t, f16(n.t[2]) + m1024); break;
        default: out.w = __builtin_bit_cast(uint32_t, f16(n.t[3]) * inv16 + m64); break;
    }
}

// LDS reads by hand: one the compiler knows of is made to wait for every global_load_lds in flight.  (The register is tied
// to itself, so that it is not copied between the read and the wait.)
__device__ __forceinline__ void lds_read(u32x4& r, uint32_t addr, int off) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "+v"(r) : "v"(addr), "n"(off) : "memory");
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void lds_read_sum(u32x2& r, uint32_t addr, int off) {
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(off) : "memory");
}
__device__ __forceinline__ void lds_read1(uint32_t& r, uint32_t addr, int off) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "+v"(r) : "v"(addr), "n"(off) : "memory");
}
// dwords at off and off + 8 bytes
__device__ __forceinline__ void lds_read_pair(u32x2& r, uint32_t addr, int off) {
    asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3" : "+v"(r) : "v"(addr), "n"(off / 4), "n"(off / 4 + 2) : "memory");
}
template <int N>
__device__ __forceinline__ void lds_wait(u32x4& r) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(r) : "n"(N));
}

template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// One workgroup's tile of TT x 32 pairs.
//
// Schedule.  A product is one block of the wave's 64 rows x one 32-pair tile: eight matrix instructions (two row tiles x {lo, hi}
// x two halves of the block) into one of two sets of D.  In their shadows, a few operations behind each: the 32 fma of the
// product before (its D set), the nibbles of the block after, the reading of the block after that, and the re-reading of an
// operand register for the product after as soon as its last use has been issued.  The last product of a step lies behind the
// step's barrier: it reads the next step's image and requests the activations and weights of the step after that, so both are
// a step on their way.
template <bool GATE_UP, int TT>
__device__ __forceinline__ void moe_gemm_tile(const MoeGemmArgs& p, const MoeSide& S, const int4 tile, uint32_t chunk0, bool shared,
                                              uint8_t* lds, float* s_factor, const int32_t* s_row, const int32_t* s_pair) {
    constexpr uint32_t kOut = GATE_UP ? 32 : 64;  // outputs per wave
    constexpr int P = kStepBlocks * TT;           // products per step
    const int n = tile.z;
    const uint32_t out_rows = S.out_rows, nb = S.nb;
    const uint32_t tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr uint32_t kChunkRows = kWaves * kOut;  // outputs per chunk
    const uint32_t chunks = min(p.per_group, (out_rows + kChunkRows - 1) / kChunkRows - chunk0);
    uint32_t row0 = chunk0 * kChunkRows + wave * kOut;
    const uint32_t rec = record_bytes(nb), row_bytes = nb * kBlockBytes;
    const uint32_t steps = padded_blocks(nb) / kStepBlocks;  // even
    const uint8_t* const wbase = S.w + static_cast<size_t>(shared ? 0 : tile.x) * (GATE_UP ? 2 : 1) * out_rows * row_bytes;

    // Requests, all straight into LDS (lane l of an instruction to the 16 bytes at place l).
    typedef __attribute__((address_space(1))) void global_void_t;
    typedef __attribute__((address_space(3))) void lds_void_t;
    // weights: five lanes a row, 320 pieces of 16 bytes a step.  (32-bit offsets: an expert's tensor and the packed rows are
    // below 4 GB, see moe_gemm_serves)
    uint32_t woff[5];
    auto weight_rows = [&](uint32_t first) {  // (a row past the end repeats the last one; its results are not stored)
#pragma unroll
        for (uint32_t i = 0; i < 5; ++i) {
            const uint32_t c = i * 64 + lane, lr = c / 5;
            uint32_t row = min(first + (GATE_UP ? lr & 31 : lr), out_rows - 1);
            if (GATE_UP && lr >= 32) row += out_rows;
            woff[i] = row * row_bytes + (c - 5 * lr) * 16;
        }
    };
    weight_rows(row0);
    uint8_t* const wimg = lds + 2 * kXBytes + wave * (2 * kWBytes);
    auto load_w_one = [&](uint32_t s, int buf, int i) {
        const uint32_t blk = min(s * kStepBlocks, nb - kStepBlocks);  // (a last, partial step: the row's last 80 bytes)
        __builtin_amdgcn_global_load_lds((global_void_t*)(wbase + blk * kBlockBytes + woff[i]),
                                         (lds_void_t*)(wimg + buf * kWBytes + i * 1024), 16, 0, 0);
    };
    // activations: a wave moves two blocks (TT = 2) or one (TT = 1) of a group of 16 pairs, four lanes the 64 bytes of a (pair,
    // block, part)
    constexpr int kXLoads = 2 * TT;
    const uint32_t group = wave % (2 * TT), xt = 16 * group + (lane >> 2);
    const uint32_t xoff = static_cast<uint32_t>(s_row[xt]) * rec + (((lane & 3) ^ twist(xt & 31)) * 16);
    auto load_x_one = [&](uint32_t s, int buf, int i) {
        const uint32_t bp = wave / (2 * TT) * kXLoads + i;  // block and part
        const uint8_t* const src = S.x + (s * (kStepBlocks * 128) + bp * 64);
        uint8_t* const dst = lds + buf * kXBytes + (bp * TT + group / 2) * 2048 + (group & 1) * 1024;
        __builtin_amdgcn_global_load_lds((global_void_t*)(src + xoff), (lds_void_t*)dst, 16, 0, 0);
    };
    const uint32_t st = 32 * (wave % TT) + (lane >> 1);  // (several waves move the same sums)
    const uint32_t soff = static_cast<uint32_t>(s_row[st]) * rec + padded_blocks(nb) * 128 + (lane & 1) * 16;
    uint8_t* const simg = lds + 2 * kXBytes + kWaves * 2 * kWBytes;
    auto load_sums = [&](uint32_t s) {  // of the pair of steps that s belongs to
        __builtin_amdgcn_global_load_lds((global_void_t*)(S.x + (s >> 1) * 32 + soff), (lds_void_t*)(simg + (wave % TT) * 1024), 16, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < 5; ++i) load_w_one(0, 0, i);
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) load_x_one(0, 0, i);
    load_sums(0);
#pragma unroll
    for (int i = 0; i < 5; ++i) load_w_one(1, 1, i);
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) load_x_one(1, 1, i);

    if (tid < kTilePairs) s_factor[tid] = S.factor[s_row[tid]];  // (for the end of a chunk)

    auto lds_at = [](const uint8_t* q) { return static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) const uint8_t*)q)); };
    const uint32_t addr0 = lds_at(lds) + r * 64 + ((g ^ twist(r)) * 16), addr1 = lds_at(lds) + r * 64 + (((2 + g) ^ twist(r)) * 16);
    const uint32_t saddr = lds_at(simg) + r * 32 + g * 8;
    const uint32_t haddr = lds_at(wimg) + r * (kStepBlocks * kBlockBytes), waddr = haddr + 4 + g * 4;

    float16v acc[2][TT], D[2][2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            D[1][rt][i] = 0.0f;
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) acc[rt][tt][i] = 0.0f;
        }
    }
    uint32_t magic = 0x64006400u;
    asm("" : "+v"(magic));
    u32x2 wq[2][2] = {};         // [parity of the block][row tile]: its dwords g and 2 + g as they came
    uint32_t wh[2][2] = {};      // its scale and bias
    u32x4 wv[2][2][2];           // [parity][row tile][half of the block]: f16
    float d[kStepBlocks][2];     // [block][row tile]: its scale, with the block sums' 2^-5
    uint32_t hold[2];            // [row tile]: the header of the even block before
    uint32_t bias[2][2][2];      // [step parity][row tile]: its four biases
    NibbleTmp tmp;
    u32x4 F[4] = {};             // operands of the product under way: lo, lo, hi, hi
    constexpr int kOps = 36;     // nibble operations of a block: 4 dwords x 9

    auto read_block = [&](auto bc, auto bufc) {  // block b of image buf, both row tiles: four reads
        constexpr int b = decltype(bc)::value, off = decltype(bufc)::value * kWBytes + b * kBlockBytes;
        // (a pair's offsets are counted in dwords up to 255: the image and the row tile go into the address)
        constexpr int tile_bytes = 32 * kStepBlocks * kBlockBytes;
        static_for<2>([&](auto rc) {
            constexpr int rt = decltype(rc)::value;
            lds_read_pair(wq[b & 1][rt], waddr + (decltype(bufc)::value * kWBytes + rt * tile_bytes), b * kBlockBytes);
            lds_read1(wh[b & 1][rt], haddr, off + rt * tile_bytes);
        });
    };
    // what a block's header says (its reads are complete: the wait before this tied the registers)
    auto open_block = [&](int b, int step_parity) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            d[b][rt] = f16_bits_to_f32(wh[b & 1][rt] & 0xFFFFu) * 0.03125f;
            if (b & 1) bias[step_parity][rt][b >> 1] = __builtin_amdgcn_perm(wh[1][rt], hold[rt], 0x07060302u);
            else hold[rt] = wh[0][rt];
        }
    };
    auto nibble_step = [&](int b, int e) {
        const int rt = e / 18, half = e / 9 % 2;
        nibble_op(e % 9, half == 0 ? wq[b & 1][rt].x : wq[b & 1][rt].y, magic, tmp, wv[b & 1][rt][half]);
    };
    auto arrived = [&](int b) {  // the last wait covered block b's reads: no use of them before this point
        asm volatile("" : "+v"(wq[b & 1][0]), "+v"(wq[b & 1][1]), "+v"(wh[b & 1][0]), "+v"(wh[b & 1][1]));
    };
    // operand c (0, 1: lo, 2, 3: hi) of product j of the step in image `buf`
    auto read_operand = [&](auto cc, auto jc, auto bufc) {
        constexpr int c = decltype(cc)::value, j = decltype(jc)::value, buf = decltype(bufc)::value;
        constexpr int blk = j / TT, tt = j % TT;
        lds_read(F[c], (c & 1) ? addr1 : addr0, buf * kXBytes + ((blk * 2 + (c < 2 ? 1 : 0)) * TT + tt) * 2048);
    };
    // bias . sums over the eight blocks of a pair of steps: half-wave g holds the four of step g.  Every tile adds it behind
    // block 2 of the pair's second step and before block 3, so that an output's bits do not depend on which of the tiles, or in
    // how full a workgroup, its pair lies.
    auto read_sums = [&](auto tc, u32x2 (&sum)[2]) {
        constexpr int tt = decltype(tc)::value;
        lds_read_sum(sum[0], saddr, tt * 1024);
        lds_read_sum(sum[1], saddr, tt * 1024 + 16);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sum[0]), "+v"(sum[1]));
    };
    auto add_bias = [&](auto tc, const u32x2 (&sum)[2]) {
        typedef _Float16 half4 __attribute__((ext_vector_type(4)));
        constexpr int tt = decltype(tc)::value;
        u32x2 b[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) b[rt] = u32x2{g ? bias[1][rt][0] : bias[0][rt][0], g ? bias[1][rt][1] : bias[0][rt][1]};
#pragma unroll
        for (int part = 1; part >= 0; --part)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
                acc[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(half4, sum[part]), __builtin_bit_cast(half4, b[rt]),
                                                                   acc[rt][tt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };

    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    constexpr std::integral_constant<int, 0> zero{};
    constexpr std::integral_constant<int, 1> one{};
    d[3][0] = d[3][1] = 0.0f;
    read_block(zero, zero);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    arrived(0);
    open_block(0, 0);
#pragma unroll
    for (int e = 0; e < kOps; ++e) nibble_step(0, e);
    read_block(one, zero);
    static_for<4>([&](auto c) { read_operand(c, zero, zero); });

    auto step = [&](uint32_t s, auto parity) {
        constexpr int B = decltype(parity)::value;  // images of this step
        const uint32_t s2 = s + 2 < steps ? s + 2 : s + 2 - steps;  // (of the next chunk: weight_rows)
        static_for<P>([&](auto jc) {
            constexpr int j = decltype(jc)::value, blk = j / TT, tt = j % TT;
            constexpr int prev_blk = j == 0 ? kStepBlocks - 1 : (j - 1) / TT, prev_tt = (j + TT - 1) % TT;
            constexpr int next_blk = (blk + 1) % kStepBlocks, after_blk = (blk + 2) % kStepBlocks;
            constexpr bool last = j == P - 1;
            // The bias term (its sums are read before the barrier that frees them).  Of two tiles, this one has block 2
            // behind it; a single tile adds block 2 in this very product, and the bias after it.
            constexpr bool with_bias = B == 1 && blk == kStepBlocks - 1;
            constexpr std::integral_constant<int, tt> this_tile{};
            u32x2 sum[2];
            if constexpr (with_bias) read_sums(this_tile, sum);
            if constexpr (with_bias && TT == 2) add_bias(this_tile, sum);
            // every wave is done with this step's image (its own last operands have arrived), and the next one has landed
            if constexpr (last) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            static_for<8>([&](auto cc) {
                constexpr int c = decltype(cc)::value, op = c / 2, rt = c % 2;
                // operand reads are answered in order, three of them younger than the one wanted here; between the
                // second and the last of a block's first product so are the four of read_block
                if constexpr (rt == 0) lds_wait<(tt == 0 && c > 0) ? 7 : 3>(F[op]);
                if constexpr (tt == 0 && c == 0) arrived(next_blk);
                __builtin_amdgcn_sched_barrier(0);
                const half8 a = __builtin_bit_cast(half8, F[op]), b = __builtin_bit_cast(half8, wv[blk & 1][rt][op & 1]);
                if constexpr (op == 0) D[j & 1][rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, float16v{}, 0, 0, 0);
                else D[j & 1][rt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, D[j & 1][rt], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);  // (the matrix instruction first, or two of them end up back to back)
                if constexpr (tt == 0 && c == 0) {
                    // (a wave's weights are its own business: no barrier, but they must have landed; everything
                    // requested in the last step's last product has had most of a step to do so)
                    if constexpr (after_blk == 0 && !last) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    read_block(std::integral_constant<int, after_blk>{}, std::integral_constant<int, after_blk < blk ? 1 - B : B>{});
                }
                if constexpr (rt == 1) read_operand(std::integral_constant<int, op>{}, std::integral_constant<int, (j + 1) % P>{},
                                                    std::integral_constant<int, last ? 1 - B : B>{});
#pragma unroll
                for (int f = 4 * c; f < 4 * c + 4; ++f)  // the product before: its fma's
                    acc[f >> 4][prev_tt][f & 15] = fmaf(d[prev_blk][f >> 4], D[(j & 1) ^ 1][f >> 4][f & 15], acc[f >> 4][prev_tt][f & 15]);
                constexpr int slot = tt * 8 + c, slots = 8 * TT;
                if constexpr (slot == slots - 1) open_block(next_blk, next_blk == 0 ? 1 - B : B);
#pragma unroll
                for (int e = slot * kOps / slots; e < (slot + 1) * kOps / slots; ++e) nibble_step(next_blk, e);
                if constexpr (last) {
                    if constexpr (c < 5) load_w_one(s2, B, c);
#pragma unroll
                    for (int i = c * kXLoads / 8; i < (c + 1) * kXLoads / 8; ++i) load_x_one(s2, B, i);
                    if constexpr (c == 7 && B == 1) load_sums(s2);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (with_bias && TT == 1) add_bias(this_tile, sum);
        });
    };
    for (uint32_t c = 0;;) {
        for (uint32_t s = 0; s < steps; s += 2) {
            if (s + 2 == steps && c + 1 < chunks) weight_rows(row0 + kChunkRows);  // (what is requested from here on is the next chunk's)
            step(s, zero);
            step(s + 1, one);
        }
#pragma unroll
        for (int f = 0; f < 32; ++f) {
            acc[f >> 4][TT - 1][f & 15] = fmaf(d[3][f >> 4], D[1][f >> 4][f & 15], acc[f >> 4][TT - 1][f & 15]);
            D[1][f >> 4][f & 15] = 0.0f;
        }
        // D layout: register i of lane (r, g) = pair 8 (i / 4) + 4 g + i % 4 of the tile, weight row r
        uint32_t out0 = row0 + r;
        int first = tile.y;
        asm volatile("" : "+v"(out0), "+s"(first));  // (or the addresses below are computed before the loop, and spilled)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const int t0 = 32 * tt + 8 * i4 + 4 * static_cast<int>(g);
                __builtin_amdgcn_sched_barrier(0);  // (four outputs at a time)
                const float4 f4 = *reinterpret_cast<const float4*>(s_factor + t0);
                const int4 pair4 = *reinterpret_cast<const int4*>(s_pair + t0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = 4 * i4 + q;
                    const float f = q == 0 ? f4.x : q == 1 ? f4.y : q == 2 ? f4.z : f4.w;
                    const float a = acc[0][tt][i] * f, b = acc[1][tt][i] * f;
                    acc[0][tt][i] = acc[1][tt][i] = 0.0f;
                    if (GATE_UP) {
                        const float h = silu(a) * b;
                        if (t0 + q < n && out0 < out_rows) S.out[static_cast<size_t>(first + t0 + q) * out_rows + out0] = h;
                    } else {
                        const int pair = q == 0 ? pair4.x : q == 1 ? pair4.y : q == 2 ? pair4.z : pair4.w;
                        float* const o = S.out + static_cast<size_t>(pair) * out_rows + out0;
                        if (t0 + q < n && out0 < out_rows) o[0] = a;
                        if (t0 + q < n && out0 + 32 < out_rows) o[32] = b;
                    }
                }
            }
        }
        if (++c == chunks) break;
        row0 += kChunkRows;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // (the last requests, which nobody reads)
}

// GATE_UP: a wave owns gate rows [r, r + 32) and up rows I + [r, r + 32); out[place] (routed: place in order, shared: token)
// receives silu(g) * u.  Else: rows [r, r + 64), activation rows by place, out[pair].
template <bool GATE_UP>
__global__ __launch_bounds__(kThreads) void moe_gemm_kernel(MoeGemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t s_x[];  // kLdsBytes
    __shared__ float s_factor[kTilePairs];
    __shared__ int32_t s_row[kTilePairs], s_pair[kTilePairs];
    // Workgroup id % 8 is the XCD: the row chunks of one tile run next to each other on one of them, so that its L2 serves the
    // tile's activations to all but the first.
    const uint32_t xcd = blockIdx.x & 7, at = blockIdx.x >> 3, chunk = at % p.groups * p.per_group, tile_no = at / p.groups * 8 + xcd;
    const int4 tile = p.tiles[tile_no];
    const int n = tile.z;
    if (n == 0) return;
    const bool shared = static_cast<uint32_t>(tile.x) == p.experts;
    const MoeSide S = shared ? p.shared : p.routed;
    if (chunk * (GATE_UP ? kWgRows / 2 : kWgRows) >= S.out_rows) return;
    if (threadIdx.x < kTilePairs) {  // (a place beyond the tile repeats its last pair; its results are not stored)
        const int place = tile.y + min(static_cast<int>(threadIdx.x), n - 1);
        const int32_t pair = shared ? place : p.order[place];
        s_row[threadIdx.x] = !GATE_UP || shared ? place : pair / static_cast<int32_t>(p.slots);
        s_pair[threadIdx.x] = pair;
    }
    __syncthreads();
    if (n > 32) moe_gemm_tile<GATE_UP, 2>(p, S, tile, chunk, shared, s_x, s_factor, s_row, s_pair);
    else moe_gemm_tile<GATE_UP, 1>(p, S, tile, chunk, shared, s_x, s_factor, s_row, s_pair);
}

// y[t, c] = sum over the slots, in slot order, of weight * o[t, s, c], then the shared expert's weight * its row.
__global__ __launch_bounds__(256) void moe_gemm_combine_kernel(const float* __restrict__ o, const float* __restrict__ o_shared,
                                                               const int32_t* __restrict__ ids, const float* __restrict__ weights,
                                                               uint32_t experts, uint32_t top_k, uint32_t slots, uint32_t hidden,
                                                               float* __restrict__ y) {
    const uint32_t t = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (c >= hidden) return;
    float4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    auto add = [&](float w, const float* row) {
        const float4 v = *reinterpret_cast<const float4*>(row + c);
        acc.x += w * v.x; acc.y += w * v.y; acc.z += w * v.z; acc.w += w * v.w;
    };
#pragma unroll 4
    for (uint32_t s = 0; s < top_k; ++s) {
        const int32_t e = ids[t * slots + s];
        if (e >= 0 && e < static_cast<int32_t>(experts)) add(weights[t * slots + s], o + static_cast<size_t>(t * slots + s) * hidden);
    }
    if (o_shared) add(weights[t * slots + top_k], o_shared + static_cast<size_t>(t) * hidden);
    *reinterpret_cast<float4*>(y + static_cast<size_t>(t) * hidden + c) = acc;
}

inline size_t up256(size_t v) { return (v + 255) / 256 * 256; }

// Scratch of a call.
struct Plan {
    size_t order, tiles, xf, hf, hsf, x, h, hp, hs, hsp, o, os, total;
    uint32_t tile_bound;
};
Plan plan(const MoeGemmShape& m) {
    Plan l;
    const size_t pairs = static_cast<size_t>(m.tokens) * m.top_k, spairs = static_cast<size_t>(m.tokens) * (m.top_k + (m.shared_inter ? 1 : 0));
    // at most one tile per 64 pairs and one more per expert that has any
    const size_t partial = pairs < m.experts ? pairs : m.experts;
    l.tile_bound = static_cast<uint32_t>(pairs / kTilePairs + partial + (m.shared_inter ? m.tokens / kTilePairs + 1 : 0) + 7) / 8 * 8;
    l.order = 0;
    l.tiles = l.order + up256(pairs * 4);
    l.xf = l.tiles + up256(static_cast<size_t>(l.tile_bound) * 16);
    l.hf = l.xf + up256(static_cast<size_t>(m.tokens) * 4);
    l.hsf = l.hf + up256(pairs * 4);
    l.x = l.hsf + up256(static_cast<size_t>(m.tokens) * 4);
    l.h = l.x + up256(static_cast<size_t>(m.tokens) * record_bytes(m.hidden / kBlockWeights));
    l.hp = l.h + up256(pairs * m.inter * 4);
    l.hs = l.hp + up256(pairs * record_bytes(m.inter / kBlockWeights));
    l.hsp = l.hs + up256(static_cast<size_t>(m.tokens) * m.shared_inter * 4);
    l.o = l.hsp + up256(static_cast<size_t>(m.tokens) * (m.shared_inter ? record_bytes(m.shared_inter / kBlockWeights) : 0));
    l.os = l.o + up256(spairs * m.hidden * 4);
    l.total = l.os + up256(m.shared_inter ? static_cast<size_t>(m.tokens) * m.hidden * 4 : 0);
    return l;
}

}  // namespace

bool moe_gemm_serves(const MoeGemmShape& m) {
    return m.experts < kMaxExperts && static_cast<uint64_t>(m.tokens) * m.top_k <= kMaxPairs && m.hidden % kBlockWeights == 0 &&
           m.inter % kBlockWeights == 0 && m.shared_inter % kBlockWeights == 0 && m.hidden >= kStepBlocks * kBlockWeights &&
           m.inter >= kStepBlocks * kBlockWeights && (m.shared_inter == 0 || m.shared_inter >= kStepBlocks * kBlockWeights) && m.hidden <= 65536 && m.inter <= 32768 &&
           m.shared_inter <= 32768;
}

size_t moe_gemm_scratch_bytes(const MoeGemmShape& m) { return plan(m).total; }

void launch_moe_gemm(const MoeGemmShape& m, const uint8_t* gate_up, const uint8_t* down, const uint8_t* shared_gate_up,
                     const uint8_t* shared_down, const float* x, const int32_t* ids, const float* weights, float* y,
                     uint8_t* scratch, hipStream_t stream) {
    const Plan l = plan(m);
    const uint32_t slots = m.top_k + (m.shared_inter ? 1 : 0), pairs = m.tokens * m.top_k;
    const uint32_t nbh = m.hidden / kBlockWeights, nbi = m.inter / kBlockWeights, nbs = m.shared_inter / kBlockWeights;
    int32_t* const order = reinterpret_cast<int32_t*>(scratch + l.order);
    int4* const tiles = reinterpret_cast<int4*>(scratch + l.tiles);
    auto f32 = [&](size_t off) { return reinterpret_cast<float*>(scratch + off); };
    static LdsCapOnce cap_up, cap_down;
    constexpr size_t lds = kLdsBytes;
    cap_up.raise(reinterpret_cast<const void*>(moe_gemm_kernel<true>), static_cast<int>(lds));
    cap_down.raise(reinterpret_cast<const void*>(moe_gemm_kernel<false>), static_cast<int>(lds));
    launch_kernel(moe_tiles_kernel, dim3(1), dim3(1024), 0, stream, ids, m.tokens, slots, m.top_k, m.experts,
                       m.shared_inter ? m.tokens : 0u, l.tile_bound, order, tiles);
    const PackJob none{nullptr, nullptr, nullptr, 0, kBlockWeights};
    launch_kernel(moe_pack_kernel, dim3(m.tokens), dim3(256), 0, stream,
                       PackJob{x, scratch + l.x, f32(l.xf), m.tokens, m.hidden}, none);
    const uint32_t widest = m.inter > m.shared_inter ? m.inter : m.shared_inter;
    // A workgroup takes as many chunks of rows as leave one workgroup per CU: it fills the pipeline and reads its routing once
    // (512 tokens, down pass, one chunk / two per workgroup: 47.0 / 42.4 us).
    const uint32_t tiles_likely = (pairs + m.experts * (kTilePairs / 2)) / kTilePairs + (m.shared_inter ? (m.tokens + kTilePairs - 1) / kTilePairs : 0);
    auto split = [&](uint32_t chunks, uint32_t& groups, uint32_t& per) {
        per = (chunks * tiles_likely + 255) / 256;
        if (per < 1) per = 1;
        if (per > chunks) per = chunks;
        groups = (chunks + per - 1) / per;
    };
    uint32_t up_groups, up_per, down_groups, down_per;
    split((widest + kWgRows / 2 - 1) / (kWgRows / 2), up_groups, up_per);
    split((m.hidden + kWgRows - 1) / kWgRows, down_groups, down_per);
    MoeGemmArgs up{{gate_up, scratch + l.x, f32(l.xf), f32(l.h), nbh, m.inter},
                   {shared_gate_up, scratch + l.x, f32(l.xf), f32(l.hs), nbh, m.shared_inter}, tiles, order, slots, m.experts, up_groups, up_per};
    launch_kernel(moe_gemm_kernel<true>, dim3(l.tile_bound * up_groups), dim3(kThreads), lds, stream, up);
    launch_kernel(moe_pack_kernel, dim3(pairs + (m.shared_inter ? m.tokens : 0)), dim3(256), 0, stream,
                       PackJob{f32(l.h), scratch + l.hp, f32(l.hf), pairs, m.inter},
                       m.shared_inter ? PackJob{f32(l.hs), scratch + l.hsp, f32(l.hsf), m.tokens, m.shared_inter} : none);
    MoeGemmArgs dn{{down, scratch + l.hp, f32(l.hf), f32(l.o), nbi, m.hidden},
                   {shared_down, scratch + l.hsp, f32(l.hsf), f32(l.os), nbs, m.hidden}, tiles, order, slots, m.experts, down_groups, down_per};
    launch_kernel(moe_gemm_kernel<false>, dim3(l.tile_bound * down_groups), dim3(kThreads), lds, stream, dn);
    launch_kernel(moe_gemm_combine_kernel, dim3((m.hidden / 4 + 255) / 256, m.tokens), dim3(256), 0, stream, f32(l.o),
                       m.shared_inter ? f32(l.os) : nullptr, ids, weights, m.experts, m.top_k, slots, m.hidden, y);
}

}  // namespace lq4
