// Few-token prefill GEMM: Y[M,N] = X[M,K] . W[N,K]^T for 2 .. 128 tokens, and more of small matrices, over Q4, Q8_0 or Q3 blocks.
//
// With so few tokens the product is bound by streaming W once, like the decode GEMV, but there
// are too many tokens for the 4x4x4 GEMV kernel and too few to fill the 128-token tiles of the
// prefill kernels.  Two launches:
//
// 1. pack_x: the activations are converted to f16 once and laid out exactly as the matrix-core
//    B operand wants them: for K step s (128 wide), token group t (16 tokens) and instruction j,
//    the 64 lanes' 16-byte operands are contiguous (1 KB).  Lane (c = lane % 16, g = lane / 16)
//    holds token 16 t + c, K offsets 128 s + 32 g + 8 j .. + 7 in the order x0 x4 x1 x5 x2 x6 x3
//    x7 (the order in which the Q4 dequantiser emits a packed dword; memory order for the sibling
//    formats).  Tokens past M and K past the end are zero-filled, so the main kernel needs no tail
//    handling on this operand.
//
// 2. gemm_q4_skinny<RT, FMT, NTG>: a workgroup of eight waves owns 16 RT weight rows against a tile
//    of NTG groups of 16 tokens.  Wave w takes K steps w, w + 8, ...; per step the load unit puts its 16 RT pieces of rows
//    (four Q4 blocks, 80 bytes) into the wave's own part of LDS, where lane (r, g) picks up block g of row r; the packed
//    operands come with fully coalesced 16-byte loads; it dequantises in registers and issues
//    v_mfma_f32_16x16x32_f16.  No barrier in the K loop: nothing is shared between waves.  Two steps are in flight per wave: the
//    packed operands are loaded without a condition (behind one, the compiler would wait for loads it cannot count), the weights by
//    hand (see dma16; with the builtin one step was in flight: 4096 x 4096 at 128 tokens 15.1 -> 14.1 us, 17408 x 5120 at 20 27.9 -> 26.7,
//    2048 x 6144 at 12 9.4 -> 8.9, Q8_0 2048 x 6144 at 128 17.6 -> 16.9, weights from memory).
//    Blocks straight from memory to the lanes (20 bytes at a row's stride) cost the address unit a clock a lane and load, as much
//    as all the activations of a 64-token step; as dense 16-byte pieces a quarter of that (17408 x 5120 at 20 tokens 29.0 -> 22.0
//    us, 4096 x 4096 at 128 tokens 15.6 -> 13.6, 2048 x 6144 at 100 14.7 -> 12.7; 64 x 2048 x 2048 is latency, 6.9 both ways).  What
//    is left of a step is its activations, four loads of 1 KB a token group through the CU's 64 bytes a clock.
//    Each wave adds its share of the LoRA delta (ranks 2 w, 2 w + 1, then 16 on) to its partial result in
//    f32; the eight partial results then meet in LDS in a fixed order and y is stored once.
//    MULTI = true: the workgroups' row tiles run over several matrices of the same K stacked one under the other
//    (lq4_gemv_multi at 9..128 rows), each with an output and a LoRA delta of its own.
//
// The LoRA factors t = A . X of ranks up to 16 come out of launch 1 as well: its waves hold matrix-core operands of X, so A,
// packed the same way once at upload, costs one more instruction an operand there, and one or two more for what f32
// activations and f32 adapters lose as f16.  The K slices of t go to memory and launch 2 adds them up.
//
// Dequantised value: half(q*d + b) with one rounding (shaders/gemm_q4_tiled.metal:57-66), f32
// accumulation.
#include "lq4_internal.hpp"

#include <cmath>
#include <type_traits>
#include <utility>

namespace lq4 {

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int kWavesK = 8;   // waves of a workgroup, each a K slice
constexpr int TK = 128;      // K per step: four Q4 blocks
constexpr uint32_t kMaxTSlices = 16;     // most K slices of t
constexpr float kRestScale = 2048.0f;    // of what an f32 value loses as f16

struct U4 {
    uint32_t v[4];
};

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }

// One packed dword (weights 8j..8j+7) -> f16 weights in the order w0 w4 w1 w5 w2 w6 w3 w7.  A
// masked dword OR-ed into the mantissa of 1024.0 (or 64.0) is the pair (1024+n_lo, 1024+n_hi);
// a packed subtract makes it (n_lo, n_hi) exactly, a packed fma applies scale and bias.
__device__ __forceinline__ U4 dequant8(uint32_t q, half2v d2, half2v b2) {
    const half2v k1024 = {static_cast<_Float16>(1024.0f), static_cast<_Float16>(1024.0f)};
    const half2v k64 = {static_cast<_Float16>(64.0f), static_cast<_Float16>(64.0f)};
    const uint32_t q8 = q >> 8;
    const half2v t0 = as_h2((q & 0x000F000Fu) | 0x64006400u) - k1024;
    const half2v t1 = as_h2((q & 0x00F000F0u) | 0x54005400u) - k64;
    const half2v t2 = as_h2((q8 & 0x000F000Fu) | 0x64006400u) - k1024;
    const half2v t3 = as_h2((q8 & 0x00F000F0u) | 0x54005400u) - k64;
    U4 out;
    out.v[0] = as_u32(__builtin_elementwise_fma(t0, d2, b2));
    out.v[1] = as_u32(__builtin_elementwise_fma(t1, d2, b2));
    out.v[2] = as_u32(__builtin_elementwise_fma(t2, d2, b2));
    out.v[3] = as_u32(__builtin_elementwise_fma(t3, d2, b2));
    return out;
}

// Sibling formats (FMT 1 = Q8_0, 2 = Q3): their decoders emit the eight weights of an instruction
// in memory order, so their activations are packed without the interleave.
// A block as a lane reads it from LDS, and the 16-byte pieces a row's four blocks of a step take there.
// A Q8_0 block as read: eight whole dwords and the odd half beside them (34-byte blocks: every other one starts inside a dword;
// the first of a step's may, so 136 bytes take nine pieces).  On a dword boundary: scale and weights 0, 1 in dword 0, weights
// 30, 31 in e, and dwords i + 1 : i shifted by two bytes are weights 4 i ..; two bytes past one: the scale in e, the weights in
// the dwords.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
struct Q4Block {
    u32x2 a[2];  // f16 scale | f16 bias << 16, weights 0..23 (nibble i of dword j = weight 8j + i)
    uint32_t e;  // weights 24..31
    __device__ __forceinline__ uint32_t dword(int i) const { return i < 4 ? a[i >> 1 & 1][i & 1] : e; }
};
struct Q8Block {
    u32x2 a[4];
    uint32_t e;
    __device__ __forceinline__ uint32_t dword(int i) const { return i < 8 ? a[i >> 1 & 3][i & 1] : e; }
};
struct Q3Block {
    u32x4 a;  // scale | bias; weight i of 16-weight half h at bits 2i of dword 1 + h; high bits: weight i at bit i of dword 3
};
template <int FMT>
struct WBlockOf {
    typedef Q4Block type;
    static constexpr uint32_t kBytes = 20, kPieces = 5;
    static constexpr int kReads = 3;
};
template <>
struct WBlockOf<1> {
    typedef Q8Block type;
    static constexpr uint32_t kBytes = 34, kPieces = 9;
    static constexpr int kReads = 5;
};
template <>
struct WBlockOf<2> {
    typedef Q3Block type;
    static constexpr uint32_t kBytes = 16, kPieces = 4;
    static constexpr int kReads = 1;
};

// Memory -> LDS, 16 or 4 bytes a lane: lane l's bytes land at LDS byte address `lds` + 16 l (or + 4 l); `base` and `lds` are
// wave-uniform.  By hand, like the LDS reads behind them and the waits: while one that the compiler knows of is in flight, it
// empties the queue in front of every LDS access and of the first use of any other load.  (The builtin's steady state was one
// unit in flight.)  The waits it places for the packed operands do not count these, so they wait for a few loads more.
// The compiler knows of no hazard either: a vector load may read a scalar register five wait states after a vector instruction
// wrote it, so each brings its own.  m0 cannot be named as written: it is reserved, and set by the compiler in front of whatever
// of its own reads it.
__device__ __forceinline__ void dma16(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void dma4(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
template <int OFF>
__device__ __forceinline__ u32x4 lds_read128(uint32_t addr) {
    u32x4 r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
    return r;
}
// two dwords (a 16-byte read that starts on any dword stalls the unit for some 45 clocks)
template <int OFF>
__device__ __forceinline__ u32x2 lds_read2x32(uint32_t addr) {
    static_assert(OFF % 4 == 0 && OFF / 4 + 1 < 256, "offsets are counted in dwords, in a byte");
    u32x2 r;
    asm volatile("ds_read2_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(r) : "v"(addr), "n"(OFF / 4), "n"(OFF / 4 + 1) : "memory");
    return r;
}
template <int OFF>
__device__ __forceinline__ uint32_t lds_read32(uint32_t addr) {
    uint32_t r;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
    return r;
}
template <int OFF>
__device__ __forceinline__ uint32_t lds_read_u16(uint32_t addr) {
    uint32_t r;
    asm volatile("ds_read_u16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
    return r;
}
// At most N LDS operations of the wave are outstanding; no use of the block moves ahead of it.
template <int N>
__device__ __forceinline__ void wait_w(Q4Block& b) {
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(b.a[0]), "+v"(b.a[1]), "+v"(b.e) : "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_w(Q8Block& b) {
    asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(b.a[0]), "+v"(b.a[1]), "+v"(b.a[2]), "+v"(b.a[3]), "+v"(b.e) : "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_w(Q3Block& b) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(b.a) : "n"(N) : "memory");
}
template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// Q8_0: two packed dwords (weights 8j..8j+7) -> half(q * d).  A sign-flipped byte (q + 128) under the
// exponent byte of 1024.0 is 1024 + 128 + q exactly; subtract, then one multiply with one rounding.
__device__ __forceinline__ U4 dequant8_q8(uint32_t qa, uint32_t qb, half2v d2) {
    const half2v k1152 = {static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
    const uint32_t ua = qa ^ 0x80808080u, ub = qb ^ 0x80808080u;
    U4 out;
    out.v[0] = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, ua, 0x04010400u)) - k1152) * d2);
    out.v[1] = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, ua, 0x04030402u)) - k1152) * d2);
    out.v[2] = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, ub, 0x04010400u)) - k1152) * d2);
    out.v[3] = as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, ub, 0x04030402u)) - k1152) * d2);
    return out;
}

// Q3: weights 8j..8j+7 -> half(q * d + b), q = low2 | hi << 2.
__device__ __forceinline__ U4 dequant8_q3(uint32_t lo, uint32_t hi, int j, half2v d2, half2v b2) {
    const half2v k1024 = {static_cast<_Float16>(1024.0f), static_cast<_Float16>(1024.0f)};
    const uint32_t lw = (lo >> (16 * (j & 1))) & 0xffffu;  // 8 two-bit fields
    const uint32_t hw = (hi >> (8 * j)) & 0xffu;                   // 8 bits
    U4 out;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const uint32_t l4 = lw >> (4 * p), h2 = hw >> (2 * p);
        const uint32_t qa = (l4 & 3u) | ((h2 & 1u) << 2);
        const uint32_t qb = ((l4 >> 2) & 3u) | ((h2 & 2u) << 1);
        out.v[p] = as_u32(__builtin_elementwise_fma(as_h2(0x64006400u | qa | (qb << 16)) - k1024, d2, b2));
    }
    return out;
}

__device__ __forceinline__ uint32_t pack_h2(float lo, float hi) {
    const half2v h = {static_cast<_Float16>(lo), static_cast<_Float16>(hi)};
    return as_u32(h);
}

__device__ __forceinline__ float load_b(const void* b, int is_f16, size_t idx) {
    return is_f16 ? static_cast<float>(static_cast<const _Float16*>(b)[idx]) : static_cast<const float*>(b)[idx];
}

// Eight activations of one token, as loaded (zeros past the last token or the end of K).
template <bool X_F16>
struct XRaw {
    uint4 c[X_F16 ? 1 : 2];
};
template <bool X_F16>
__device__ __forceinline__ XRaw<X_F16> load_x(const void* __restrict__ xv, uint32_t m, uint32_t k, uint32_t token, uint32_t koff) {
    XRaw<X_F16> r;
    const bool live = token < m && koff < k;
    const uint8_t* const at = static_cast<const uint8_t*>(xv) + (live ? (static_cast<size_t>(token) * k + koff) * (X_F16 ? 2 : 4) : 0);
#pragma unroll
    for (int l = 0; l < (X_F16 ? 1 : 2); ++l) {
        const uint4 v = *reinterpret_cast<const uint4*>(at + 16 * l);
        r.c[l] = live ? v : make_uint4(0, 0, 0, 0);
    }
    return r;
}
// ... as f16.  INTERLEAVE: in the x0 x4 x1 x5 .. order of the Q4 decoder; false = memory order (sibling formats).
template <bool X_F16, bool INTERLEAVE>
__device__ __forceinline__ uint4 x_operand(const XRaw<X_F16>& r) {
    uint4 out;
    if constexpr (X_F16) {
        const uint4 c = r.c[0];
        if (!INTERLEAVE) return c;
        out.x = __builtin_amdgcn_perm(c.z, c.x, 0x05040100u);  // x0..x7 -> x0 x4 x1 x5 x2 x6 x3 x7
        out.y = __builtin_amdgcn_perm(c.z, c.x, 0x07060302u);
        out.z = __builtin_amdgcn_perm(c.w, c.y, 0x05040100u);
        out.w = __builtin_amdgcn_perm(c.w, c.y, 0x07060302u);
    } else {
        const float4 lo = __builtin_bit_cast(float4, r.c[0]), hi = __builtin_bit_cast(float4, r.c[1]);
        if (INTERLEAVE) {
            out.x = pack_h2(lo.x, hi.x);
            out.y = pack_h2(lo.y, hi.y);
            out.z = pack_h2(lo.z, hi.z);
            out.w = pack_h2(lo.w, hi.w);
        } else {
            out.x = pack_h2(lo.x, lo.y);
            out.y = pack_h2(lo.z, lo.w);
            out.z = pack_h2(hi.x, hi.y);
            out.w = pack_h2(hi.z, hi.w);
        }
    }
    return out;
}
// What f32 activations lose in x_operand<false, true>, times 2^11 (so that it is a normal f16 wherever it matters).  At most
// 16 is lost (half a place of the largest f16); the clamp to that keeps an activation which became an infinity from
// turning up here as another infinity of the other sign.
__device__ __forceinline__ uint4 x_operand_rest(const XRaw<false>& r, uint4 rounded) {
    const float4 lo = __builtin_bit_cast(float4, r.c[0]), hi = __builtin_bit_cast(float4, r.c[1]);
    auto rest = [](float a, float b, uint32_t q) {
        const half2v h = as_h2(q);
        const float da = __builtin_amdgcn_fmed3f(a - static_cast<float>(h[0]), -16.0f, 16.0f);
        const float db = __builtin_amdgcn_fmed3f(b - static_cast<float>(h[1]), -16.0f, 16.0f);
        return pack_h2(da * kRestScale, db * kRestScale);
    };
    return make_uint4(rest(lo.x, hi.x, rounded.x), rest(lo.y, hi.y, rounded.y), rest(lo.z, hi.z, rounded.z), rest(lo.w, hi.w, rounded.w));
}

// grid (K steps, token groups), 256 threads: 4 instructions x 64 lanes.
template <bool X_F16, bool INTERLEAVE>
__global__ __launch_bounds__(256) void pack_x_kernel(const void* __restrict__ xv, uint32_t m, uint32_t k, uint4* __restrict__ xp) {
    const uint32_t s = blockIdx.x, t = blockIdx.y, groups = gridDim.y;
    const int j = threadIdx.x >> 6, lane = threadIdx.x & 63;
    xp[((static_cast<size_t>(s) * groups + t) * 4 + j) * 64 + lane] =
        x_operand<X_F16, INTERLEAVE>(load_x<X_F16>(xv, m, k, 16 * t + (lane & 15), s * TK + 32 * (lane >> 4) + 8 * j));
}

// Token groups in a row of the slices of t: [K slice][rank 0..15][token of its group][group], so that a lane of the product
// gets a rank's factors of all its workgroup's groups in one load.
__host__ __device__ inline uint32_t t_groups(uint32_t groups) { return groups <= 2 ? groups : (groups + 3) & ~3u; }

// Adapters whose t = A . X the packing launch computes: `a` packed by gemm_skinny_pack_lora_a, `part` their sums over a K slice
// (t_groups).
struct PackLora {
    uint32_t count;
    uint32_t has_rest;  // bit v: a f32 adapter, the image of A's rest lies behind that of A
    const uint4* a[kMaxViews];
    float* part[kMaxViews];
};

// The packing launch with adapters (Q4): grid (K slices, token groups, runs of NV adapters), WAVES waves; a wave takes J of the four instructions of a
// K step, a workgroup WAVES J / 4 steps at a time, slice p of P the runs of so many steps p, p + P, ...  NV: adapters at a
// time (those past the count repeat the last one and are dropped).  A_REST: some adapter is f32.
// t is exact to f32 rounding, as the launch for t that the larger kernels need: f32 activations and f32 adapters are the sum
// of two f16 values, the second one scaled by 2^11, and the three products that matter are summed in f32.
// It is bound by latency: one round trip for everything a step needs (activations and the operands of all adapters are
// requested together), one barrier, and as many workgroups as its slices allow.  16 workgroups of 1024 threads that fetched
// adapter by adapter behind the activations took 4.0 us at K 2048 and 64 rows, where the plain form takes 2.1, and a
// projection of 2048 rows 9.7 (f32) and 9.2 us (f16 activations); 8.5 and 8.0 so, 7.1 and 7.0 without an adapter.  J and
// WAVES: see pack_lora_form.
template <bool X_F16, int NV, bool A_REST, int J, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void pack_x_lora_kernel(const void* __restrict__ xv, uint32_t m, uint32_t k,
                                                                      uint4* __restrict__ xp, uint32_t steps, uint32_t slices,
                                                                      uint32_t groups, PackLora la) {
    const uint32_t t = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t token = 16 * t + (lane & 15), rest_off = steps * 256;
    const int j0 = wave % (4 / J) * J;
    const uint32_t v0 = blockIdx.z * NV;
    const uint4* a_of[NV];
    bool has_rest[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const uint32_t i = v0 + v < la.count ? v0 + v : la.count - 1;
        a_of[v] = la.a[i];
        has_rest[v] = la.has_rest >> i & 1;
    }
    float4v acc[NV], rest[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = rest[v] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr uint32_t kRun = WAVES * J / 4;
    for (uint32_t s = blockIdx.x * kRun + wave / (4 / J); s < steps; s += slices * kRun) {
        XRaw<X_F16> raw[J];
        uint4 a[NV][J], ar[A_REST ? NV : 1][J];
#pragma unroll
        for (int j = 0; j < J; ++j) raw[j] = load_x<X_F16>(xv, m, k, token, s * TK + 32 * (lane >> 4) + 8 * (j0 + j));
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const uint32_t at = (s * 4 + j0 + j) * 64 + lane;
                a[v][j] = a_of[v][at];
                if constexpr (A_REST) ar[v][j] = a_of[v][at + (has_rest[v] ? rest_off : 0)];
            }
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const uint4 x = x_operand<X_F16, true>(raw[j]);
            uint4 xr;
            if constexpr (!X_F16) xr = x_operand_rest(raw[j], x);
            if (v0 == 0) xp[((static_cast<size_t>(s) * groups + t) * 4 + j0 + j) * 64 + lane] = x;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const half8 av = __builtin_bit_cast(half8, a[v][j]), xv8 = __builtin_bit_cast(half8, x);
                acc[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, xv8, acc[v], 0, 0, 0);
                if constexpr (!X_F16) rest[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, __builtin_bit_cast(half8, xr), rest[v], 0, 0, 0);
                if constexpr (A_REST) {
                    const uint4 r = has_rest[v] ? ar[v][j] : make_uint4(0, 0, 0, 0);
                    rest[v] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, r), xv8, rest[v], 0, 0, 0);
                }
            }
        }
    }
    // the waves' sums, in wave order
    __shared__ float4v part[NV][WAVES][64];
#pragma unroll
    for (int v = 0; v < NV; ++v) part[v][wave][lane] = acc[v] + rest[v] * (1.0f / kRestScale);
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        if (v % WAVES != wave || v0 + v >= la.count) continue;
        float4v sum = part[v][0][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) sum += part[v][w][lane];
        float* const to = la.part[v0 + v] + ((static_cast<size_t>(blockIdx.x) * 16 + 4 * (lane >> 4)) * 16 + (lane & 15)) * t_groups(groups) + t;
#pragma unroll
        for (int i = 0; i < 4; ++i) to[i * 16 * t_groups(groups)] = sum[i];  // element i of lane (c, g): rank 4 g + i, token c of the group
    }
}

// The sum over the four lanes l, l + 16, l + 32, l + 48, in all of them: (0 + 1) + (2 + 3).
__device__ __forceinline__ float sum_over_lane_groups(float v) {
    auto f32 = [](uint32_t u) { return __builtin_bit_cast(float, u); };
    const auto p = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t b = __builtin_bit_cast(uint32_t, f32(p[0]) + f32(p[1]));
    const auto q = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return f32(q[0]) + f32(q[1]);
}

// RT: 16-row weight tiles per wave (rows per workgroup = 16 RT).  grid (ceil(N / 16 RT), token tiles).
// FMT: 0 = Q4, 1 = Q8_0, 2 = Q3 blocks.
// NTG: 16-token groups a workgroup computes (1, 2 or 4), grid.y tiles of so many; a token tile with fewer groups re-reads its
// last group and drops the results.  Fixed per instantiation, like the prefetches of the K loop below:
// a load behind a run-time condition makes the compiler wait for loads it cannot count, and the
// pipeline collapses to one unit in flight.
// MULTI: w, n, y and lora come from `views`, the view that holds this workgroup's row tile.  LORA: 0 = without the LoRA
// step (a plain call would pay 0.1 us for the branches around it); 1, 2: see where the factors are requested.
// A wave's part of LDS: two steps of weights, and at the end its accumulators.
template <int RT, int NTG, int FMT>
constexpr uint32_t kWaveBytes = 1024 * (2 * ((16 * RT * WBlockOf<FMT>::kPieces + 63) / 64) > RT * NTG ? 2 * ((16 * RT * WBlockOf<FMT>::kPieces + 63) / 64) : RT * NTG);
struct NoViews {};
template <int RT, int FMT, int NTG, bool MULTI, int LORA>
__global__ __launch_bounds__(64 * kWavesK) void gemm_q4_skinny(const uint8_t* __restrict__ w, uint32_t n, uint32_t k,
                                                                const uint4* __restrict__ xp, uint32_t m,
                                                                float* __restrict__ y, LoraEpilogue lora,
                                                                typename std::conditional<MULTI, SkinnyViews, NoViews>::type views) {
    extern __shared__ float4v red[];  // kWaveBytes a wave

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lr = lane & 15;
    const int g = lane >> 4;

    uint32_t row_tile = blockIdx.x;
    if constexpr (MULTI) {
        uint32_t v = 0, first = 0;  // view and its first row tile
        for (uint32_t tiles = (views.n[0] + 16 * RT - 1) / (16 * RT); row_tile - first >= tiles;) {  // (grid.x = the views' tiles)
            first += tiles;
            ++v;
            tiles = (views.n[v] + 16 * RT - 1) / (16 * RT);
        }
        row_tile -= first;
        w = views.w[v];
        n = views.n[v];
        y = views.y[v];
        lora = views.lora[v];
    }
    const uint32_t n0 = row_tile * (16 * RT);
    const uint32_t groups = (m + 15) / 16;             // token groups in X (and in the packed image)
    const uint32_t tg0 = blockIdx.y * NTG;  // first token group of this workgroup
    const uint32_t ntg = groups - tg0 < NTG ? groups - tg0 : NTG;
    const uint32_t nb = k / kBlockWeights;
    const uint32_t steps_total = (nb + 3) / 4;
    const uint32_t cnt = steps_total > static_cast<uint32_t>(wave) ? (steps_total - wave + kWavesK - 1) / kWavesK : 0;

    // ---- weights: a wave's step is 16 RT rows of kPieces 16-byte pieces, which the load unit puts into the wave's part of LDS
    typedef typename WBlockOf<FMT>::type WBlock;
    constexpr uint32_t kBytes = WBlockOf<FMT>::kBytes, kPieces = WBlockOf<FMT>::kPieces;
    constexpr int kLoads = (16 * RT * kPieces + 63) / 64;
    const size_t row_bytes = static_cast<size_t>(nb) * kBytes;
    const uintptr_t w_first = reinterpret_cast<uintptr_t>(w) + n0 * row_bytes;
    const uint32_t w_odd = static_cast<uint32_t>(w_first & 3);  // (a piece starts on a dword)
    const uint8_t* const w_base = reinterpret_cast<const uint8_t*>(w_first - w_odd);
    const size_t w_rest = ((n - n0) * row_bytes + w_odd + 3) & ~static_cast<size_t>(3);  // bytes from w_base to the end
    const uint32_t w_left = w_rest < 0xfffffffcu ? static_cast<uint32_t>(w_rest) : 0xfffffffcu;
    // Q3: sixteen rows of four pieces lie four rows apart in the banks, so a row's pieces change places with its number
    auto place = [](uint32_t piece, uint32_t row) { return FMT == 2 ? piece ^ (row >> 2 & 3) : piece; };
    auto piece_off = [&](uint32_t unit) {  // of the wave's unit-th piece, at step 0
        unit = unit < 16 * RT * kPieces ? unit : 16 * RT * kPieces - 1;
        const uint32_t row = unit / kPieces, real = n0 + row < n ? row : n - 1 - n0;
        return ((w_odd + real * static_cast<uint32_t>(row_bytes)) & ~3u) + place(unit % kPieces, row) * 16;
    };
    uint32_t w_off[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) w_off[i] = piece_off(i * 64 + lane);
    const uint32_t w_reach = ((w_odd + (n - n0 < 16 * RT ? n - n0 - 1 : 16 * RT - 1) * static_cast<uint32_t>(row_bytes)) & ~3u) + kPieces * 16;
    uint8_t* const w_lds = reinterpret_cast<uint8_t*>(red) + wave * kWaveBytes<RT, NTG, FMT>;
    const uint32_t w_lds_at = static_cast<uint32_t>(reinterpret_cast<size_t>((__attribute__((address_space(3))) uint8_t*)w_lds));
    uint32_t w_read[RT], w_shift[RT];  // where the lane's block of row tile r lies in a step; Q8_0: how
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        w_read[r] = (16 * r + lr) * (kPieces * 16) + (FMT == 2 ? place(g, 16 * r + lr) : g) * kBytes;
        w_shift[r] = 0;
        if constexpr (FMT == 1) {
            const uint32_t row = n0 + 16 * r + lr < n ? 16 * r + lr : n - 1 - n0;
            const uint32_t at = ((w_odd + row * static_cast<uint32_t>(row_bytes)) & 2) + g * kBytes;  // 2 bytes past a dword or on it
            w_read[r] += (w_odd + row * static_cast<uint32_t>(row_bytes)) & 2;
            w_shift[r] = (at & 2) == 0 ? 2 : 0;
        }
        w_read[r] += w_lds_at;
    }
    auto load_w = [&](uint32_t s, int stage) {
        const uint32_t at = s * (4 * kBytes);
        const uint32_t to = w_lds_at + stage * (kLoads * 1024);
        if (at + w_reach <= w_left) {
#pragma unroll
            for (int i = 0; i < kLoads; ++i) dma16(to + i * 1024, w_base, w_off[i] + at);
        } else {
            // Its last pieces would reach past the end of the matrix.  The last row dword by dword, those past the end read its last
            // one; of the rows before it (at least 16 bytes a row) only pieces of blocks past the end of K do, which are dropped: as
            // far back as they must.  (Everything dword by dword, 0.15 us: 96 x 300 x 3104 6.4 us, K 3072 6.1.)
            const uint32_t last = n - 1 - n0;  // (of a tile in front of the last one: none of its rows)
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                const uint32_t off = w_off[i] + at;
                if ((i * 64 + lane) / kPieces != last) dma16(to + i * 1024, w_base, off + 16 <= w_left ? off : w_left - 16);
            }
            if (last < 16 * RT && lane < static_cast<int>(4 * kPieces)) {
                const uint32_t off = ((w_odd + last * static_cast<uint32_t>(row_bytes)) & ~3u) + place(lane >> 2, last) * 16 + (lane & 3) * 4 + at;
                dma4(to + last * (kPieces * 16), w_base, off < w_left ? off : w_left - 4);
            }
        }
    };
    // the lane's blocks of a step; read_w is followed by wait_w<reads of later row tiles> before a use
    auto read_w = [&](WBlock& b, int r, auto stage_c) {
        // (offsets of a two-dword read end at 1 KB, so the second step's place goes into the address)
        const uint32_t at = w_read[r] + decltype(stage_c)::value * kLoads * 1024;
        if constexpr (FMT == 0) {
            b.a[0] = lds_read2x32<0>(at);
            b.a[1] = lds_read2x32<8>(at);
            b.e = lds_read32<16>(at);
        } else if constexpr (FMT == 1) {
            const uint32_t whole = at + (w_shift[r] ? 0 : 2);
            b.a[0] = lds_read2x32<0>(whole);
            b.a[1] = lds_read2x32<8>(whole);
            b.a[2] = lds_read2x32<16>(whole);
            b.a[3] = lds_read2x32<24>(whole);
            b.e = lds_read_u16<0>(at + (w_shift[r] ? 32 : 0));
        } else {
            b.a = lds_read128<0>(at);
        }
    };

    // ---- LoRA: wave w adds the ranks 2 w, 2 w + 1 (then 16 on) of scale * B[row, :] . t[token, :] to its own partial result in f32, so the
    // delta is spread over all waves and joins their reduction.  The factors of its first two ranks are requested ahead of
    // everything else (behind the K loop their whole latency would stand: the launch is latency from end to end).
    //   LORA = 2: they are what the accumulators start from.  The first step waits for them, but no register is held: 118
    //   instead of 142 at 16 rows x 32 tokens, so that a second workgroup shares the CU (32768 x 1024 at 16 rows 20.2 -> 15.6
    //   us, 16384 x 4096 22.1 -> 20.3).
    //   LORA = 1: they are held through the K loop and added behind it, for rows of one to three steps a wave, where the first
    //   step's wait is not made up for (4096 x 2048 at 64 rows 11.8 -> 10.9).  (Of two row tiles, B is not held beside one
    //   token group, for the second workgroup's sake, and nothing beside four, for lack of registers.)
    // The choice is K's alone (lora_form), as it decides the order of the sum.
    // B as raw bits.  t, where it comes in K slices (LoraEpilogue::a set, so at most 16 ranks): lane (lr, g) takes slices g,
    // g + 4, ... of its token.
    constexpr bool kEarlyT = LORA == 2 || RT * NTG < 8, kEarlyB = kEarlyT && (LORA == 2 || RT == 1 || NTG > 1);
    typedef float TVec __attribute__((ext_vector_type(NTG)));
    TVec t_slice[2][kMaxTSlices / 4];
    uint32_t b_raw[2][RT][4];
    auto first_rank = [&](int p) {  // wave w: ranks 2 w, 2 w + 1 (those past the end read rank 0 and are dropped)
        const uint32_t jj = 2 * wave + p;
        return jj < lora.rank ? jj : 0;
    };
    auto load_t = [&]() {
        if (!lora.a) return;
        const uint32_t tg = t_groups(groups);
        auto load_slices = [&](int h0) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int h = h0; h < h0 + 2; ++h) {
                    uint32_t slice = g + 4 * h;
                    slice = slice < lora.t_slices ? slice : lora.t_slices - 1;
                    t_slice[p][h] = *reinterpret_cast<const TVec*>(lora.t + ((slice * 16 + first_rank(p)) * 16 + lr) * tg + tg0);
                }
        };
        load_slices(0);
        if (lora.t_slices > 8) load_slices(2);
    };
    auto load_b_raw = [&]() {
        auto each = [&](auto load) {
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    uint32_t row = n0 + 16 * r + 4 * g + v;
                    row = row < n ? row : n - 1;
                    load(r, v, static_cast<size_t>(row) * lora.rank);
                }
        };
        if (lora.rank & 1) {
            each([&](int r, int v, size_t row) {
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const size_t idx = row + first_rank(p);
                    b_raw[p][r][v] = lora.b_is_f16 ? static_cast<uint32_t>(static_cast<const uint16_t*>(lora.b)[idx]) : static_cast<const uint32_t*>(lora.b)[idx];
                }
            });
        } else if (lora.b_is_f16) {
            each([&](int r, int v, size_t row) {  // both ranks in a dword
                b_raw[0][r][v] = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(lora.b) + row + first_rank(0));
            });
        } else {
            struct __attribute__((packed, aligned(4))) Two {
                uint32_t v[2];
            };
            each([&](int r, int v, size_t row) {
                const Two two = *reinterpret_cast<const Two*>(static_cast<const uint32_t*>(lora.b) + row + first_rank(0));
                b_raw[0][r][v] = two.v[0];
                b_raw[1][r][v] = two.v[1];
            });
        }
    };
    if (LORA && lora.rank) {
        if constexpr (kEarlyT) load_t();
        if constexpr (kEarlyB) load_b_raw();
    }
    struct Unit {
        uint4 x[NTG][4];  // [token group][instruction]
    };
    uint32_t xg[NTG];  // packed-image group of token group t (clamped to the last one)
#pragma unroll
    for (int t = 0; t < NTG; ++t) xg[t] = tg0 + t < groups ? tg0 + t : groups - 1;
    // i-th step of this wave
    auto load_x_of = [&](Unit& u, uint32_t i) {
        const uint4* xs = xp + static_cast<size_t>(wave + i * kWavesK) * groups * 256 + lane;
#pragma unroll
        for (int t = 0; t < NTG; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) u.x[t][j] = xs[(xg[t] * 4 + j) * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    // (the packed operands first: the loads behind them for which the compiler waits too many, not counting those of the weights, are
    // then the next unit's operands and not its weights)
    auto load = [&](Unit& u, uint32_t i, int stage) {
        load_x_of(u, i);
        load_w(wave + i * kWavesK, stage);
    };

    float4v acc[RT][NTG];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < NTG; ++t) acc[r][t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    auto add_rank = [&](const float (&tv)[NTG], const float (&bv)[RT][4]) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < NTG; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[r][t][v] = fmaf(bv[r][v], tv[t], acc[r][t][v]);
    };
    auto t_of = [&](uint32_t jj, float (&tv)[NTG]) {  // t in memory
#pragma unroll
        for (int t = 0; t < NTG; ++t) {
            uint32_t tok = 16 * (tg0 + t) + lr;
            tok = tok < m ? tok : m - 1;
            tv[t] = lora.t[static_cast<size_t>(tok) * lora.rank + jj];
        }
    };
    auto add_requested = [&]() {  // the two ranks whose factors have been requested
        if (!lora.rank) return;
        if constexpr (!kEarlyT) load_t();
        if constexpr (!kEarlyB) load_b_raw();
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t jj = 2 * wave + p;
            if (jj >= lora.rank) continue;
            float tv[NTG], bv[RT][4];
            if (lora.a) {  // the slices, added up in the same order whatever the tile is
#pragma unroll
                for (int t = 0; t < NTG; ++t) {
                    auto slice = [&](int h) { return static_cast<float>(t_slice[p][h][t]); };
                    float v = g < static_cast<int>(lora.t_slices) ? slice(0) : 0.0f;
#pragma unroll
                    for (int h = 1; h < static_cast<int>(kMaxTSlices) / 4; ++h) v += g + 4 * h < static_cast<int>(lora.t_slices) ? slice(h) : 0.0f;
                    tv[t] = sum_over_lane_groups(v);
                }
            } else {
                t_of(jj, tv);
            }
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    uint32_t raw = b_raw[p][r][v];
                    if (lora.b_is_f16 && !(lora.rank & 1)) raw = p ? b_raw[0][r][v] >> 16 : b_raw[0][r][v] & 0xffffu;
                    bv[r][v] = lora.scale * (lora.b_is_f16 ? f16_bits_to_f32(raw) : __builtin_bit_cast(float, raw));
                }
            add_rank(tv, bv);
        }
    };

    // LATER: loads issued behind this unit's
    auto compute = [&](const Unit& u, uint32_t i, auto stage_c, auto later_c) {
        const bool live = (wave + i * kWavesK) * 4 + g < nb;  // K tail: a block past the end of the row counts as zero
        WBlock blk[RT];
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(later_c)::value) : "memory");  // this unit has landed
#pragma unroll
        for (int r = 0; r < RT; ++r) read_w(blk[r], r, stage_c);
        static_for<RT>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            wait_w<WBlockOf<FMT>::kReads * (RT - 1 - r)>(blk[r]);
            const WBlock& wb = blk[r];
            uint32_t sb;
            if constexpr (FMT == 1) sb = live ? (w_shift[r] ? wb.dword(0) : wb.e) : 0u;  // scale only (the low half)
            else if constexpr (FMT == 2) sb = live ? wb.a[0] : 0u;
            else sb = live ? wb.dword(0) : 0u;
            const half2v d2 = as_h2(__builtin_amdgcn_perm(sb, sb, 0x01000100u));
            const half2v b2 = as_h2(__builtin_amdgcn_perm(sb, sb, 0x03020302u));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                U4 a;
                if constexpr (FMT == 0) {
                    a = dequant8(wb.dword(j + 1), d2, b2);
                } else if constexpr (FMT == 1) {
                    a = dequant8_q8(__builtin_amdgcn_alignbyte(wb.dword(2 * j + 1), wb.dword(2 * j), w_shift[r]),
                                    __builtin_amdgcn_alignbyte(wb.dword(2 * j + 2), wb.dword(2 * j + 1), w_shift[r]), d2);
                } else {
                    a = dequant8_q3(wb.a[1 + (j >> 1)], wb.a[3], j, d2, b2);
                }
#pragma unroll
                for (int t = 0; t < NTG; ++t)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(half8, a), __builtin_bit_cast(half8, u.x[t][j]), acc[r][t], 0, 0, 0);
            }
        });
    };

    // Two units in flight.  Every unit that has a successor two places on prefetches it without a
    // condition; the last two or three units are written out.  (A redundant clamped prefetch instead
    // would be waited for by whatever reuses its registers.)
    // (the scheduling fences keep a unit's arithmetic from being hoisted across the loads around it,
    // which would hold both units' temporaries live at once and spill)
#define LQ4_FENCE() __builtin_amdgcn_sched_barrier(0)
    constexpr std::integral_constant<int, 0> s0{}, none{};
    constexpr std::integral_constant<int, 1> s1{};
    constexpr std::integral_constant<int, kLoads + 4 * NTG> unit{};
    if (cnt > 1) {
        Unit u0, u1;
        load_w(wave, 0);
        load_w(wave + kWavesK, 1);
        LQ4_FENCE();
        load_x_of(u0, 0);
        load_x_of(u1, 1);
        if constexpr (LORA == 2) add_requested();
        uint32_t i = 0;
        for (; i + 3 < cnt; i += 2) {
            compute(u0, i, s0, unit);
            LQ4_FENCE();
            load(u0, i + 2, 0);
            LQ4_FENCE();
            compute(u1, i + 1, s1, unit);
            LQ4_FENCE();
            load(u1, i + 3, 1);
            LQ4_FENCE();
        }
        if (cnt - i == 3) {
            compute(u0, i, s0, unit);
            LQ4_FENCE();
            load(u0, i + 2, 0);
            LQ4_FENCE();
            compute(u1, i + 1, s1, unit);
            LQ4_FENCE();
            compute(u0, i + 2, s0, none);
        } else {
            compute(u0, i, s0, unit);
            LQ4_FENCE();
            compute(u1, i + 1, s1, none);
        }
    } else if (cnt == 1) {
        Unit u0;
        load_w(wave, 0);
        LQ4_FENCE();
        load_x_of(u0, 0);
        if constexpr (LORA == 2) add_requested();
        compute(u0, 0, s0, none);
    } else {
        if constexpr (LORA == 2) add_requested();
    }
#undef LQ4_FENCE

    if constexpr (LORA == 1) add_requested();
    if (LORA) {
        for (uint32_t jj = wave + 2 * kWavesK; jj < lora.rank; jj += kWavesK) {  // the other ranks
            float tv[NTG], bv[RT][4];
            t_of(jj, tv);
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    uint32_t row = n0 + 16 * r + 4 * g + v;
                    row = row < n ? row : n - 1;
                    bv[r][v] = lora.scale * load_b(lora.b, lora.b_is_f16, static_cast<size_t>(row) * lora.rank + jj);
                }
            add_rank(tv, bv);
        }
    }

    // ---- the eight K slices meet in LDS, each wave's in its own part of it (its weights are done with), and are added as (w, w + 4),
    //      then (w, w + 2), then (0, 1): a fixed order, so the result does not depend on timing.  Wave v sums and stores the
    //      16 x 16 tiles v, v + 8, ...  (One barrier; three rounds of half the waves each, and wave 0 storing alone, took 1.4 us.)
    constexpr int kTiles = RT * NTG;
    {
        float4v* const own = red + wave * (kWaveBytes<RT, NTG, FMT> / 16) + lane;
#pragma unroll
        for (int i = 0; i < kTiles; ++i) own[i * 64] = acc[i / NTG][i % NTG];
    }
    __syncthreads();
    // element v of tile (r, t) in lane (lr, g): token 16 (tg0 + t) + lr, weight row n0 + 16 r + 4 g + v
    const bool vec_ok = (n & 3u) == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0;
#pragma unroll
    for (int i0 = 0; i0 < kTiles; i0 += kWavesK) {
        const int i = i0 + wave;
        if (i >= kTiles) return;  // uniform
        float4v part[kWavesK];
#pragma unroll
        for (int v = 0; v < kWavesK; ++v) part[v] = red[v * (kWaveBytes<RT, NTG, FMT> / 16) + i * 64 + lane];
#pragma unroll
        for (int half = kWavesK / 2; half >= 1; half >>= 1)
#pragma unroll
            for (int v = 0; v < half; ++v) part[v] += part[v + half];
        const int r = i / NTG, t = i % NTG;
        const uint32_t gn = n0 + 16 * r + 4 * g, tok = 16 * (tg0 + t) + lr;
        if (gn >= n || static_cast<uint32_t>(t) >= ntg || tok >= m) continue;
        const float4v val = part[0];
        float* dst = y + static_cast<size_t>(tok) * n + gn;
        if (vec_ok) {
            *reinterpret_cast<float4v*>(dst) = val;
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (gn + v < n) dst[v] = val[v];
        }
    }
}

// gemm_q4_skinny's LORA: see there.  (Eight waves: K 1024 is one step a wave, 3072 three.)
inline int lora_form(uint32_t k) { return k > 1024 && k <= 3072 ? 1 : 2; }

// (RT 2 with four token groups, and Q8_0, take more LDS than a kernel gets unasked)
template <auto Kernel>
void raise_lds(size_t bytes) {
    static LdsCapOnce cap;
    if (bytes > 64 * 1024) cap.raise(reinterpret_cast<const void*>(Kernel), 160 * 1024);
}

// `views`: null, or the matrices of a stacked launch (Q4; w, n, y and lora are then not read).
template <int RT, int FMT, int NTG>
void launch_ntg(const uint8_t* w, uint32_t n, uint32_t k, const uint4* xp, uint32_t m, float* y,
                const LoraEpilogue& lora, const SkinnyViews* views, hipStream_t stream) {
    const uint32_t groups = (m + 15) / 16;
    constexpr size_t lds = kWavesK * kWaveBytes<RT, NTG, FMT>;
    const uint32_t token_tiles = (groups + NTG - 1) / NTG;
    const dim3 block(64 * kWavesK);
    if constexpr (FMT == 0) {
        auto launch = [&](uint32_t tiles, uint32_t with_lora, auto multi, auto views_arg) {
            constexpr bool kMulti = decltype(multi)::value;
            const dim3 grid(tiles, token_tiles);
            auto go = [&](auto lora_c) {
                constexpr auto kernel = gemm_q4_skinny<RT, FMT, NTG, kMulti, decltype(lora_c)::value>;
                raise_lds<kernel>(lds);
                launch_kernel(kernel, grid, block, lds, stream, w, n, k, xp, m, y, lora, views_arg);
            };
            if (!with_lora) go(std::integral_constant<int, 0>{});
            else if (lora_form(k) == 1) go(std::integral_constant<int, 1>{});
            else go(std::integral_constant<int, 2>{});
        };
        if (views) {
            uint32_t tiles = 0, with_lora = 0;
            for (uint32_t v = 0; v < views->count; ++v) {
                tiles += (views->n[v] + 16 * RT - 1) / (16 * RT);
                with_lora |= views->lora[v].rank;
            }
            launch(tiles, with_lora, std::true_type{}, *views);
        } else {
            launch((n + 16 * RT - 1) / (16 * RT), lora.rank, std::false_type{}, NoViews{});
        }
    } else {
        constexpr auto kernel = gemm_q4_skinny<RT, FMT, NTG, false, 0>;
        raise_lds<kernel>(lds);
        launch_kernel(kernel, dim3((n + 16 * RT - 1) / (16 * RT), token_tiles), block, lds,
                           stream, w, n, k, xp, m, y, lora, NoViews{});
    }
}

}  // namespace

// Adapters whose t = A . X the packing launch computes (LoraEpilogue::a set, no launch of its own): one matrix-core operand
// holds sixteen ranks.  (At any number of rows: 2048 x 2048 at 65..128 rows 12.7-13.3 us with a launch of its own in front,
// 9.7-10.5 so.)
bool gemm_skinny_computes_t(uint32_t rank) { return rank != 0 && rank <= 16; }

// A [rank <= 16, K] (f32 or f16, host memory) as the kernel's matrix-core operand, f16: for K step s (128 wide) and
// instruction j the 64 lanes' 16-byte operands are contiguous; lane (r = lane % 16, g = lane / 16) holds row r,
// K offsets 128 s + 32 g + 8 j .. + 7 in the order x0 x4 x1 x5 x2 x6 x3 x7 of the packed activations.  Rows past
// the rank and K past the end are zero.  (Read row by row, sixteen rows K * 2 bytes apart, every workgroup's loads
// of a step fell on a few memory channels at once and the launch took 4 us longer.)
// Behind it, for an f32 adapter, a second image with what the first one lost, times 2^11.
size_t gemm_skinny_packed_lora_a_bytes(uint32_t k, int a_is_f16) { return static_cast<size_t>((k + TK - 1) / TK) * 4 * 64 * 16 * (a_is_f16 ? 1 : 2); }
void gemm_skinny_pack_lora_a(const void* a, int a_is_f16, uint32_t rank, uint32_t k, void* out) {
    const uint32_t steps = (k + TK - 1) / TK;
    const size_t image = static_cast<size_t>(steps) * 4 * 64 * 8;
    for (uint32_t s = 0; s < steps; ++s)
        for (uint32_t j = 0; j < 4; ++j)
            for (uint32_t lane = 0; lane < 64; ++lane) {
                const uint32_t r = lane % 16, g = lane / 16;
                const uint32_t k0 = s * TK + 32 * g + 8 * j;
                _Float16* o = static_cast<_Float16*>(out) + ((static_cast<size_t>(s) * 4 + j) * 64 + lane) * 8;
                for (uint32_t e = 0; e < 8; ++e) {
                    const uint32_t src = (e >> 1) + 4 * (e & 1);  // x0 x4 x1 x5 x2 x6 x3 x7
                    float v = 0.0f;
                    if (r < rank && k0 + src < k) {
                        const size_t idx = static_cast<size_t>(r) * k + k0 + src;
                        v = a_is_f16 ? static_cast<float>(static_cast<const _Float16*>(a)[idx]) : static_cast<const float*>(a)[idx];
                    }
                    o[e] = static_cast<_Float16>(v);
                    const float lost = v - static_cast<float>(o[e]);
                    if (!a_is_f16) o[image + e] = static_cast<_Float16>(std::fabs(lost) < INFINITY ? lost * kRestScale : 0.0f);
                }
            }
}

// Where this kernel serves a shape rather than the large-tile kernel, whose tiles of 96 tokens and more leave most CUs idle, or run
// as K slices, until a product is large: up to 16 tokens always; then matrices of up to n rows (the first entry that holds them)
// with K within its bounds.  Measured over 256..24576 rows and K 512..17408 at 24..2048 tokens, f16 activations (with f32 ones
// this kernel leads by more); us there / here on both sides of the lines:
//   17..32 tokens: 4096 x 17408 27.1 / 20.1, 5120 x 17408 30.1 / 24.1, 17408 x 17408 90.7 / 85.7
//   33..64 (at 64): 4096 x 17408 27.0 / 24.2; 8192 x 14336 38.1 / 32.5; 12288 x 6144 27.9 / 27.2; 16384 x 512 8.9 / 8.3, 16384 x 5120 30.6 / 26.1;
//     20480 x 1024 13.7 / 11.3, 20480 x 3072 25.4 / 24.1; 24576 x 2048 22.0 / 20.8 (at 40 19.2 / 19.1), 32768 x 1024 14.6 / 17.5
//   65..128 (at 128): 1024 x 17408 23.4 / 21.8; 2048 x 14336 24.8 / 23.1, 2048 x 17408 27.1 / 26.9; 2080 x 8192 19.5 / 19.9 (at 72 19.6 / 15.0), 2560 x 9728 20.9 / 22.1;
//     4096 x 7168 21.5 / 18.8, 4096 x 8192 22.4 / 20.4; 8192 x 3584 22.9 / 20.1, 8192 x 4096 21.9 / 22.1; 12288 x 512 10.2 / 11.1, 12288 x 1024 14.7 / 13.8, 12288 x 2560 24.5 / 23.1;
//     16384 x 1536 22.3 / 20.3, 16384 x 2048 23.6 / 25.6
//   (16384 and more rows at 33..64 tokens, and 8193 and more at 65..128, with K of at most 1024 stay with the large tiles, as
//   tests/test_gemm_tiles.py has them.)
//   129..192 (at 192): 512 x 17408 22.9 / 22.1; 1024 x 10240 19.8 / 18.6; 2048 x 6144 19.9 / 17.3, 2048 x 10240 22.4 / 24.4; 3072 x 4096 20.2 / 17.0,
//     3072 x 6144 21.1 / 23.6; 4096 x 4096 22.4 / 18.7; 6144 x 3072 22.3 / 20.2; 8192 x 512 9.9 / 11.1, 8192 x 1024 14.6 / 13.6, 8192 x 2048 24.2 / 18.6
//   193..256 (at 256): 1024 x 10240 21.5 / 19.2; 2048 x 2048 19.8 / 9.9, 2048 x 6144 20.2 / 18.7; 3072 x 4096 20.4 / 19.2; 4096 x 3072 22.5 / 18.3, 4096 x
//     4096 22.3 / 22.4; 6144 x 512 10.2 / 11.1, 6144 x 1024 14.8 / 13.9, 6144 x 2048 23.6 / 18.8; 8192 x 2048 23.4 / 24.0
//   257..384 (at 384): 512 x 6144 20.2 / 15.6, 512 x 10240 19.8 / 20.4; 1024 x 4096 17.4 / 15.6, 1024 x 6144 19.4 / 19.6; 2048 x 3072 19.4 / 16.4, 2048 x 4096
//     19.9 / 20.3; 3072 x 2048 21.1 / 16.2; 4096 x 512 9.9 / 11.4, 4096 x 1024 14.6 / 14.3, 4096 x 2048 21.9 / 19.8
//   385..512 (at 512): 512 x 6144 19.5 / 17.1, 512 x 10240 21.2 / 22.7; 1024 x 4096 18.2 / 16.9; 2048 x 2048 20.4 / 15.4, 2048 x 3072 20.1 / 20.2; 3072 x 1024
//     14.8 / 14.6, 3072 x 2048 22.4 / 20.5; 4096 x 2048 23.0 / 25.2
//   513..768 (at 768): 256 x 4096 19.6 / 16.1; 512 x 3072 18.3 / 15.9; 1024 x 2048 17.4 / 14.8, 1024 x 4096 20.6 / 21.6; 2048 x 1024 14.5 / 15.3
//   769..1024 (at 1024): 256 x 3072 18.4 / 15.8; 512 x 2048 19.8 / 15.1, 512 x 3072 17.6 / 18.5; 1024 x 512 9.6 / 10.0, 1024 x 1024 19.5 / 12.6, 1024 x 2048 17.8 / 18.2
// With an adapter the large-tile kernel has a launch for t in front, so the lines lie further out (up to 128 tokens):
//   33..64: 4096 x 17408 37.2 / 29.2; 8192 x 14336 45.4 / 34.5; 12288 x 6144 36.1 / 33.6; 16384 x 5120 40.9 / 28.6; 24576 x 2560 38.9 / 29.0
//   65..128: 1024 x 17408 32.3 / 24.0; 4096 x 10240 33.9 / 26.9; 8192 x 4096 33.5 / 25.7; 12288 x 2560 37.8 / 28.4; 16384 x 1024 26.5 / 22.5, 16384 x 2048 40.2 / 32.3
// The sibling formats' decoders are longer (Q8_0; Q3 alike or better); above 128 tokens they have two thirds of the K of Q4's
// lines, and not the tallest matrices (at 192 4096 x 4096 24.3 / 24.5, at 256 2048 x 4096 20.2 / 16.3, 3072 x 3072 19.5 / 21.4, 6144 x 1024 14.4 / 15.4, at
// 384 2048 x 2048 19.3 / 17.6, 2048 x 3072 18.6 / 22.3, 4096 x 1024 13.9 / 16.3, at 768 1024 x 1024 16.9 / 13.9, 1024 x 2048 18.1 / 20.5):
//   33..64: 4096 x 12288 30.6 / 24.4; 8192 x 8192 30.5 / 24.6; 12288 x 2048 18.2 / 16.6, 12288 x 3072 21.7 / 21.9; 16384 x 2048 22.7 / 17.6
//   65..128: 512 x 17408 23.4 / 18.9; 2048 x 8192 20.6 / 19.1, 2048 x 10240 22.0 / 21.8; 4096 x 6144 21.8 / 19.4; 8192 x 2048 20.1 / 15.8, 8192 x 3072 21.4 / 21.8
// This kernel packs X into the context's scratch.  The large tiles use none where they run a product whole (rows of fewer than
// four steps, or a last round that is nearly full): such a call needs nothing of the context, can be captured on a new one, takes
// the same kernel whether scratch has grown or not, and replays beside other calls.  It keeps that above 128 tokens and in the
// entries marked `sliced`, but for a product inside a call that works in the scratch anyway, also where it would be faster here (us there / here: 129 x 64 x 512 8.1 / 4.4, 256 x 1000 x 384 7.8 / 5.3, 160 x 4096 x
// 768 12.3 / 8.3, 160 x 8192 x 1024 15.3 / 12.4, 40 x 20196 x 1152 15.5 / 13.8; Q8_0 192 x 6144 x 768 12.8 / 13.8, 104 x 8104 x 64 6.9 / 8.6).
namespace {
struct ShapeLimit {
    uint32_t n, k_min, k_max;
    bool sliced = false;  // only what the large tiles run as K slices
};
constexpr ShapeLimit kPlain64[] = {{4096, 0, 17408}, {8192, 0, 14336}, {12288, 0, 6144}, {16384, 1024, 5120}, {20480, 1056, 3072, true}};
constexpr ShapeLimit kPlain128[] = {{1024, 0, 17408}, {2048, 0, 14336}, {4096, 0, 8192}, {8192, 0, 3584}, {12288, 1056, 2560, true}, {16384, 1056, 1536, true}};
constexpr ShapeLimit kPlain192[] = {{512, 0, 14336}, {1024, 0, 10240}, {2048, 0, 6144}, {4096, 0, 4096}, {6144, 0, 3072}, {8192, 1024, 2048}};
constexpr ShapeLimit kPlain256[] = {{1024, 0, 10240}, {2048, 0, 6144}, {3072, 0, 4096}, {4096, 0, 3072}, {6144, 1024, 2048}};
constexpr ShapeLimit kPlain384[] = {{512, 0, 8192}, {1024, 0, 4096}, {2048, 0, 3072}, {3072, 0, 2048}, {4096, 1024, 2048}};
constexpr ShapeLimit kPlain512[] = {{512, 0, 6144}, {1024, 0, 4096}, {2048, 512, 2048}, {3072, 1024, 2048}};
constexpr ShapeLimit kPlain768[] = {{256, 0, 4096}, {512, 0, 3072}, {1024, 0, 2048}};
constexpr ShapeLimit kPlain1024[] = {{256, 0, 3072}, {512, 0, 2048}, {1024, 768, 1536}};
constexpr ShapeLimit kLora64[] = {{4096, 0, 17408}, {8192, 0, 14336}, {12288, 0, 6144}, {16384, 0, 5120}, {24576, 0, 2560}};
constexpr ShapeLimit kLora128[] = {{1024, 0, 17408}, {4096, 0, 10240}, {8192, 0, 4096}, {12288, 0, 2560}, {16384, 1024, 2048}};
constexpr ShapeLimit kSibling64[] = {{4096, 0, 12288}, {8192, 0, 8192}, {12288, 0, 2560}, {16384, 512, 2048, true}};
constexpr ShapeLimit kSibling128[] = {{512, 0, 17408}, {2048, 0, 8192}, {4096, 0, 6144}, {8192, 0, 2560, true}};
}  // namespace

bool gemm_skinny_wants(uint32_t n, uint32_t k, uint32_t m, int fmt, bool with_lora, int x_is_f16, bool in_state) {
    if (k < kBlockWeights) return false;
    if (m <= 16) return true;
    if (m <= 32) return static_cast<uint64_t>(n) * k <= (1ull << 28);
    auto sliced = [&] { return in_state || (fmt ? gemm_sibling_scratch_floats(fmt, n, k, m, x_is_f16, 0) : gemm_wreg_scratch_floats(n, k, m, 0, x_is_f16 != 0)) != 0; };
    auto within = [&](const auto& limits, bool narrowed = false) {
        for (const ShapeLimit& l : limits)
            if (n <= l.n) return (narrowed ? l.k_min <= 512 && k >= l.k_min && k + k / 2 <= l.k_max : k >= l.k_min && k <= l.k_max) && (!l.sliced || sliced());
        return false;
    };
    if (m <= 128) {
        if (fmt) return m <= 64 ? within(kSibling64) : within(kSibling128);
        if (with_lora) return m <= 64 ? within(kLora64) : within(kLora128);
        return m <= 64 ? within(kPlain64) : within(kPlain128);
    }
    if (with_lora || !sliced()) return false;
    if (m <= 256) return m <= 192 ? within(kPlain192, fmt) : within(kPlain256, fmt);
    if (m <= 512) return m <= 384 ? within(kPlain384, fmt) : within(kPlain512, fmt);
    if (m <= 1024) return m <= 768 ? within(kPlain768, fmt) : within(kPlain1024, fmt);
    return false;
}

namespace {

// The form of the packing launch with adapters: as many slices as there may be, and of these as few steps one after the other
// as possible (each is a round trip to memory).  A rule on K alone, so that t has the same bits in every launch.
struct PackLoraForm {
    int j, waves;
    uint32_t slices;
};
inline PackLoraForm pack_lora_form(uint32_t steps) {
    PackLoraForm f{steps <= 8 ? 1 : 2, steps <= 32 ? 4 : steps <= 64 ? 8 : 16, 0};
    const uint32_t run = static_cast<uint32_t>(f.waves * f.j / 4), runs = (steps + run - 1) / run;
    f.slices = runs < kMaxTSlices ? runs : kMaxTSlices;
    return f;
}

}  // namespace

// Packed X, then the slices of t of the adapters whose t the packing launch computes.
size_t gemm_skinny_scratch_bytes(uint32_t k, uint32_t m, uint32_t adapters) {
    const size_t steps = (k / kBlockWeights + 3) / 4, groups = (m + 15) / 16;
    return (steps * groups * 256 + adapters * pack_lora_form(static_cast<uint32_t>(steps)).slices * t_groups(static_cast<uint32_t>(groups)) * 64) * sizeof(uint4);
}

namespace {

template <int NV, int J, int WAVES>
void launch_pack_lora_form(const void* x, int x_is_f16, uint32_t m, uint32_t k, uint4* xp, uint32_t steps, uint32_t slices,
                           uint32_t groups, const PackLora& la, hipStream_t stream) {
    const dim3 grid(slices, groups, (la.count + NV - 1) / NV);
    auto launch = [&](auto kernel) {
        launch_kernel(kernel, grid, dim3(64 * WAVES), 0, stream, x, m, k, xp, steps, slices, groups, la);
    };
    if constexpr (NV * WAVES < 64) {  // (four f32 adapters and sixteen waves: not enough registers, launch_pack_lora)
        if (la.has_rest) return x_is_f16 ? launch(pack_x_lora_kernel<true, NV, true, J, WAVES>) : launch(pack_x_lora_kernel<false, NV, true, J, WAVES>);
    }
    x_is_f16 ? launch(pack_x_lora_kernel<true, NV, false, J, WAVES>) : launch(pack_x_lora_kernel<false, NV, false, J, WAVES>);
}

template <int NV>
void launch_pack_lora_nv(const void* x, int x_is_f16, uint32_t m, uint32_t k, uint4* xp, uint32_t steps, uint32_t groups,
                         const PackLora& la, hipStream_t stream) {
    const PackLoraForm f = pack_lora_form(steps);
    if (f.j == 1) launch_pack_lora_form<NV, 1, 4>(x, x_is_f16, m, k, xp, steps, f.slices, groups, la, stream);
    else if (f.waves == 4) launch_pack_lora_form<NV, 2, 4>(x, x_is_f16, m, k, xp, steps, f.slices, groups, la, stream);
    else if (f.waves == 8) launch_pack_lora_form<NV, 2, 8>(x, x_is_f16, m, k, xp, steps, f.slices, groups, la, stream);
    else launch_pack_lora_form<NV, 2, 16>(x, x_is_f16, m, k, xp, steps, f.slices, groups, la, stream);
}

void launch_pack_lora(const void* x, int x_is_f16, uint32_t m, uint32_t k, uint4* xp, uint32_t steps, uint32_t groups,
                      const PackLora& la, hipStream_t stream) {
    if (la.count <= 1) launch_pack_lora_nv<1>(x, x_is_f16, m, k, xp, steps, groups, la, stream);
    else if (la.count <= 2 || (la.has_rest && pack_lora_form(steps).waves == 16)) launch_pack_lora_nv<2>(x, x_is_f16, m, k, xp, steps, groups, la, stream);
    else launch_pack_lora_nv<4>(x, x_is_f16, m, k, xp, steps, groups, la, stream);
}

template <int FMT>
void launch_fmt(const uint8_t* w, uint32_t n, uint32_t k, const void* x, int x_is_f16, uint32_t m, float* y,
                LoraEpilogue lora, SkinnyViews* views, void* packed_x, hipStream_t stream) {
    const uint32_t steps = (k / kBlockWeights + 3) / 4, groups = (m + 15) / 16;
    uint4* xp = static_cast<uint4*>(packed_x);
    constexpr bool kInterleave = FMT == 0;
    PackLora la{};
    auto produce_t = [&](LoraEpilogue& e) {  // e.a: packed A; e.t becomes the place of the slices
        if (!e.rank || !e.a) return;
        const uint32_t v = la.count++;
        la.a[v] = static_cast<const uint4*>(e.a);
        la.has_rest |= (e.b_is_f16 ? 0u : 1u) << v;
        e.t_slices = pack_lora_form(steps).slices;
        la.part[v] = reinterpret_cast<float*>(xp + static_cast<size_t>(steps) * groups * 256) + static_cast<size_t>(v) * e.t_slices * t_groups(groups) * 256;
        e.t = la.part[v];
    };
    uint32_t tiles16 = (n + 15) / 16;
    if (views) {
        tiles16 = 0;
        for (uint32_t v = 0; v < views->count; ++v) {
            tiles16 += (views->n[v] + 15) / 16;
            produce_t(views->lora[v]);
        }
    } else {
        produce_t(lora);
    }
    if (FMT == 0 && la.count) {
        launch_pack_lora(x, x_is_f16, m, k, xp, steps, groups, la, stream);
    } else {
        const dim3 grid(steps, groups), block(256);
        if (x_is_f16) launch_kernel((pack_x_kernel<true, kInterleave>), grid, block, 0, stream, x, m, k, xp);
        else launch_kernel((pack_x_kernel<false, kInterleave>), grid, block, 0, stream, x, m, k, xp);
    }
    // Every workgroup reads the whole packed X of its token tile, so a wider row tile halves that traffic, at the price of
    // fewer workgroups to balance over the compute units.
    if (groups == 1) {
        // Two row tiles where one of them would need a second round of workgroups.  (8192 x 2048 at 16 tokens 6.1 / 5.7 us)
        if (tiles16 > 256) launch_ntg<2, FMT, 1>(w, n, k, xp, m, y, lora, views, stream);
        else launch_ntg<1, FMT, 1>(w, n, k, xp, m, y, lora, views, stream);
        return;
    }
    // A launch's cost by tile: so much once, so much for every round of 256 workgroups (small tiles share a CU, whence their low
    // second figure), relative to 16 rows x 64 tokens = 100.  Fitted to 159 launches at 17..128 tokens (Q4 256..17408 rows, K
    // 512..17408, 41 sets of q, k and v with adapters, Q8_0 and Q3 alike): the tile so chosen is 0.8 % behind the best of the
    // five on average, 11 % at worst.  us at 16 x 64 / 16 x 32 / 32 x 32 / 32 x 64 / 16 x 16, packing included: 8192 x 2048 at 64
    // tokens 12.1 / 11.0 / 9.9 / 9.4 / -; 1153 x 9024 at 38 16.2 / 12.6 / 14.9 / 18.8 / 10.3; 2088 x 2336 at 83 11.2 / 8.4 / 7.6 / 8.9 / 9.8;
    // 4190 x 4416 at 49 17.5 / 15.8 / 15.1 / 12.1 / 17.4; q, k and v of 3584 + 2 x 512 rows at 66 tokens, two layers, 46.8 / 38.4 / 33.7 / 40.2 /
    // 50.8; Q8_0 2048 x 5120 at 48 12.1 / 9.4 / 11.5 / 14.5 / -.
    struct Tile {
        int rt, ntg, first, each;
    };
    constexpr Tile kTiles[] = {{1, 4, 10, 90}, {1, 2, 24, 57}, {2, 2, FMT ? 26 : 23, FMT ? 80 : 74}, {2, 4, 14, 134}, {1, 1, 24, 46}};
    int best = 0, best_cost = 0;
    for (int i = 0; i < 5; ++i) {
        const uint32_t wgs = (tiles16 + kTiles[i].rt - 1) / kTiles[i].rt * ((groups + kTiles[i].ntg - 1) / kTiles[i].ntg);
        const int cost = kTiles[i].first + kTiles[i].each * static_cast<int>((wgs + 255) / 256);
        if (i == 0 || cost < best_cost) {
            best = i;
            best_cost = cost;
        }
    }
    if (best == 0) launch_ntg<1, FMT, 4>(w, n, k, xp, m, y, lora, views, stream);
    else if (best == 1) launch_ntg<1, FMT, 2>(w, n, k, xp, m, y, lora, views, stream);
    else if (best == 2) launch_ntg<2, FMT, 2>(w, n, k, xp, m, y, lora, views, stream);
    else if (best == 3) launch_ntg<2, FMT, 4>(w, n, k, xp, m, y, lora, views, stream);
    else launch_ntg<1, FMT, 1>(w, n, k, xp, m, y, lora, views, stream);
}

}  // namespace

void launch_gemm_skinny(const uint8_t* w, uint32_t n, uint32_t k, const void* x, int x_is_f16, uint32_t m, float* y,
                        const LoraEpilogue& lora, void* packed_x, hipStream_t stream, int fmt) {
    if (fmt == 1) launch_fmt<1>(w, n, k, x, x_is_f16, m, y, lora, nullptr, packed_x, stream);
    else if (fmt == 2) launch_fmt<2>(w, n, k, x, x_is_f16, m, y, lora, nullptr, packed_x, stream);
    else launch_fmt<0>(w, n, k, x, x_is_f16, m, y, lora, nullptr, packed_x, stream);
}

void launch_gemm_skinny_views(SkinnyViews views, uint32_t k, const float* x, uint32_t m, void* packed_x, hipStream_t stream) {
    launch_fmt<0>(nullptr, 0, k, x, 0, m, nullptr, LoraEpilogue{}, &views, packed_x, stream);
}

}  // namespace lq4
