// Matrix products of the encoder's training step: fp32 in, fp32 sums, on the 16-bit matrix cores of gfx950.
//
// An fp32 number is the sum of three bf16 numbers (8 + 8 + 8 bits, each piece rounded to nearest: the third takes what is
// left exactly).  Of the nine products of pieces the six largest are taken, x0 y0, x0 y1, x1 y0, x1 y1, x0 y2, x2 y0: what is left out
// is below 2^-26 of |x y|, at any magnitude (ENLARGED below), under the rounding of one fp32 addition.  Six v_mfma_f32_32x32x16_bf16 cost 192 clocks where the same
// product on v_mfma_f32_32x32x2_f32 takes 512, and their fp32 accumulator rounds once per 16 products instead of once per 2.
//
// gemm_f32_kernel (rows of A along k): a workgroup makes one 64 x 64 tile of C.  Four waves (a group) hold 32 x 32 of it each and step through
// K by 16; where the tiles are too few to fill the chip, 2 or 4 groups share a tile, each with its own steps and its own LDS stages, and
// add up at the end in a fixed order (the same bits on every call).  A step: 8 floats per thread travel global -> registers two steps
// ahead, are split (6.5 vector instructions each) and written to one of two stages as 16-byte fragments, eight consecutive k of one row; the
// product reads them with ds_read_b128.  The next step's split is laid between the products (one after the other, odd groups the other way round, 2048 x 512 x 2048
// 34.2 us and with a matrix added 38.3, so 32.0 and 33.8; 4096 x 512 x 512 20.0 and 18.7, 8192 x 768 x 256 28.3 and 26.1).  What bounds it: a 64 x 64 x 16
// step reads 24 KB and writes 12 KB of LDS (288 clocks at 128 bytes a clock) beside 192 of products.  Smaller where it counts than the traffic of operands split beforehand: 6 bytes an element through L2.
//
// gemm_f32_rows_kernel (rows of A and B across k: gradients of weights): there 32 lanes read 128 consecutive bytes of one k, so a wave loads what
// its fragments hold straight into registers, no LDS and no barrier: 64 x 64 of C over the wave's share of the steps, the next step split
// under the 24 products of this one, the one after it on its way; the waves of a workgroup add up in LDS at the end.  With rows along
// k a lane would read 32 bytes of a row of its own: 38 and 43 us against 36 and 38 (2048 x 512 x 2048 and 2048 x 2048 x 512).
//
// Few tiles over many tokens leave compute units idle, each of the others a serial chain over K: there workgroups take shares of K (rows_shares), whose
// sums a second launch adds up in their order.
//
// us, 2048 tokens, this / the library's fp32 product and torch's elementwise kernels (calls one behind the other; up to a tenth between boxes): QKV 2048 x 1536 x 512 26.5 to 28.7 / 33.5, its
// output 10.8 / 18; feed-forward 2048 x 2048 x 512 31.7 / 36.0 (with bias and GELU 36.0 / 45.4, with GELU's derivative 36.7 / 45.4), 2048 x 512 x 2048 31.7 / 34.1 (with a matrix added 32.0 / 41.0);
// gradients of weights 512 x 2048 x 2048 and 2048 x 512 x 2048 30.3 / 38, 512 x 1536 x 2048 26.0 / 29.4, 512 x 512 x 2048 14.9 / 18.2 (through the first kernel 44, 39, 35, 31); 8192 tokens 79 / 97, 31 / 36,
// 103 / 126 (119 / 147, 133 / 156), 93 / 119 (95 / 128) and 103 / 121, 85 / 98, 33 / 54.
// Error against float64 at K = 2048 2.5e-7 to 3.5e-7, the library's 8.1e-7.
//
// Values that are not finite (or become so: bf16 ends half a step below fp32) do not split; an element of C that comes out not
// finite is summed again in plain fp32.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "gemm_f32_internal.h"

namespace {

using namespace proteus_gemm;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float  f32x2  __attribute__((ext_vector_type(2)));
typedef float  f32x16 __attribute__((ext_vector_type(16)));

constexpr int GT        = 64;                       // rows and columns of a tile
constexpr int GK        = 16;                       // k of a step
constexpr int CHUNK     = GT * 16 + 64;             // bytes of 8 k of all rows of one piece (64 more: the two halves of a step in different banks)
constexpr int PIECE     = 2 * CHUNK;
constexpr int OPERAND   = 3 * PIECE;
constexpr int STAGE     = 2 * OPERAND;              // of one group

__device__ __forceinline__ uint32_t pack2(const float a, const float b) {
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
// bf16 has fp32's range but not its smallest numbers: below 2^-109 the third piece, below 2^-117 the second would fall under 2^-133, where bf16
// ends.  Operands are therefore split 2^16 times as large, which leaves nothing of an fp32 number out, subnormals among them, and sums are
// 2^32 times the result.  (What overflows that way, operands from 2^112 and sums from 2^96 on, is not finite and summed again in plain fp32.)
// Relative error (2-norm) against float64 of operands about 2^-113, 2^-120, 2^-126, as they are / so: 2.8e-7, 3.5e-5, 2.2e-3 / 5.5e-8 (the library 1.4e-7).
// A multiplication per element: 2048 x 512 x 2048 31.7 -> 32.6 us, 512 x 2048 x 2048 28.3 -> 29.7.
constexpr float ENLARGED = 0x1p16f, REDUCED = 0x1p-32f;
__device__ __forceinline__ float low(const uint32_t w)  { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float high(const uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// Four consecutive k of one row into the three pieces' fragments, `piece` bytes apart.
__device__ __forceinline__ void split_to_lds(char* at, const float4& from, const int piece = PIECE)
{
    const float4 v = make_float4(from.x * ENLARGED, from.y * ENLARGED, from.z * ENLARGED, from.w * ENLARGED);
    uint2 p;
    p.x = pack2(v.x, v.y); p.y = pack2(v.z, v.w);
    *reinterpret_cast<uint2*>(at) = p;
    const float a = v.x - low(p.x), b = v.y - high(p.x), c = v.z - low(p.y), d = v.w - high(p.y);
    p.x = pack2(a, b); p.y = pack2(c, d);
    *reinterpret_cast<uint2*>(at + piece) = p;
    p.x = pack2(a - low(p.x), b - high(p.x)); p.y = pack2(c - low(p.y), d - high(p.y));
    *reinterpret_cast<uint2*>(at + 2 * piece) = p;
}

// A thread's share of an operand: four consecutive k of one row (of A, or of B^T) per step.  KC: k is the contiguous dimension in memory,
// else the row is.  Loads are unconditional (so that they stay in flight over the branches of the step): what lies outside the matrix
// is out of the buffer's range and comes back as zero.
template <bool KC> struct Source {
    static constexpr uint32_t OUT = 0x80000000u;               // (matrices end below 2^31 bytes)
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t at;                                               // of the thread's row at k = 0
    int k, K, pitch;
    __device__ __forceinline__ Source(const float* X, const int ld, const int row, const int rows, const int k_, const int K_)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc((void*)X, 0, (uint32_t)((KC ? (size_t)(rows - 1) * ld + K_ : (size_t)(K_ - 1) * ld + rows) * 4), 0x00020000)),
          at(row < rows ? (KC ? (uint32_t)row * (uint32_t)ld * 4u : (uint32_t)row * 4u) : OUT), k(k_), K(K_), pitch(ld * 4) {}
    __device__ __forceinline__ float4 fetch(const int k0) const
    {
        if (KC) return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, k0 + k < K ? at + (uint32_t)(k0 + k) * 4u : OUT, 0, 0));     // (K is a multiple of 4)
        const uint32_t o = at + (uint32_t)(k0 + k) * (uint32_t)pitch;          // (rows of k past K lie behind the end, and so does all of a row outside: below 2^32)
        auto one = [&](const int i) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, o + (uint32_t)(i * pitch), 0, 0)); };
        return make_float4(one(0), one(1), one(2), one(3));
    }
};

// Barrier for LDS alone: loads from memory stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); }

// One element of A B in plain fp32.
template <bool AK, bool BK>
__device__ __forceinline__ float plain_dot(const GemmArgs& g, const int m, const int n)
{
    float s = 0.f;
    for (int k = 0; k < g.K; ++k)
        s = __builtin_fmaf(AK ? g.A[(size_t)m * g.lda + k] : g.A[(size_t)k * g.lda + m], BK ? g.B[(size_t)n * g.ldb + k] : g.B[(size_t)k * g.ldb + n], s);
    return s;
}

// Does a row (of A, or of B^T) hold a NaN at k0 <= k < k1?  (Plain loads, which nothing keeps inside the matrix: k1 <= K.)
template <bool KC>
__device__ __forceinline__ bool any_nan(const float* __restrict__ X, const int ld, const int row, const int rows, const int k0, const int k1)
{
    if (row >= rows) return false;
    bool found = false;
#pragma unroll 8
    for (int k = k0; k < k1; ++k) { const float v = KC ? X[(size_t)row * ld + k] : X[(size_t)k * ld + row]; found |= v != v; }
    return found;
}

__device__ __forceinline__ float gelu(const float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(const float x) {
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    return __builtin_fmaf(x, 0.39894228040143268f * expf(-0.5f * x * x), cdf);
}

// Element (m, n); `h` is that of g.h where the epilogue reads it.
template <int EPI> constexpr bool reads_h() { return EPI == PROTEUS_GEMM_ADD || EPI == PROTEUS_GEMM_GELU_GRAD; }
template <int EPI>
__device__ __forceinline__ void write(const GemmArgs& g, const int m, const int n, float v, const float h = 0.f)
{
    if (g.bias) v += g.bias[n];
    const size_t at = (size_t)m * g.ldc + n;
    if (EPI == PROTEUS_GEMM_F32)        static_cast<float*>(g.C)[at] = v;
    else if (EPI == PROTEUS_GEMM_BF16)  static_cast<__bf16*>(g.C)[at] = (__bf16)v;
    else if (EPI == PROTEUS_GEMM_GELU)  { g.H[at] = v; static_cast<float*>(g.C)[at] = gelu(v); }
    else if (EPI == PROTEUS_GEMM_ADD)   static_cast<float*>(g.C)[at] = v + h;
    else                                static_cast<float*>(g.C)[at] = v * gelu_grad(h);
}

// AK, BK: k contiguous in A [M][K] / B [N][K]; else A is [K][M] / B [K][N]
template <bool AK, bool BK, int G, int EPI>
__global__ __launch_bounds__(G * 256, 4)
void gemm_f32_kernel(const GemmArgs g)
{
    extern __shared__ __align__(16) char lds[];               // [G][2 stages]; at the end [G][4 waves][16][64] sums
    const int tile = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);      // consecutive tiles (of the same rows of A) on one XCD
    if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
    const int m0 = tile / g.tiles_n * GT, n0 = tile % g.tiles_n * GT;
    const int t = threadIdx.x & 255, lane = t & 63;
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), wave = __builtin_amdgcn_readfirstlane(t >> 6);
    char* const mine = lds + group * 2 * STAGE;

    // what the thread fetches of a step: four k of one row of either operand
    const int ra = AK ? t >> 2 : t & 63, ka = (AK ? t & 3 : t >> 6) * 4;
    const int rb = BK ? t >> 2 : t & 63, kb = (BK ? t & 3 : t >> 6) * 4;
    char* const wa = mine + (ka >> 3) * CHUNK + ra * 16 + (ka & 4) * 2;
    char* const wb = mine + OPERAND + (kb >> 3) * CHUNK + rb * 16 + (kb & 4) * 2;
    // and the fragments its wave reads
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const char* const fa = mine + (lane >> 5) * CHUNK + (wm + (lane & 31)) * 16;
    const char* const fb = mine + OPERAND + (lane >> 5) * CHUNK + (wn + (lane & 31)) * 16;

    const int rounds = ((g.K + GK - 1) / GK + 2 * G - 1) / (2 * G) * 2;       // (an even number; steps past the end are zeros)
    const Source<AK> sa(g.A, g.lda, m0 + ra, g.M, ka, g.K);
    const Source<BK> sb(g.B, g.ldb, n0 + rb, g.N, kb, g.K);
    float4 va[2], vb[2];
    auto load = [&](const int round, const int slot) {
        const int k = (round * G + group) * GK;
        va[slot] = sa.fetch(k);
        vb[slot] = sb.fetch(k);
    };
    auto store = [&](const int slot) { split_to_lds(wa + slot * STAGE, va[slot]); split_to_lds(wb + slot * STAGE, vb[slot]); };
    f32x16 acc = {};
    auto multiply = [&](const int slot) {
        bf16x8 a[3], b[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            a[p] = *reinterpret_cast<const bf16x8*>(fa + slot * STAGE + p * PIECE);
            b[p] = *reinterpret_cast<const bf16x8*>(fb + slot * STAGE + p * PIECE);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
    };
    load(0, 0);
    load(1, 1);
    store(0);
    auto step = [&](const int round, const int s) {
        // stage s of this round is written, stage 1 - s (of the round before) is read
        lds_barrier();
        load(round + 2, s);
        multiply(s);
        store(1 - s);
        __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);            // the fragments; then, over and over,
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        // a product,
            __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);       // vector instructions of the split,
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);        // a piece to LDS
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int r = 0; r < rounds; r += 2) {
        step(r, 0);
        step(r + 1, 1);
    }

    // what the epilogue reads, sent for under the groups' exchange (the last row and column in the place of what lies outside; one by one,
    // us: 2048 x 2048 x 512 with a matrix added 38.4, so 32.1, with GELU's derivative 42.4 and 36.9, 3000 x 2048 x 512 60.9 and 56.6, 8192 x 512 x 256 30.1 and 26.4)
    const int n = n0 + wn + (lane & 31);
    auto row = [&](const int q, const int i) { return m0 + wm + 8 * q + 4 * (lane >> 5) + i; };
    float hv[16 / G];
    if constexpr (reads_h<EPI>())
#pragma unroll
        for (int e = 0; e < 16 / G; ++e) hv[e] = g.h[(size_t)min(row((e >> 2) * G + group, e & 3), g.M - 1) * g.ldc + min(n, g.N - 1)];
    // ---- the groups' sums together: group i takes every G-th quad of accumulators of every wave ----
    if (G > 1) {
        float* const red = reinterpret_cast<float*>(lds);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; ++i) red[((group * 4 + wave) * 16 + i) * 64 + lane] = acc[i];
        __syncthreads();
    }
    uint32_t again = 0;                                        // of the lane's 16 elements those that are not finite
#pragma unroll
    for (int e = 0; e < 16 / G; ++e) {
        const int q = (e >> 2) * G + group, i = e & 3, m = row(q, i);
        float v;
        if (G == 1) v = acc[e];
        else {
            const float* red = reinterpret_cast<const float*>(lds) + (wave * 16 + q * 4 + i) * 64 + lane;
            v = red[0];
#pragma unroll
            for (int o = 1; o < G; ++o) v += red[o * 4 * 16 * 64];
        }
        if (m >= g.M || n >= g.N) continue;
        if (fabsf(v) <= 3.4028234e38f) write<EPI>(g, m, n, v * REDUCED, reads_h<EPI>() ? hv[e] : 0.f);
        else again |= 1u << (q * 4 + i);
    }
    if (__builtin_amdgcn_ballot_w64(again != 0) == 0) return;
    // Where a row of A or a column of B holds a NaN so do their elements (a run that has diverged: all of them); the others are summed again.
    const int k0 = lane >> 5 ? g.K / 2 : 0, k1 = lane >> 5 ? g.K : g.K / 2;
    const bool nan_a = any_nan<AK>(g.A, g.lda, m0 + wm + (lane & 31), g.M, k0, k1), nan_b = any_nan<BK>(g.B, g.ldb, n, g.N, k0, k1);
    const uint64_t in_a = __builtin_amdgcn_ballot_w64(nan_a), in_b = __builtin_amdgcn_ballot_w64(nan_b);
    const uint32_t rows_a = (uint32_t)in_a | (uint32_t)(in_a >> 32), cols_b = (uint32_t)in_b | (uint32_t)(in_b >> 32);
    for (; again; again &= again - 1) {
        const int e = __builtin_ctz(again), r = 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3), m = m0 + wm + r;
        write<EPI>(g, m, n, (rows_a >> r | cols_b >> (lane & 31)) & 1 ? __builtin_nanf("") : plain_dot<AK, BK>(g, m, n), reads_h<EPI>() ? g.h[(size_t)m * g.ldc + n] : 0.f);
    }
}

// The same with tiles of 128 x 128, 64 x 64 of them a wave: two thirds of the LDS traffic per product (24 KB read and 12 KB written per 64 x 64 x 16 become 12 and 6) and half of the splitting, which is
// laid between the products.  G groups of four waves share a tile, each with its own steps and stages.  What bounds it: the products (8192 x 2048 x 512 at 1000 to 1060 TFLOP/s of bf16,
// a library product of bf16 reaches 1300), at a tile per compute unit the fill and the epilogue.  Without the order below, split and then products, the odd group the other way
// round: 2048 x 2048 x 512 31.3 us, so 28.8 (64 x 64 tiles 36.3), 8192 tokens with one group 108 and 97 (128).  Loads four steps ahead: 29.5.
constexpr int WT       = 128;
constexpr int WCHUNK   = WT * 16 + 64, WPIECE = 2 * WCHUNK, WOPERAND = 3 * WPIECE, WSTAGE = 2 * WOPERAND;
template <bool AK, bool BK, int G, int EPI>
__global__ __launch_bounds__(G * 256, 2)
void gemm_f32_wide_kernel(const GemmArgs g)
{
    extern __shared__ __align__(16) char lds[];               // [G][2 stages]; at the end [2][4 waves][32][64] sums
    const int tile = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);      // consecutive tiles (of the same rows of A) on one XCD
    if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
    const int m0 = tile / g.tiles_n * WT, n0 = tile % g.tiles_n * WT;
    const int t = threadIdx.x & 255, lane = t & 63, half = lane >> 5, r0 = lane & 31;
    const int group = G > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    char* const mine = lds + group * 2 * WSTAGE;

    // what the thread fetches of a step: four k of two rows, 64 apart, of either operand
    const int ra = AK ? t >> 2 : t & 63, ka = (AK ? t & 3 : t >> 6) * 4;
    const int rb = BK ? t >> 2 : t & 63, kb = (BK ? t & 3 : t >> 6) * 4;
    char* const wa = mine + (ka >> 3) * WCHUNK + ra * 16 + (ka & 4) * 2;
    char* const wb = mine + WOPERAND + (kb >> 3) * WCHUNK + rb * 16 + (kb & 4) * 2;
    // and the fragments its wave reads
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;
    const char* const fa = mine + half * WCHUNK + (wm + r0) * 16;
    const char* const fb = mine + WOPERAND + half * WCHUNK + (wn + r0) * 16;

    const int rounds = ((g.K + GK - 1) / GK + 2 * G - 1) / (2 * G) * 2;       // (an even number; steps past the end are zeros)
    const Source<AK> sa0(g.A, g.lda, m0 + ra, g.M, ka, g.K), sa1(g.A, g.lda, m0 + ra + 64, g.M, ka, g.K);
    const Source<BK> sb0(g.B, g.ldb, n0 + rb, g.N, kb, g.K), sb1(g.B, g.ldb, n0 + rb + 64, g.N, kb, g.K);
    float4 va[2][2], vb[2][2];
    auto load = [&](const int round, const int slot) {
        const int k = (round * G + group) * GK;
        va[slot][0] = sa0.fetch(k); va[slot][1] = sa1.fetch(k);
        vb[slot][0] = sb0.fetch(k); vb[slot][1] = sb1.fetch(k);
    };
    auto store = [&](const int slot) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            split_to_lds(wa + slot * WSTAGE + i * 64 * 16, va[slot][i], WPIECE);
            split_to_lds(wb + slot * WSTAGE + i * 64 * 16, vb[slot][i], WPIECE);
        }
    };
    f32x16 acc[2][2] = {};
    auto multiply = [&](const int slot) {
        bf16x8 a[2][3], b[2][3];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i][p] = *reinterpret_cast<const bf16x8*>(fa + slot * WSTAGE + p * WPIECE + i * 32 * 16);
                b[i][p] = *reinterpret_cast<const bf16x8*>(fb + slot * WSTAGE + p * WPIECE + i * 32 * 16);
            }
        constexpr int P[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][P[p][0]], b[j][P[p][1]], acc[i][j], 0, 0, 0);
    };
    load(0, 0);
    load(1, 1);
    store(0);
    auto step = [&](const int round, const int s) {
        // stage s of this round is written, stage 1 - s (of the round before) is read
        lds_barrier();
        load(round + 2, s);
        multiply(s);
        store(1 - s);
        __builtin_amdgcn_sched_group_barrier(0x100, 12, 0);           // the fragments; then, over and over,
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        // a product,
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);        // vector instructions of the split,
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);        // and every second time a piece to LDS
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int r = 0; r < rounds; r += 2) {
        step(r, 0);
        step(r + 1, 1);
    }

    // (as above)
    float hv[2 / G][32];
    if constexpr (reads_h<EPI>())
#pragma unroll
        for (int i = 0; i < 2 / G; ++i)
#pragma unroll
            for (int e = 0; e < 32; ++e) {
                const int m = m0 + wm + 32 * (G == 2 ? group : i) + 8 * ((e >> 2) & 3) + 4 * half + (e & 3), n = n0 + wn + 32 * (e >> 4) + r0;
                hv[i][e] = g.h[(size_t)min(m, g.M - 1) * g.ldc + min(n, g.N - 1)];
            }

    // ---- the groups' sums together: group i takes the i-th 32 rows of every wave's 64, and hands on the others ----
    if constexpr (G == 2) {
        float* const red = reinterpret_cast<float*>(lds);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) red[((group * 4 + wave) * 32 + j * 16 + e) * 64 + lane] = group ? acc[0][j][e] : acc[1][j][e];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float other = red[(((1 - group) * 4 + wave) * 32 + j * 16 + e) * 64 + lane];
                acc[0][j][e] = (group ? acc[1][j][e] : acc[0][j][e]) + other;
            }
    }
#pragma unroll
    for (int i = 0; i < 2 / G; ++i) {
        const int mw = m0 + wm + 32 * (G == 2 ? group : i);
        uint32_t again = 0;                                    // of the lane's 32 elements those that are not finite
#pragma unroll
        for (int e = 0; e < 32; ++e) {
            const float v = acc[i][e >> 4][e & 15];
            const int m = mw + 8 * ((e >> 2) & 3) + 4 * half + (e & 3), n = n0 + wn + 32 * (e >> 4) + r0;
            if (m >= g.M || n >= g.N) continue;
            if (fabsf(v) <= 3.4028234e38f) write<EPI>(g, m, n, v * REDUCED, reads_h<EPI>() ? hv[i][e] : 0.f);
            else again |= 1u << e;
        }
        if (__builtin_amdgcn_ballot_w64(again != 0) == 0) continue;
        // (as above)
        const int k0 = half ? g.K / 2 : 0, k1 = half ? g.K : g.K / 2;
        const uint64_t in_a = __builtin_amdgcn_ballot_w64(any_nan<AK>(g.A, g.lda, mw + r0, g.M, k0, k1));
        const uint32_t rows_a = (uint32_t)in_a | (uint32_t)(in_a >> 32);
        uint32_t cols_b[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint64_t in_b = __builtin_amdgcn_ballot_w64(any_nan<BK>(g.B, g.ldb, n0 + wn + 32 * j + r0, g.N, k0, k1));
            cols_b[j] = (uint32_t)in_b | (uint32_t)(in_b >> 32);
        }
        for (; again; again &= again - 1) {
            const int e = __builtin_ctz(again), r = 8 * ((e >> 2) & 3) + 4 * half + (e & 3), n = n0 + wn + 32 * (e >> 4) + r0;
            const bool nan = (rows_a >> r | (e >> 4 ? cols_b[1] : cols_b[0]) >> r0) & 1;
            write<EPI>(g, mw + r, n, nan ? __builtin_nanf("") : plain_dot<AK, BK>(g, mw + r, n), reads_h<EPI>() ? g.h[(size_t)(mw + r) * g.ldc + n] : 0.f);
        }
    }
}

// Eight consecutive k of one row, and the three pieces' fragments of them.
struct Raw { float4 lo, hi; };
struct Frags { bf16x8 x[3]; };
__device__ __forceinline__ Frags split(const Raw& r)
{
    float v[8] = {r.lo.x, r.lo.y, r.lo.z, r.lo.w, r.hi.x, r.hi.y, r.hi.z, r.hi.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] *= ENLARGED;
    uint32_t p[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        p[0][i] = pack2(v[2 * i], v[2 * i + 1]);
        const float a = v[2 * i] - low(p[0][i]), b = v[2 * i + 1] - high(p[0][i]);
        p[1][i] = pack2(a, b);
        p[2][i] = pack2(a - low(p[1][i]), b - high(p[1][i]));
    }
    Frags f;
#pragma unroll
    for (int i = 0; i < 3; ++i) f.x[i] = __builtin_bit_cast(bf16x8, make_uint4(p[i][0], p[i][1], p[i][2], p[i][3]));
    return f;
}

// A lane's share of an operand whose rows run across k: columns lane % 32 and 32 further, k from 8 (lane / 32) on.
struct RowSource {
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t at[2], pitch;                                     // of the lane's columns at its first k; bytes per k
    __device__ __forceinline__ RowSource(const float* X, const int ld, const int col, const int cols, const int k, const int K)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc((void*)X, 0, (uint32_t)(((size_t)(K - 1) * ld + cols) * 4), 0x00020000)), pitch((uint32_t)ld * 4u)
    {
#pragma unroll
        for (int i = 0; i < 2; ++i) at[i] = col + 32 * i < cols ? (uint32_t)(col + 32 * i) * 4u + (uint32_t)k * pitch : 0x80000000u;
    }
    __device__ __forceinline__ void fetch(const int k0, Raw (&r)[2]) const
    {
        // (rows of k past K lie behind the end; so does what a column past the last reads)
        const uint32_t o = (uint32_t)k0 * pitch;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, at[i] + o + (uint32_t)j * pitch, 0, 0));
            r[i].lo = make_float4(v[0], v[1], v[2], v[3]); r[i].hi = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
};

// Accumulators e0 to e0 + COUNT of a 64 x 64 tile at (m0, n0), a lane's sums of each.
template <int COUNT>
__device__ __forceinline__ void finish_rows(const GemmArgs& g, const int m0, const int n0, const int e0, const float (&v)[COUNT])
{
    const int lane = threadIdx.x & 63, r0 = lane & 31, half = lane >> 5;
    auto row = [&](const int e) { return 32 * (e >> 5) + 8 * ((e >> 2) & 3) + 4 * half + (e & 3); };       // of accumulator e, in the tile
    auto column = [&](const int e) { return n0 + 32 * ((e >> 4) & 1) + r0; };
    uint32_t again = 0;                                        // of the lane's elements those that are not finite
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
        const int e = e0 + i;
        if (m0 + row(e) >= g.M || column(e) >= g.N) continue;
        if (fabsf(v[i]) <= 3.4028234e38f) write<PROTEUS_GEMM_F32>(g, m0 + row(e), column(e), v[i] * REDUCED);
        else again |= 1u << i;
    }
    if (__builtin_amdgcn_ballot_w64(again != 0) == 0) return;
    // (as above)
    uint32_t rows_a[2], cols_b[2];
    const int k0 = half ? g.K / 2 : 0, k1 = half ? g.K : g.K / 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint64_t in_a = __builtin_amdgcn_ballot_w64(any_nan<false>(g.A, g.lda, m0 + 32 * i + r0, g.M, k0, k1));
        const uint64_t in_b = __builtin_amdgcn_ballot_w64(any_nan<false>(g.B, g.ldb, n0 + 32 * i + r0, g.N, k0, k1));
        rows_a[i] = (uint32_t)in_a | (uint32_t)(in_a >> 32);
        cols_b[i] = (uint32_t)in_b | (uint32_t)(in_b >> 32);
    }
    for (; again; again &= again - 1) {
        const int e = e0 + __builtin_ctz(again), j = (e >> 4) & 1;
        const bool nan = ((e >> 5 ? rows_a[1] : rows_a[0]) >> (row(e) & 31) | (j ? cols_b[1] : cols_b[0]) >> r0) & 1;
        write<PROTEUS_GEMM_F32>(g, m0 + row(e), column(e), nan ? __builtin_nanf("") : plain_dot<false, false>(g, m0 + row(e), column(e)));
    }
}

// Where tile `tile` lies: consecutive ones are those of a line along the shorter side of the matrix, so that an XCD's share is as square as may be
// (512 x 2048 of 2048 tokens 28.5 us, with lines along the longer side 36.5).
__device__ __forceinline__ void tile_at(const GemmArgs& g, const int tile, int& m0, int& n0)
{
    const int tiles_m = g.tiles / g.tiles_n;
    const bool wide = tiles_m < g.tiles_n;
    m0 = (wide ? tile % tiles_m : tile / g.tiles_n) * GT;
    n0 = (wide ? tile / tiles_m : tile % g.tiles_n) * GT;
}

template <int W>
__global__ __launch_bounds__(W * 64, 2)
void gemm_f32_rows_kernel(const GemmArgs g)
{
    extern __shared__ __align__(16) float red[];              // [W][64 accumulators][64 lanes]
    // consecutive tiles of one share of K on one XCD: 512 x 512 x 8192 in four shares, whose operands then come to one or two
    // of the eight caches, 32 us, with the shares of a tile on one XCD 42
    const int unit = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3), share = unit / g.tiles, tile = unit % g.tiles;
    if (share >= g.shares) return;
    int m0, n0;
    tile_at(g, tile, m0, n0);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = lane & 31, half = lane >> 5;

    const RowSource sa(g.A, g.lda, m0 + r0, g.M, 8 * half, g.K);
    const RowSource sb(g.B, g.ldb, n0 + r0, g.N, 8 * half, g.K);
    // (a share but the last is an even number of rounds: what is past its end, the next one's, is loaded but not multiplied)
    const int begin = share * g.steps, steps = min((g.K + GK - 1) / GK - begin, g.steps), rounds = steps > wave ? (steps - wave + W - 1) / W : 0;         // this wave's
    Raw ra[2][2], rb[2][2];
    Frags a[2][2], b[2][2];
    f32x16 acc[2][2] = {};
    auto load = [&](const int round, const int s) { const int k0 = (begin + round * W + wave) * GK; sa.fetch(k0, ra[s]); sb.fetch(k0, rb[s]); };      // (zeros past the end)
    auto step = [&](const int round, const int s) {
        // send for the step after the next; split the next under this step's products
        load(round + 2, s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i) { a[1 - s][i] = split(ra[1 - s][i]); b[1 - s][i] = split(rb[1 - s][i]); }
        constexpr int P[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][i].x[P[p][0]], b[s][j].x[P[p][1]], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        // a product,
            __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);        // vector instructions
        }
    };
    if (rounds > 0) {
        load(0, 0);
        load(1, 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) { a[0][i] = split(ra[0][i]); b[0][i] = split(rb[0][i]); }
        for (int r = 0; r < rounds; r += 2) {
            step(r, 0);
            step(r + 1, 1);                                    // (past the last round: zeros)
        }
    }

    // ---- the waves' sums together: wave w takes accumulators w (64 / W) to (w + 1) (64 / W) ----
    float v[64 / W];
#pragma unroll
    for (int e = 0; e < 64; ++e) red[(wave * 64 + e) * 64 + lane] = acc[e >> 5][(e >> 4) & 1][e & 15];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 64 / W; ++e) {
        v[e] = red[(wave * (64 / W) + e) * 64 + lane];
#pragma unroll
        for (int w = 1; w < W; ++w) v[e] += red[(w * 64 + wave * (64 / W) + e) * 64 + lane];
    }
    if (g.shares > 1) {
        float* to = g.part + ((size_t)share * g.tiles + tile) * (GT * GT) + wave * (64 / W) * 64 + lane;
#pragma unroll
        for (int e = 0; e < 64 / W; ++e) to[e * 64] = v[e];
        return;
    }
    finish_rows<64 / W>(g, m0, n0, wave * (64 / W), v);
}

// The shares' sums of a tile together, in their order: W sixteenths of a tile per workgroup, four accumulators per wave.  With eight waves the workgroups behind those make column sums; without any,
// four waves are the faster ones (shares of 88 x 48 x 7834 in all 13.5 us with eight, 12.8 with four).
template <int W>
__global__ __launch_bounds__(W * 64)
void gemm_f32_rows_sum_kernel(const PendingSums sums)
{
    static_assert(proteus_train::CS_BLOCK == 512, "eight waves");
    constexpr int PER = 16 / W;                                    // workgroups per tile
    const int id = (int)blockIdx.x;
    if constexpr (W * 64 == proteus_train::CS_BLOCK) {
        __shared__ float red[proteus_train::CS_BLOCK / 64][proteus_train::CS_COLS];
        const int behind = id - sums.first[sums.count] * PER;
        if (behind >= 0) {
            int c = 0;
            while (behind >= sums.first_column[c + 1]) ++c;
            const proteus_train::ColumnSums& of = sums.columns[c];
            proteus_train::column_sums(of.a, of.out, 0, of.rows, of.cols, behind - sums.first_column[c], red);
            return;
        }
    }
    int p = 0;
    while (id / PER >= sums.first[p + 1]) ++p;
    const GemmArgs& g = sums.product[p];
    const int tile = id / PER - sums.first[p], e0 = (id % PER) * (W * 4) + (threadIdx.x >> 6) * 4;
    const float* from = g.part + (size_t)tile * (GT * GT) + e0 * 64 + (threadIdx.x & 63);
    const size_t pitch = (size_t)g.tiles * (GT * GT);
    float v[4] = {};
#pragma unroll 4
    for (int s = 0; s < g.shares; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += from[s * pitch + i * 64];
    int m0, n0;
    tile_at(g, tile, m0, n0);
    finish_rows<4>(g, m0, n0, e0, v);
}

// Groups of gemm_f32_wide_kernel, 0: tiles of 64 x 64.  Us, M x N x K (tiles of 128 x 128), 64 x 64 / 128 x 128.
// Two groups while the tiles leave a compute unit one each and few idle, later where the epilogue is long, since nothing runs under that of a lone workgroup: 1536 x 1536 x 512 (144) 25.2 / 25.7, 2048 x 1280
// x 512 (160) 25.8 / 26.0, 5000 x 512 x 2048 (160) 88 / 72, 4096 x 768 x 768 (192) 39 / 35, 6400 x 512 x 512 (200) 31.8 / 27.7, 4096 x 1024 x 1024 (256) 64 / 50, 8192 x 512 x 2048 (256) 123 / 90; 4096 x 512 x 2048 (128)
// 59 / 70; with GELU and with its derivative 1536 x 2048 x 512 (192) 32.0 / 32.0 and 31.9 / 33.3, 1792 x 2048 (224) 37.3 / 33.5 and 38.0 / 34.5, 2048 x 2048 (256) 39.1 / 35.2 and 39.6 / 36.3.
// One group where there are more tiles of 64 x 64 than the chip holds at once (six per compute unit): 4096 x 1536 x 512 (384) 50 / 53, 4480 x 1536 (420) 57 / 55, 7000 x 876 x 884 (385) 103 / 79, 16384 x 512 x 2048 (512)
// 234 / 182, 8192 x 1536 x 512 (768) 92 / 77; GELU 3584 x 2048 x 512 (448) 64.3 / 64.3, 4600 x 2048 (576) 81.0 / 82.8, 5632 x 2048 (704) 97 / 88, 8192 x 2048 (1024) 138 / 119.
// Where the epilogue reads a matrix, which it keeps in registers, only two workgroups instead of three share a compute unit, and rounds of 512 that end nearly empty lose: a matrix added 14400 x 512 x 2048 (452)
// 219 / 183, 18000 x 512 x 512 (564) 70 / 85, 20000 x 512 x 2048 (628) 286 / 290, 24000 x 512 x 512 (752) 90 / 89, x 2048 344 / 309, 16000 x 768 x 768 (750) 130 / 121, 32768 x 512 x 512 (1024) 120 / 116, 11000 x 1536 x 512
// (1032) 10 % more; GELU's derivative 4096 x 2048 x 512 (512) 72 / 72, 2048 x 4096 x 1024 (512) 131 / 120, 5632 x 2048 x 512 (704) 98 / 107, 7200 x 2048 (912) 128 / 132, 3600 x 4096 x 1024 (928) 229 / 213, 8192 x 2048 x 512
// (1024) 138 / 133, 9000 x 2048 (1136) 154 / 163, 10000 x 2048 (1264) 169 / 166, 16384 x 2048 (2048) 279 / 272.
// Not for a short K: 13000 x 512 x 256 and 4992 x 1536 x 256 3 to 9 % more.  And only where a fifth of the tiles' area at most lies outside (counted in tiles of 64): 20480 x 64 x 512 17 / 24, 30000 x 64 x 2048 60 / 77, 65536 x
// 64 x 512 37 / 53, 129 x 10244 x 512 19 / 27, 40000 x 192 x 512 63 / 66 and with a matrix added 61 / 79, 30000 x 320 x 512 76 / 71.
int wide_groups(int M, int N, int K, int epilogue)
{
    if (K < 512) return 0;
    const int64_t tiles = ((M + (int64_t)WT - 1) / WT) * ((N + (int64_t)WT - 1) / WT), small = ((M + (int64_t)GT - 1) / GT) * ((N + (int64_t)GT - 1) / GT);
    if (5 * small < 16 * tiles) return 0;
    const bool grad = epilogue == PROTEUS_GEMM_GELU_GRAD, add = epilogue == PROTEUS_GEMM_ADD;
    if (tiles <= 256) return tiles >= (grad || epilogue == PROTEUS_GEMM_GELU ? 216 : 160) ? 2 : 0;
    if (small <= 6 * 256) return 0;
    if (!grad && !add) return 1;
    const double filled = (double)tiles / (double)((tiles + 511) / 512 * 512);
    return filled >= (add ? 0.9 : 0.95) || (K >= (add ? 768 : 1024) && filled >= 0.7) || (tiles > 1200 && filled >= 0.8) ? 1 : 0;
}

template <bool AK, bool BK, int EPI>
int gemm_go(GemmArgs g, hipStream_t st, PendingSums* sums = nullptr)
{
    const int tm = (g.M + GT - 1) / GT;
    g.tiles_n = (g.N + GT - 1) / GT;
    g.tiles   = tm * g.tiles_n;
    g.per_xcd = (g.tiles * g.shares + 7) / 8;
    const dim3 grid((unsigned)g.per_xcd * 8);
    if constexpr (!AK) {
        // Waves per tile, of which a SIMD holds two: 8 while there is a tile at most per compute unit, 4 up to two or for several rounds, 2 for a single round of
        // four.  Us with 2 / 4 / 8, 512 and 2048 tokens: 256 tiles 17.0 / 11.8 / 11.1 and 49 / 31 / 29, 288 25.0 / 16.7 / 19.7 and 79 / 47 / 51, 768 28.4 / 25.6 / 29.8 and 91 / 79 / 84,
        // 896 29.9 / 31.3 / 38.2 and 95 / 98 / 105, 1024 31.6 / 32.7 / 38.9 and 103 / 104 / 111, 2048 64 / 61 / 76 and 209 / 203 / 221.
#define GO(W_) hipLaunchKernelGGL((gemm_f32_rows_kernel<W_>), grid, dim3(W_ * 64), (size_t)W_ * 64 * 64 * 4, st, g)
        if (g.tiles <= 256)                        GO(8);
        else if (g.tiles > 768 && g.tiles <= 1024) GO(2);
        else                                       GO(4);
#undef GO
        if (g.shares > 1) {
            PendingSums own;
            PendingSums& p = sums ? *sums : own;
            p.product[p.count] = g;
            p.first[p.count + 1] = p.first[p.count] + g.tiles;
            ++p.count;
            if (!sums) return gemm_sums(own, st);
        }
    } else {
        // Groups per tile, of which a compute unit holds four: as many as its tiles leave room for in one round.  Us with 1 / 2 / 4, K = 512 and 2048, X W^T: 256 tiles
        // 16.2 / 13.1 / 10.8 and 51 / 40 / 33, 288 18.7 / 16.6 / 18.9 and 61 / 52 / 57, 512 20.8 / 19.0 / 19.8 and 70 / 63 / 64, 544 25.4 / 26.7 / 27.7 and 88 / 90 / 88, 1024 35.4 / 35.0 / 37.6 and
        // 128 / 122 / 125, 2048 66 / 67 / 73 and 245 / 237 / 250; X W the same but for 1024 and 2048 tiles, K = 2048, 130 / 127 / 135 and 247 / 250 / 270.
#define GO(G_) do { \
            constexpr size_t sums = (G_) > 1 ? (size_t)(G_) * 4 * 16 * 64 * 4 : 0; \
            hipLaunchKernelGGL((gemm_f32_kernel<AK, BK, G_, EPI>), grid, dim3(G_ * 256), G_ * 2 * STAGE > sums ? G_ * 2 * STAGE : sums, st, g); \
        } while (0)
        if (const int groups = wide_groups(g.M, g.N, g.K, EPI)) {
            g.tiles_n = (g.N + WT - 1) / WT;
            g.tiles   = (g.M + WT - 1) / WT * g.tiles_n;
            g.per_xcd = (g.tiles + 7) / 8;
            auto kern = groups == 2 ? gemm_f32_wide_kernel<AK, BK, 2, EPI> : gemm_f32_wide_kernel<AK, BK, 1, EPI>;
            const size_t bytes = (size_t)groups * 2 * WSTAGE;
            if (bytes > 64 * 1024) {      // (per device, cheap: set on every call)
                const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
                if (attr != hipSuccess) return (int)attr;
            }
            hipLaunchKernelGGL(kern, dim3((unsigned)g.per_xcd * 8), dim3(groups * 256), bytes, st, g);
            return (int)hipGetLastError();
        }
        if (g.tiles > 512)      GO(1);
        else if (g.tiles > 256) GO(2);
        else                    GO(4);
#undef GO
    }
    return (int)hipGetLastError();
}

// Gradients of weights: shares of K for workgroups of their own where the tiles leave compute units idle, so that at most 256 workgroups of 8 waves, one
// per compute unit, are launched; at least 256 of K each (a round of 8 waves, two by two) and at most 32 of them, whose sums the second launch
// adds up, and only where a workgroup is spared 1536 of K: that launch takes 4 us of the device and 3 of the host, which is what bounds a training step of fewer
// tokens (2 x 600, d_model 256, 3 layers 1025 us, from 768 spared on and a launch per product 1065).  One, shares of 256, 512 and 1024, and the library, us:
// 128 x 128 of 2048 tokens 23 / 9.9 / 11.8 / 16 / 14, of 8192 75 / 14 / 14 / 17 / 45; 512 x 512 of 2048 24 / 14.3 / 14.3 / 18 / 15, of 8192 77 / 33 / 33 / 33 / 55;
// 256 x 1024 of 1024 15.2 / 12.5 / 13.6 / 15.1 / 9.7; 64 x 64 of 32768 283 with one, 44, 33 and 25 with 128, 64 and 32, library 117; 128 x 128 of 700 11.9 / 11.7 (two shares).
struct Shares { int number, steps; };
Shares rows_shares(int M, int N, int K)
{
    constexpr int UNIT = 2 * 8, MOST = 32;
    const int64_t tiles = (int64_t)((M + (int64_t)GT - 1) / GT) * ((N + (int64_t)GT - 1) / GT);
    const int steps = (K + GK - 1) / GK, units = (steps + UNIT - 1) / UNIT, most = tiles > 128 ? 1 : min((int)(256 / tiles), MOST);
    const int per = (units + most - 1) / most * UNIT;
    if (K - per * GK < 1536) return {1, steps};
    return {(steps + per - 1) / per, per};
}

bool off16(const void* p) { return ((uintptr_t)p & 15) != 0; }

}  // namespace

extern "C" size_t proteus_gemm_f32_workspace_bytes(int M, int N, int K, int form)
{
    if (form != PROTEUS_GEMM_TN || M <= 0 || N <= 0 || K <= 0 || K >= (1 << 29)) return 0;      // (2 GiB of a matrix are refused)
    const Shares c = rows_shares(M, N, K);
    return c.number > 1 ? (size_t)c.number * ((M + GT - 1) / GT) * ((N + GT - 1) / GT) * (GT * GT * 4) : 0;
}

extern "C" int proteus_gemm_f32(const float* A, const float* B, const float* bias, const float* h, void* C, float* H,
                                int M, int N, int K, int lda, int ldb, int ldc, int form, int epilogue, void* stream)
{
    return proteus_gemm_f32_ws(A, B, bias, h, C, H, M, N, K, lda, ldb, ldc, form, epilogue, nullptr, 0, stream);
}

namespace {

int gemm(const float* A, const float* B, const float* bias, const float* h, void* C, float* H, int M, int N, int K, int lda, int ldb, int ldc,
         int form, int epilogue, void* ws, size_t ws_bytes, PendingSums* sums, void* stream)
{
    if (!A || !B || !C || (epilogue == PROTEUS_GEMM_GELU && !H) || ((epilogue == PROTEUS_GEMM_GELU_GRAD || epilogue == PROTEUS_GEMM_ADD) && !h)) return PROTEUS_ERR_NULL_POINTER;
    if (form < 0 || form > PROTEUS_GEMM_TN || epilogue < 0 || epilogue > PROTEUS_GEMM_ADD || (form == PROTEUS_GEMM_TN && epilogue != PROTEUS_GEMM_F32)
        || (form == PROTEUS_GEMM_NN && epilogue == PROTEUS_GEMM_GELU) || (form == PROTEUS_GEMM_NT && (epilogue == PROTEUS_GEMM_BF16 || epilogue == PROTEUS_GEMM_GELU_GRAD)))
        return PROTEUS_ERR_UNSUPPORTED;
    if (M <= 0 || N <= 0 || K <= 0 || ldc < N || lda < (form == PROTEUS_GEMM_TN ? M : K) || ldb < (form == PROTEUS_GEMM_NT ? K : N)) return PROTEUS_ERR_BAD_SHAPE;
    // (tiles are numbered in 32 bits)
    if ((int64_t)((M + (int64_t)GT - 1) / GT) * ((N + (int64_t)GT - 1) / GT) > (1 << 30)) return PROTEUS_ERR_TOO_LARGE;
    // (buffer offsets, those of the steps past the end among them)
    const int64_t bytes_a = ((int64_t)(form == PROTEUS_GEMM_TN ? K : M) + 512) * lda * 4, bytes_b = ((int64_t)(form == PROTEUS_GEMM_NT ? N : K) + 512) * ldb * 4;
    if (bytes_a >= (1LL << 31) || bytes_b >= (1LL << 31)) return PROTEUS_ERR_TOO_LARGE;
    // rows that are read 16 bytes at a time
    if (off16(A) || off16(B) || off16(C)) return PROTEUS_ERR_BAD_ALIGNMENT;
    if (form != PROTEUS_GEMM_TN && (K % 4 || lda % 4)) return PROTEUS_ERR_BAD_SHAPE;
    if (form == PROTEUS_GEMM_NT && ldb % 4) return PROTEUS_ERR_BAD_SHAPE;
    Shares cut = {1, (K + GK - 1) / GK};
    if (ws && form == PROTEUS_GEMM_TN) {
        if (off16(ws)) return PROTEUS_ERR_BAD_ALIGNMENT;
        const size_t need = proteus_gemm_f32_workspace_bytes(M, N, K, form);
        if (need && ws_bytes >= need) cut = rows_shares(M, N, K);
    }
    const GemmArgs g = {A, B, bias, h, C, H, M, N, K, lda, ldb, ldc, 0, 0, 0, static_cast<float*>(ws), cut.number, cut.steps};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // (what the training step asks for; nothing else is built)
#define GO(AK_, BK_, E_) case E_: return gemm_go<AK_, BK_, E_>(g, st)
    if (form == PROTEUS_GEMM_NN) switch (epilogue) {
        GO(true, false, PROTEUS_GEMM_F32);
        GO(true, false, PROTEUS_GEMM_BF16);
        GO(true, false, PROTEUS_GEMM_GELU_GRAD);
        GO(true, false, PROTEUS_GEMM_ADD);
    }
    else if (form == PROTEUS_GEMM_NT) switch (epilogue) {
        GO(true, true, PROTEUS_GEMM_F32);
        GO(true, true, PROTEUS_GEMM_GELU);
        GO(true, true, PROTEUS_GEMM_ADD);
    }
    else return gemm_go<false, false, PROTEUS_GEMM_F32>(g, st, sums);
#undef GO
    return PROTEUS_ERR_UNSUPPORTED;
}

}  // namespace

extern "C" int proteus_gemm_f32_ws(const float* A, const float* B, const float* bias, const float* h, void* C, float* H,
                                   int M, int N, int K, int lda, int ldb, int ldc, int form, int epilogue, void* ws, size_t ws_bytes, void* stream)
{
    return gemm(A, B, bias, h, C, H, M, N, K, lda, ldb, ldc, form, epilogue, ws, ws_bytes, nullptr, stream);
}

int proteus_gemm::gemm_begin(const float* A, const float* B, float* C, int M, int N, int K, int lda, int ldb, int ldc, void* ws, size_t ws_bytes, PendingSums& sums, void* stream)
{
    return gemm(A, B, nullptr, nullptr, C, nullptr, M, N, K, lda, ldb, ldc, PROTEUS_GEMM_TN, PROTEUS_GEMM_F32, ws, ws_bytes, sums.count < PendingSums::MOST ? &sums : nullptr, stream);
}

int proteus_gemm::gemm_sums(PendingSums& sums, void* stream)
{
    const int tiles = sums.first[sums.count], columns = sums.first_column[sums.column_count];
    if (tiles + columns == 0) return PROTEUS_OK;
    if (columns) hipLaunchKernelGGL(gemm_f32_rows_sum_kernel<8>, dim3((unsigned)(tiles * 2 + columns)), dim3(512), 0, reinterpret_cast<hipStream_t>(stream), sums);
    else         hipLaunchKernelGGL(gemm_f32_rows_sum_kernel<4>, dim3((unsigned)(tiles * 4)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), sums);
    sums.count = sums.column_count = 0;
    return (int)hipGetLastError();
}
