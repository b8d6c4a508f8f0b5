// Matrix products of the encoder's inference: C = act(A B^T + bias), bf16 operands and result, fp32 sums (gfx950).
//
// A workgroup makes a BM x BN tile of C and steps through K by 64.  Both operands have k contiguous and travel global -> LDS directly
// (buffer_load ... lds, 16 bytes a lane) as rows of 128 bytes whose 16-byte chunks are XOR-swizzled, STAGES - 1 steps ahead, each stage an LDS object of its own
// (so that the compiler sees that a read of one does not wait for loads into another).  Bias and GELU are added to the fp32 sums, which are then rounded once.
//
// What bounds it: LDS at 64 x 64 of C per wave (16 KB read per 128 clocks of matrix instructions and compute unit, its whole rate), a quarter less at 128 x 64; and the
// rounds of workgroups (one to three of them on a compute unit).  8192 tokens, d_model 512, us, the library's product and torch's GELU / this: QKV 24 to 27 / 18.9, output 13 / 8.4, feed-forward
// 39.5 / 27.7 and 21.7 / 20.8; a call costs the host 3, the library's 18 to 21.
// Where K is long and there are many rows the library is ahead (10000 x 512 x 2048 24.4 / 29.7, 32768 49 / 59, 65536 99 / 132; 4096 x 2304 x 768 19.5 / 23.7, 8192 x 3072 x 1024 53 / 59), by less than
// the layer's other launches gain up to the sizes that encoder.py names.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "proteus_hip.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float  f32x2  __attribute__((ext_vector_type(2)));
typedef float  f32x16 __attribute__((ext_vector_type(16)));

constexpr int HK = 64;                              // k of a step: rows of 128 bytes in LDS
constexpr uint32_t OUTSIDE = 0x80000000u;           // beyond any buffer here: reads as zeros

struct Args {
    const uint16_t *A, *B, *bias;
    uint16_t* C;
    int M, N, K;
    long lda, ldb, ldc;
    int tiles_n, tiles, per_xcd;
};

#define HB_LDS(T, p) ((__attribute__((address_space(3))) T*)(p))

// chunk c of row r lies at slot c ^ swizzle(r): 16 consecutive rows' reads of one chunk touch all 64 banks once
__device__ __forceinline__ int swizzle(const int r) { return (r >> 1) & 7; }

__device__ __forceinline__ uint32_t pack2(const float a, const float b)
{
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
__device__ __forceinline__ float low(const uint32_t w)  { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float high(const uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// x Phi(x) with Phi(-|x|) = erfc(|x| / sqrt 2) / 2 by Abramowitz & Stegun 7.1.26 (absolute error 1.5e-7, and the factor exp(-x^2 / 2) keeps the
// tail's relative error small): a third of erff's instructions.
__device__ __forceinline__ float gelu(const float x)
{
    const float ax = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(ax, 0.3275911f * 0.70710678f, 1.0f));
    float p = __builtin_fmaf(t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
    p = __builtin_fmaf(t, p, 0.5f * 1.421413741f);
    p = __builtin_fmaf(t, p, 0.5f * -0.284496736f);
    p = __builtin_fmaf(t, p, 0.5f * 0.254829592f) * t;
    const float tail = p * __builtin_amdgcn_exp2f(x * x * (-0.5f * 1.44269504f));
    const float r = __builtin_fmaf(-ax, tail, fmaxf(x, 0.0f));
    return x > 40.0f ? x : r;                       // (infinity; NaN stays NaN through ax)
}

// BM x BN of C by WM x WN waves
template <int BM, int BN, int WM, int WN, int STAGES, bool GELU>
__global__ __launch_bounds__(WM * WN * 64, 1)
void gemm_bf16_kernel(const Args g)
{
    constexpr int WAVES = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32;       // 32 x 32 tiles of a wave
    constexpr int STAGE = (BM + BN) * 128, LOADS = (BM + BN) / 8 / WAVES;      // bytes; loads of a wave per stage, of 8 rows each
    constexpr int PITCH = TN * 64 + 16;                                        // of a row of a wave's tile of C in LDS, bytes
    static_assert((BM + BN) % (8 * WAVES) == 0 && BM % 8 == 0, "whole loads");
    __shared__ __align__(1024) unsigned char s0[STAGE];
    __shared__ __align__(1024) unsigned char s1[STAGE];
    __shared__ __align__(1024) unsigned char s2[STAGES > 2 ? STAGE : 16];
    __shared__ __align__(1024) unsigned char s3[STAGES > 3 ? STAGE : 16];

    const int tile = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);         // consecutive tiles (of the same rows of A) on one XCD
    if ((int)(blockIdx.x >> 3) >= g.per_xcd || tile >= g.tiles) return;
    const int m0 = tile / g.tiles_n * BM, n0 = tile % g.tiles_n * BN;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5, col = lane & 31;

    // ---- loads: a wave's load i fills rows 8 (i WAVES + wave) .. + 7 of the stage (A's rows, then B's); lane l asks for the chunk that belongs in slot l % 8 ----
    const int rows_a = min(BM, g.M - m0), rows_b = min(BN, g.N - n0);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)(g.A + (size_t)m0 * g.lda), 0, (int)(((rows_a - 1) * g.lda + g.K) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)(g.B + (size_t)n0 * g.ldb), 0, (int)(((rows_b - 1) * g.ldb + g.K) * 2), 0x00020000);
    uint32_t at[LOADS];
    int chunk[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = 8 * (i * WAVES + wave) + (lane >> 3);
        const bool is_a = 8 * i * WAVES < BM && row < BM;
        const int r = is_a ? row : row - BM;
        chunk[i] = (lane & 7) ^ swizzle(row);
        const bool ok = is_a ? r < rows_a : r < rows_b;
        at[i] = ok ? (uint32_t)((r * (is_a ? g.lda : g.ldb) + 8 * chunk[i]) * 2) : OUTSIDE;
    }
    auto issue = [&](const int step, unsigned char* to) {
        const int k0 = step * HK;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const bool is_a = 8 * (i * WAVES + wave) < BM;                     // (the same for a whole wave)
            const uint32_t o = k0 + 8 * chunk[i] < g.K ? at[i] + (uint32_t)k0 * 2u : OUTSIDE;
            unsigned char* d = to + 1024 * (i * WAVES + wave);
            if (is_a) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, HB_LDS(void, d), 16, o, 0, 0, 0);
            else      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, HB_LDS(void, d), 16, o, 0, 0, 0);
        }
    };
    // ---- fragments: row of the operand, chunk 2 ks + half ----
    const int wm = wave / WN * (TM * 32), wn = wave % WN * (TN * 32);
    f32x16 acc[TM][TN] = {};
    auto multiply = [&](const unsigned char* from) {
#pragma unroll
        for (int ks = 0; ks < HK / 16; ++ks) {
            bf16x8 a[TM], b[TN];
            const int slot = ((2 * ks + half) ^ swizzle(col)) * 16;            // (32 rows further swizzle alike)
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const bf16x8*>(from + (wm + 32 * i + col) * 128 + slot);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = *reinterpret_cast<const bf16x8*>(from + (BM + wn + 32 * j + col) * 128 + slot);
            // rows of the accumulator are columns of C, so that a lane ends up with four of them side by side
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
        }
    };
    const int steps = (g.K + HK - 1) / HK;
    auto round = [&](const int step, unsigned char* mine, unsigned char* next) {
        // The oldest stage in flight has landed for every wave, and everybody has read the one before it: the products of the last fragments may still
        // be to come behind the barrier, so that their reads are waited for here (without that a stage was written over before it was read).
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((STAGES - 2) * LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(step + STAGES - 1, next);                                        // (past the end: zeros)
        // Two stages: the loads leave before the products, not behind them, where the compiler puts them and where the next step waits for all of
        // their way; the fragments of 16 k are read under the products of the 16 before.  Us, left alone / so: 8192 x 2048 x 512 (GELU) 29.6 / 27.3, 8192 x 1536 x 512 19.0 / 18.0, 6000 x 1536 x
        // 512 16.1 / 15.3, 12288 x 2304 x 768 50 / 45, 65536 x 2048 x 512 228 / 207.  (Three steps ahead there is no hurry, and the reads come first: 2048 x 512 x 2048 8.4 / 9.5.)
        if constexpr (STAGES == 2) __builtin_amdgcn_sched_barrier(0);
        multiply(mine);
        if constexpr (STAGES == 2) {
            constexpr int READS = TM + TN, PRODUCTS = TM * TN, PAIRS = READS < PRODUCTS ? READS : PRODUCTS;
            __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
#pragma unroll
            for (int ks = 1; ks < HK / 16; ++ks) {
#pragma unroll
                for (int i = 0; i < PAIRS; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);         // a product,
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);         // a fragment
                }
                if (READS > PAIRS)    __builtin_amdgcn_sched_group_barrier(0x100, READS - PAIRS, 0);
                if (PRODUCTS > PAIRS) __builtin_amdgcn_sched_group_barrier(0x008, PRODUCTS - PAIRS, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, PRODUCTS, 0);
        }
    };
    issue(0, s0);
    if (STAGES > 2) issue(1, s1);
    if (STAGES > 3) issue(2, s2);
    for (int s = 0; s < steps; s += STAGES) {                                  // (steps past the end multiply zeros: without branches the compiler's own waits stay exact)
        if constexpr (STAGES == 2) { round(s, s0, s1); round(s + 1, s1, s0); }
        if constexpr (STAGES == 3) { round(s, s0, s2); round(s + 1, s1, s0); round(s + 2, s2, s1); }
        if constexpr (STAGES == 4) { round(s, s0, s3); round(s + 1, s1, s0); round(s + 2, s2, s1); round(s + 3, s3, s2); }
    }
    // ---- the tile through LDS, so that rows leave in whole lines ----
    float bias[TN][4][4];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint2 b = g.bias ? *reinterpret_cast<const uint2*>(g.bias + min(n0 + wn + 32 * j + 8 * q + 4 * half, g.N - 4)) : make_uint2(0u, 0u);
            bias[j][q][0] = low(b.x); bias[j][q][1] = high(b.x); bias[j][q][2] = low(b.y); bias[j][q][3] = high(b.y);
        }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                           // (zeros past the end still on their way)
    __syncthreads();
    constexpr int PER = STAGE / (32 * PITCH) < WAVES ? STAGE / (32 * PITCH) : WAVES;      // waves whose 32 rows fit one stage
    static_assert(PER * 2 >= WAVES, "two stages hold a block of rows of every wave");
    unsigned char* const own = wave < PER ? s0 + wave * (32 * PITCH) : s1 + (wave - PER) * (32 * PITCH);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * q + e] + bias[j][q][e];
                if (GELU)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = gelu(v[e]);
                *reinterpret_cast<uint2*>(own + col * PITCH + (32 * j + 8 * q + 4 * half) * 2) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
            }
        __builtin_amdgcn_wave_barrier();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                     // (the wave's own rows: no other wave reads them)
        constexpr int CPR = TN * 4, RPI = 64 / CPR;                            // 16-byte chunks of a row, rows an instruction
#pragma unroll
        for (int r = 0; r < 32; r += RPI) {
            const int row = r + lane / CPR, c = lane % CPR, m = m0 + wm + 32 * i + row, n = n0 + wn + 8 * c;
            const uint4 v = *reinterpret_cast<const uint4*>(own + row * PITCH + c * 16);
            if (m < g.M && n < g.N) *reinterpret_cast<uint4*>(g.C + (size_t)m * g.ldc + n) = v;
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

template <int BM, int BN, int WM, int WN, int STAGES>
int go(Args g, const bool gelu, hipStream_t st)
{
    g.tiles_n = (g.N + BN - 1) / BN;
    g.tiles   = (g.M + BM - 1) / BM * g.tiles_n;
    g.per_xcd = (g.tiles + 7) / 8;
    const dim3 grid((unsigned)g.per_xcd * 8), block(WM * WN * 64);
    if (gelu) hipLaunchKernelGGL((gemm_bf16_kernel<BM, BN, WM, WN, STAGES, true>), grid, block, 0, st, g);
    else      hipLaunchKernelGGL((gemm_bf16_kernel<BM, BN, WM, WN, STAGES, false>), grid, block, 0, st, g);
    return (int)hipGetLastError();
}

}  // namespace

extern "C" int proteus_gemm_bf16(const uint16_t* A, const uint16_t* B, const uint16_t* bias, uint16_t* C,
                                 int M, int N, int K, int lda, int ldb, int ldc, int gelu, void* stream)
{
    if (!A || !B || !C) return PROTEUS_ERR_NULL_POINTER;
    if (M <= 0 || N <= 0 || K <= 0 || lda < K || ldb < K || ldc < N || N % 8 || K % 8 || lda % 8 || ldb % 8 || ldc % 8) return PROTEUS_ERR_BAD_SHAPE;
    if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15 || ((uintptr_t)bias & 7)) return PROTEUS_ERR_BAD_ALIGNMENT;
    // (a tile's rows, and the steps past the end, within 31 bits of its first; tiles numbered in 32 bits)
    const int64_t reach = 2 * ((int64_t)256 * (lda > ldb ? lda : ldb) + K + 1024);
    if (reach >= (1LL << 31) || (int64_t)((M + (int64_t)63) / 64) * ((N + (int64_t)63) / 64) > (1 << 28)) return PROTEUS_ERR_TOO_LARGE;
    const Args g = {A, B, bias, C, M, N, K, lda, ldb, ldc, 0, 0, 0};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    auto tiles = [&](const int64_t bm, const int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    auto filled = [&](const int64_t t, const int64_t slots) { return (double)t / (double)((t + slots - 1) / slots * slots); };     // share of the rounds' slots
    // Small tiles until there is one for every compute unit, since a workgroup is a chain over K; its loads then run three steps ahead, as there is no other workgroup to
    // wait under.  From there on larger tiles, which read less LDS per product, unless their last round is mostly empty.  Us, 64 x 64 / 128 x 64, both four stages /
    // 128 x 64 two stages / 128 x 128 four stages / 128 x 128 two / 256 x 256 two, for M x N x K:
    //   2048 x 512 x 512 4.5 / 5.6 / 6.1 / 7.7 / 7.5 / 14.7, of 2048 8.7 / 11.7 / 14.5 / 17.6 / 18.5 / 42;  4096 x 512 x 512 6.2 / 6.1 / 6.5 / 8.0 / 7.9 / 15.0, of 2048 14.6 / 13.5 / 17.7 / 18.4 / 20.1 / 43
    //   8192 x 512 x 512 10.5 / 10.5 / 8.3 / 8.8 / 8.6 / 15.5, of 2048 26.8 / 25.5 / 22.8 / 21.2 / 24.3 / 44;  4096 x 2048 x 512 (GELU) 21.6 / 22.8 / 17.5 / 20.4 / 16.5 / 24.7
    //   6000 x 1536 x 512 20.7 / 22.9 / 16.0 / 21.9 / 19.1 / 17.7;  8192 x 1536 x 512 26.8 / 27.0 / 21.7 / 22.6 / 20.6 / 18.9;  6000 x 2048 x 512 (GELU) 30.0 / 33.0 / 23.8 / 29.1 / 24.0 / 26.1;  8192 x 2048 x 512
    //   (GELU) 40 / 43 / 30.0 / 37.8 / 29.0 / 27.8;  12288 x 1536 x 512 40.5 / 39.8 / 28.2 / 35.6 / 28.6 / 33.1;  16384 x 1536 x 512 54 / 53 / 36.7 / 44 / 35.3 / 36.6;  65536 x 2048 x 512 (GELU) 374 / 419 / 279 / 318 / 256 / 216
    //   half-empty tiles are not told apart: 200000 x 64 x 64 21.6 / 24.0 / 14.3 / 33.7 / 18.1 / 28.1 (the library 31.6), 70000 x 256 x 256 30.7 / 31.1 / 19.8 / 26.9 / 24.6 / 23.5 (34.5)
    if (tiles(64, 64) <= 256)   return go<64, 64, 2, 2, 4>(g, gelu != 0, st);
    if (tiles(128, 64) <= 256)  return go<128, 64, 2, 2, 4>(g, gelu != 0, st);
    if (tiles(128, 128) <= 256) return K >= 1024 ? go<128, 128, 2, 2, 4>(g, gelu != 0, st) : go<128, 64, 2, 2, 2>(g, gelu != 0, st);
    const int64_t large = tiles(256, 256);
    if (tiles(128, 128) > 512 && (large <= 256 ? large >= 192 : filled(large, 256) > 0.8)) return go<256, 256, 2, 4, 2>(g, gelu != 0, st);
    if (filled(tiles(128, 128), 512) >= 0.7) return go<128, 128, 2, 2, 2>(g, gelu != 0, st);
    return go<128, 64, 2, 2, 2>(g, gelu != 0, st);
}
