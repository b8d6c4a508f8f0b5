// What the embedding kernels that go through distance grids share (we_grid.hip, we_aniso_grid.hip): the layout of their
// workspace, the pieces of the preparation, and the passes of a workgroup over its grids.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "proteus_hip.h"

namespace proteus_we_grid {

constexpr int WG_OBS     = 16;                    // observers per workgroup (one tile of the 16x16x4 product)
constexpr int WG_FLUSH   = 2048;                  // sources between two flushes
constexpr int WG_ROWS    = 1216;                  // rows of 16 cells in LDS: 77 824 bytes, two workgroups of 8 waves per compute unit
constexpr int WG_R0      = 8;                     // rows in front of the first node (zeros, read by the product)
constexpr int WG_OCT     = 8;                     // extra rows per octave: six nodes reach five rows into the next one (8: a shift in the address)
constexpr int WG_MAX_WINDOWS = 16;
constexpr int WG_MAX_TERMS = 24;                  // of the expansion of the anisotropic phase

constexpr float WG_OVERSAMPLING = 3.5f;
constexpr float WG_UNIT  = 4096.0f;               // coordinates are scaled by this power of two (see the spread)
constexpr float WG_MAGIC = 12582912.0f;           // 1.5 x 2^23: t + WG_MAGIC holds rint(t) in its low bits
constexpr uint32_t WG_MAGIC_BITS = 0x4B400000u;

// The rows of one of GP grids that share the LDS.
template <int GP> struct WgGrid {
    static constexpr int ROWS  = WG_ROWS / GP;
    static constexpr int TRASH = ROWS - 6;        // the rows of sources that belong to no cell
    static constexpr int CELLS = TRASH - WG_R0 - 5 - WG_OCT * 10;      // cells per window (n < 2^11)
    static_assert(WG_R0 + CELLS - 1 + WG_OCT * 10 + 6 <= TRASH, "rows of the spread");
    static_assert(WG_R0 + 8 * ((CELLS + 6) / 2 / 8 + 1) * 2 + 8 <= ROWS, "rows of the product");
};
constexpr int WG_GROUPS  = (WgGrid<1>::CELLS + 5 + 1) / 2 / 8 + 1;     // groups of 8 rows of the tables

struct WgParams {                 // head of the workspace, written by the preparation
    float inv_h, h;
    float cb_mid, b_max;          // anisotropic: middle of the C-beta scales, length of the longest C-beta vector
    int   terms;                  // anisotropic: terms of the expansion, 0: sum directly
    int   pad[59];
};
struct WgWave { double rev; float q, dq; };      // k h / 2 pi; 1/phihat and its derivative at theta = k h

// even polynomial 1/phihat(theta), relative error 3e-10 for |theta| <= pi/3.5
__device__ const double WG_Q[8] = {0.5144796916399992, 0.1467794687271181, 0.022356478641989086, 0.0024221529567290006,
                                 0.00020978467048036778, 1.54869506429115e-05, 9.95433626001851e-07, 7.199788952850109e-08};

struct WgBox { float lo[3], hi[3], bad, pad; };  // of 64 tokens, unpadded ones only; bad: one of them is not finite

struct WgLayout { size_t counts, waves, table, boxes, sources, sources_b, lengths, terms, tiles, bytes; int npad, nkt, nbox, blocks; };

__host__ __device__ inline WgLayout wg_layout(int Z, int N, int K, bool aniso)
{
    WgLayout l;
    l.nkt    = (K + 15) / 16;
    l.npad   = (N + 63) / 64 * 64 + 512;          // the stream reads up to an iteration (256 sources) past the end
    l.nbox   = (N + 63) / 64;
    l.blocks = (l.npad + 255) / 256;              // of the preparation, per batch item
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    l.counts    = sizeof(WgParams);
    l.waves     = l.counts + up((size_t)Z * 4);
    l.table     = l.waves + up((size_t)l.nkt * 16 * sizeof(WgWave));
    l.boxes     = l.table + (size_t)WG_GROUPS * l.nkt * 64 * 16;
    l.sources   = l.boxes + up((size_t)Z * l.nbox * sizeof(WgBox));
    l.sources_b = l.sources + up((size_t)Z * l.npad * 16);
    l.lengths   = l.sources_b + (aniso ? up((size_t)Z * l.npad * 16) : 0);
    l.terms     = l.lengths + (aniso ? up((size_t)Z * l.blocks * 4) : 0);
    l.tiles     = l.terms + (aniso ? (size_t)WG_MAX_TERMS * l.nkt * 16 * 8 : 0);
    l.bytes     = l.tiles + (aniso ? up((size_t)l.nkt * 4) : 0);
    return l;
}

// ---------------------------------------------------------------------------------------------------------------
// Preparation

__device__ __forceinline__ int wg_count_padded(const uint8_t* m, const int from, const int to, const int tid)
{
    int c = 0;
    int j = from + tid;
#pragma unroll 1
    for (; j + 3 * 256 < to; j += 4 * 256) {
        const int a = m[j], b = m[j + 256], d = m[j + 512], e = m[j + 768];
        c += (a != 0) + (b != 0) + (d != 0) + (e != 0);
    }
    for (; j < to; j += 256) c += m[j] != 0;
    return c;
}

// One block of 256 threads takes 256 tokens of a batch item: unpadded ones to the front of the item's list of sources, with
// their token index; padded and surplus slots get coordinates at infinity, which no cell takes.  Returns the thread's slot.
__device__ __forceinline__ int wg_compact(const float* __restrict__ coords, const int layout, const uint8_t* __restrict__ mask, char* __restrict__ ws,
                                          const WgLayout& L, const int N, const int block)
{
    const int z = block / L.blocks, b = block % L.blocks;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ int s_cnt[3][4];
    const size_t zN = (size_t)z * N;
    const float* cz = coords + zN * 3;
    const uint8_t* mz = mask ? mask + zN : nullptr;
    float4* src = reinterpret_cast<float4*>(ws + L.sources) + (size_t)z * L.npad;
    const int j = b * 256 + tid;
    const bool in = j < N;
    const bool valid = in && !(mz && mz[j]);
    int below = 0, total = 0;
    if (mz) {
        below = wg_count_padded(mz, 0, min(b * 256, N), tid);
        total = below + wg_count_padded(mz, min(b * 256, N), N, tid);
        for (int o = 32; o > 0; o >>= 1) { below += __shfl_xor(below, o); total += __shfl_xor(total, o); }
    }
    const uint64_t bal = __builtin_amdgcn_ballot_w64(valid);
    if (lane == 0) { s_cnt[0][wave] = below; s_cnt[1][wave] = total; s_cnt[2][wave] = __builtin_popcountll(bal); }
    __syncthreads();
    below = total = 0;
    int base = 0;
    for (int w = 0; w < 4; ++w) { below += s_cnt[0][w]; total += s_cnt[1][w]; base += w < wave ? s_cnt[2][w] : 0; }
    const int n = N - total;                                        // unpadded tokens of the item
    const int before = min(b * 256, N) - below + base + __builtin_popcountll(bal & ((1ull << lane) - 1ull));   // unpadded tokens in front of j
    if (b == 0 && tid == 0) reinterpret_cast<int*>(ws + L.counts)[z] = n;
    const float inf = __builtin_inff();
    float4 v = make_float4(inf, inf, inf, __builtin_bit_cast(float, in ? j : -1));
    if (valid) {
        if (layout == PROTEUS_COORDS_SOA) { v.x = cz[j]; v.y = cz[(size_t)N + j]; v.z = cz[2 * (size_t)N + j]; }
        else { v.x = cz[3 * (size_t)j]; v.y = cz[3 * (size_t)j + 1]; v.z = cz[3 * (size_t)j + 2]; }
        v.x *= WG_UNIT; v.y *= WG_UNIT; v.z *= WG_UNIT;
    }
    if (b * 4 + wave < L.nbox) {
        float lo[3] = {v.x, v.y, v.z}, hi[3] = {valid ? v.x : -inf, valid ? v.y : -inf, valid ? v.z : -inf};
        const bool bad = valid && !(fabsf(v.x) + fabsf(v.y) + fabsf(v.z) < 3.0e38f);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            for (int o = 32; o > 0; o >>= 1) { lo[c] = fminf(lo[c], __shfl_xor(lo[c], o)); hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], o)); }
        const bool any_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
        if (lane == 0) {
            WgBox* box = reinterpret_cast<WgBox*>(ws + L.boxes) + (size_t)z * L.nbox + b * 4 + wave;
            *box = WgBox{{lo[0], lo[1], lo[2]}, {hi[0], hi[1], hi[2]}, any_bad ? inf : 0.f, 0.f};
        }
    }
    const int slot = in ? (valid ? before : n + (j - before)) : j;
    if (slot < L.npad) src[slot] = v;
    return slot;
}

// Largest of a value over the 256 threads of a block (NaN and infinity count as infinity).
__device__ __forceinline__ float wg_block_max(float v)
{
    __shared__ float s_max[4];
    const int lane = threadIdx.x & 63;
    const bool bad = __builtin_amdgcn_ballot_w64(!(v < 3.0e38f)) != 0;
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    __syncthreads();
    if (lane == 0) s_max[threadIdx.x >> 6] = bad ? __builtin_inff() : v;
    __syncthreads();
    return fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
}

// Several at once: sums of the first SUMS values, largest of the others.  (Its LDS is not guarded against a second call in one kernel.)
template <int SUMS, int COUNT>
__device__ __forceinline__ void wg_block_reduce(float (&v)[COUNT])
{
    __shared__ float s_red[COUNT][4];
    const float inf = __builtin_inff();
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
        if (i >= SUMS) v[i] = v[i] < 3.0e38f ? v[i] : inf;
        for (int o = 32; o > 0; o >>= 1) { const float w = __shfl_xor(v[i], o); v[i] = i < SUMS ? v[i] + w : fmaxf(v[i], w); }
        if ((threadIdx.x & 63) == 0) s_red[i][threadIdx.x >> 6] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
        const float x = s_red[i][0], y = s_red[i][1], z = s_red[i][2], w = s_red[i][3];
        v[i] = i < SUMS ? x + y + z + w : fmaxf(fmaxf(x, y), fmaxf(z, w));
    }
}

// Largest of a thread's share of the wavenumbers, for the 256 threads of a block; infinite if one of them is not finite.
__device__ __forceinline__ float wg_largest(const float* __restrict__ wavenumbers, const int K)
{
    float km = 0.f;
    bool bad = false;
    for (int k = threadIdx.x; k < K; k += 256) { const float w = fabsf(wavenumbers[k]); bad |= !(w < 3.0e38f); km = fmaxf(km, w); }
    return bad ? __builtin_inff() : km;
}

// Cells per unit of length for the largest wavenumber, rounded to float once: h is its exact inverse from here on.  Wavenumbers beyond
// any use (wavelengths below 0.11, where the coefficients of the spreading kernel would lose bits as denormals) give an infinite
// value, which sends every workgroup to the direct sums.
__device__ __forceinline__ float wg_cells_per_length(const float km)
{
    const float inv_h = fmaxf(km * (WG_OVERSAMPLING / 3.14159265f) * 1.000001f, 1.0e-6f);
    return inv_h < 64.0f ? inv_h : __builtin_inff();
}

// Wave `unit` fills 8 rows of the tables for 16 wavenumbers: cosine and sine of k h (row + 1/2), two rows of four per lane.
__device__ __forceinline__ void wg_fill_tables(const float* __restrict__ wavenumbers, char* __restrict__ ws, const WgLayout& L, const int K, const double h, const int unit)
{
    const int lane = threadIdx.x & 63;
    const int kt = unit % L.nkt, g = unit / L.nkt;
    const int k = kt * 16 + (lane & 15);
    const double rev = (k < K ? (double)wavenumbers[k] : 0.0) * h * 0.15915494309189533577;
    float c[4];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const double y = (double)(8 * g + 4 * s + (lane >> 4)) + 0.5;
        const double ph = rev * y;
        const float f = (float)(ph - __builtin_floor(ph));
        c[2 * s]     = __builtin_amdgcn_cosf(f);
        c[2 * s + 1] = __builtin_amdgcn_sinf(f);
    }
    reinterpret_cast<float4*>(ws + L.table)[((size_t)g * L.nkt + kt) * 64 + lane] = make_float4(c[0], c[1], c[2], c[3]);
    if (g == 0 && lane < 16) {
        const double th = rev * 6.283185307179586477, t2 = th * th;
        double q = 0.0, dq = 0.0;
#pragma unroll
        for (int i = 7; i >= 0; --i) q = q * t2 + WG_Q[i];
#pragma unroll
        for (int i = 7; i >= 1; --i) dq = dq * t2 + 2 * i * WG_Q[i];
        WgWave w; w.rev = rev; w.q = (float)q; w.dq = (float)(dq * th);
        reinterpret_cast<WgWave*>(ws + L.waves)[k] = w;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Pieces of the main kernels

__device__ __forceinline__ float wg_lane(const float v, const int l)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

__device__ __forceinline__ float wg_vgpr(float v)
{
    asm volatile("" : "+v"(v));      // keep a constant in a vector register: an instruction with a literal or scalar operand issues in 4 clocks, one without in 2.4
    return v;
}

// distance of a pair: 1/r (a hardware reciprocal square root) and r, with one Newton step, to half an ulp
__device__ __forceinline__ void wg_distance(const float dx, const float dy, const float dz, float& r2, float& inv, float& r)
{
    r2  = dx * dx + dy * dy + dz * dz;
    inv = __builtin_amdgcn_rsqf(r2);
    const float r0 = r2 * inv;
    r = __builtin_fmaf(__builtin_fmaf(-r0, r0, r2), 0.5f * inv, r0);
}

typedef __attribute__((address_space(3))) uint32_t wg_lds_u32;
struct wg_true { static constexpr bool value = true; };
struct wg_false { static constexpr bool value = false; };
typedef float wg_f4 __attribute__((ext_vector_type(4)));

// The spreading kernel: the node at offset +a (a = 1/2, 3/2, 5/2) from the middle of a source's cell gets E_a(x) + x O_a(x), the one
// at -a E_a(x) - x O_a(x), x in [-1/2, 1/2] being the source's position in the cell; E and O quadratic in x^2.
struct WgKernel {
    float e[3][3], o[3][3];
    __device__ __forceinline__ explicit WgKernel(const float f)
    {
        constexpr float E[3][3] = {{0.8198235f, -0.41093102f, 0.08094943f}, {0.15015647f, 0.37342498f, -0.1214422f}, {0.0018756188f, 0.037506126f, 0.04049774f}};
        constexpr float O[3][3] = {{0.65685374f, -0.43981674f, 0.14080364f}, {0.40670425f, 0.057586372f, -0.069855906f}, {0.013345578f, 0.05343353f, 0.01371953f}};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) { e[i][j] = wg_vgpr(f * E[i][j]); o[i][j] = wg_vgpr(f * O[i][j]); }
    }
    // Weights of the six nodes, first to last, times c.  Where they are denormals none may come out as -0, whose bit pattern is
    // 2^31: the outermost weight falls to 2.54e-6 of a full one at the edge of the cell, 2.66 units at the smallest `scale`
    // (1.048e6), and E c is rounded to a whole unit.  With c > 1/2 (the isotropic 2^e h / r) at least 0.8 units are left.
    // SMALL_C: c may be anything above zero, and the outermost pair takes c last: E - x O is a normal number above zero.
    template <bool SMALL_C = false>
    __device__ __forceinline__ void weights(const float x, const float c, float (&w)[6]) const
    {
        const float x2 = x * x, xc = x * c;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const float E = __builtin_fmaf(__builtin_fmaf(e[i][2], x2, e[i][1]), x2, e[i][0]), O = __builtin_fmaf(__builtin_fmaf(o[i][2], x2, o[i][1]), x2, o[i][0]);
            if (SMALL_C && i == 2) {
                w[0] = __builtin_fmaf(-O, x, E) * c;
                w[5] = __builtin_fmaf(O, x, E) * c;
                continue;
            }
            const float t = E * c;
            w[2 - i] = __builtin_fmaf(-O, xc, t);
            w[3 + i] = __builtin_fmaf(O, xc, t);
        }
    }
};

// Opaque copy of a thread's index: keeps the addresses of the passes over the grids out of registers between them.
__device__ __forceinline__ int wg_again(int v) { asm volatile("" : "+v"(v)); return v; }

// How far away can a source be?  The farthest corner of the boxes around every 64 tokens, from the middle of the observers, plus
// the observers' own radius (in units of the scaled coordinates; infinite if anything is not finite).
template <int WAVES>
__device__ __forceinline__ float wg_reach(const float4& me, const bool ok, const WgBox* __restrict__ boxes, const int nbox, float* s_red)
{
    const int tid = threadIdx.x, lane = tid & 63;
    float lo[3] = {3.0e38f, 3.0e38f, 3.0e38f}, hi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
    if (ok) { lo[0] = hi[0] = me.x; lo[1] = hi[1] = me.y; lo[2] = hi[2] = me.z; }
#pragma unroll
    for (int c = 0; c < 3; ++c)
        for (int o = 8; o > 0; o >>= 1) { lo[c] = fminf(lo[c], __shfl_xor(lo[c], o)); hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], o)); }
    const float mx = 0.5f * (lo[0] + hi[0]), my = 0.5f * (lo[1] + hi[1]), mz = 0.5f * (lo[2] + hi[2]);
    const float ex = hi[0] - mx, ey = hi[1] - my, ez = hi[2] - mz;
    float far2 = 0.f;
    for (int b = tid; b < nbox; b += WAVES * 64) {
        const WgBox q = boxes[b];
        const float dx = fmaxf(q.hi[0] - mx, mx - q.lo[0]), dy = fmaxf(q.hi[1] - my, my - q.lo[1]), dz = fmaxf(q.hi[2] - mz, mz - q.lo[2]);
        const float d2 = dx * dx + dy * dy + dz * dz + q.bad;
        if (q.lo[0] <= q.hi[0] || q.bad != 0.f) far2 = d2 < 3.0e38f ? fmaxf(far2, d2) : __builtin_inff();       // (NaN counts as infinity and stays)
    }
    for (int o = 32; o > 0; o >>= 1) far2 = fmaxf(far2, __shfl_xor(far2, o));
    if (lane == 0) s_red[tid >> 6] = far2;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) far2 = fmaxf(far2, s_red[w]);
    return (__builtin_sqrtf(far2) + __builtin_sqrtf(ex * ex + ey * ey + ez * ez)) * 1.00001f;
}

// Pairs of a workgroup's observers that no cell takes: a list per wave in the LDS that the grids no longer need.
// (What follows the grids finds its lane by itself: kept over the windows the thread's index costs the spread a register.)
__device__ __forceinline__ int wg_lane_id() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
struct WgPair { float r, m, A; int obs; };                     // distance, 1/r, (anisotropic) A; in units of length

// Every wave searches its share of the sources for them, 256 on their way while the 256 before are looked at: only what lies within
// `reach2` (squared, scaled) of an observer in `near` is placed.  (One wave per observer, which waits for memory at every 64 sources and does
// the sums as it meets them, took as long as the spread where most workgroups have such an observer: compact chains, us before and now,
// isotropic 1 x 16384 with the sums 476 / 384, 1 x 65536 5348 / 4608, 1 x 8192 anisotropic 249 / 155.)  find(j, dx, dy, dz, pair): does source j's pair have no cell?
// Returns (to all threads) whether the lists hold all of them, and the lists' lengths to the first lanes; a list is in the order of the sources.
template <int WAVES, class Find>
__device__ __forceinline__ bool wg_collect(uint32_t* s_grid, int* s_cnt, const int wave, const uint32_t near, const float4* __restrict__ src, const int n, const float4& me,
                                           const float reach2, int& lengths, Find find)
{
    constexpr int CAP = WG_ROWS * WG_OBS * 4 / 16 / WAVES, BATCH = 4;
    const int lane = wg_lane_id();
    WgPair* const list = reinterpret_cast<WgPair*>(s_grid) + wave * CAP;
    const int share = (n + WAVES * 64 * BATCH - 1) / (WAVES * 64 * BATCH) * (64 * BATCH);
    const int end = min((wave + 1) * share, n);
    int count = 0;
    float4 next[BATCH];
    if (wave * share < end)
#pragma unroll
        for (int i = 0; i < BATCH; ++i) next[i] = src[wave * share + 64 * i + lane];
    for (int j0 = wave * share; j0 < end && count <= CAP; j0 += 64 * BATCH) {
        float4 q[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) q[i] = next[i];
        if (j0 + 64 * BATCH < end)
#pragma unroll
            for (int i = 0; i < BATCH; ++i) next[i] = src[j0 + 64 * (BATCH + i) + lane];        // (less than 256 past n: inside the list's padding)
        for (uint32_t left = near; left; left &= left - 1) {
            const int o = __builtin_ctz(left);
            const float xi = wg_lane(me.x, o), yi = wg_lane(me.y, o), zi = wg_lane(me.z, o);
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                const int j = j0 + 64 * i + lane;
                const float dx = xi - q[i].x, dy = yi - q[i].y, dz = zi - q[i].z;
                const bool close = j < n && dx * dx + dy * dy + dz * dz <= reach2;
                if (__builtin_amdgcn_ballot_w64(close) == 0) continue;
                WgPair p;
                p.obs = o;
                const uint64_t hits = __builtin_amdgcn_ballot_w64(find(j, dx, dy, dz, p) && close);
                const int at = count + __builtin_popcountll(hits & ((1ull << lane) - 1ull));
                if ((hits >> lane & 1) && at < CAP) list[at] = p;
                count += __builtin_popcountll(hits);
            }
        }
    }
    if (lane == 0) s_cnt[wave] = count;
    __syncthreads();
    lengths = lane < WAVES ? s_cnt[lane] : 0;
    return __builtin_amdgcn_ballot_w64(lengths > CAP) == 0;
}

// add(pair) for the listed pairs of observer o, in the order of the sources.
template <int WAVES, class Add>
__device__ __forceinline__ void wg_listed(const uint32_t* s_grid, const int lengths, const int o, Add add)
{
    constexpr int CAP = WG_ROWS * WG_OBS * 4 / 16 / WAVES;
    for (uint64_t some = __builtin_amdgcn_ballot_w64(lengths > 0); some; some &= some - 1) {
        const int w = __builtin_ctzll(some);
        const WgPair* list = reinterpret_cast<const WgPair*>(s_grid) + w * CAP;
        const int count = __builtin_amdgcn_readlane(lengths, w);
        for (int i0 = 0; i0 < count; i0 += 64) {
            const int lane = wg_lane_id();
            const WgPair mine = list[min(i0 + lane, count - 1)];
            uint64_t todo = __builtin_amdgcn_ballot_w64(i0 + lane < count && mine.obs == o);
            while (todo) {
                const int b = __builtin_ctzll(todo);
                todo &= todo - 1;
                WgPair p;
                p.r = wg_lane(mine.r, b); p.m = wg_lane(mine.m, b); p.A = wg_lane(mine.A, b);
                add(p);
            }
        }
    }
}

// The sums over these pairs, dealt out over the waves: sum(U, observer, first) does U times 64 wavenumbers, of the workgroup's `tiles` of 16 those from
// `first` on.  U = 1 where the lists hold all pairs and larger units would leave waves idle; otherwise up to MAX_U: a pair is fetched once for
// all of them.  Us, tokens in places of 20, 100 and 1000, 0.03 apart, 1 x 1100, K = 256, so / with 64 wavenumbers a unit always and over-full
// lists an observer at a time: 30 / 39, 42 / 145, 177 / 941; 1 x 16384 in places of 1000 1380 / 4120.
template <int U> struct WgWide { static constexpr int value = U; };
template <int WAVES, int MAX_U, class Sum>
__device__ __forceinline__ void wg_near_units(const int wave, const uint32_t near, const int tiles, const bool listed, Sum sum)
{
    const bool wide = !listed || __builtin_popcount(near) * ((tiles + 4 * MAX_U - 1) / (4 * MAX_U)) >= WAVES;
    const int step = wide ? 4 * MAX_U : 4;
    int unit = 0;
    for (uint32_t left = near; left; left &= left - 1) {
        const int o = __builtin_ctz(left);
        for (int first = 0; first < tiles; first += step) {
            if ((unit++ & (WAVES - 1)) != wave) continue;
            const int some = min(tiles - first, step);
            if (MAX_U > 2 && some > 8) sum(WgWide<MAX_U>{}, o, first);
            else if (some > 4)         sum(WgWide<2>{}, o, first);
            else                       sum(WgWide<1>{}, o, first);
        }
    }
}

// The integers of GP grids in LDS, of which the first `used` rows hold anything.
template <int GP, int THREADS>
__device__ __forceinline__ void wg_clear(uint32_t* s_grid, const int used)
{
    const int tid = threadIdx.x;
#pragma unroll
    for (int g = 0; g < GP; ++g)
        for (int i = tid; i < used * (WG_OBS / 4); i += THREADS) reinterpret_cast<uint4*>(s_grid)[g * WgGrid<GP>::ROWS * (WG_OBS / 4) + i] = make_uint4(0, 0, 0, 0);
}

template <bool SIGNED>
__device__ __forceinline__ wg_f4 wg_float4(const uint4& v)
{
    if (SIGNED) return wg_f4{(float)(int)v.x, (float)(int)v.y, (float)(int)v.z, (float)(int)v.w};
    return wg_f4{(float)v.x, (float)v.y, (float)v.z, (float)v.w};
}

// A flush: the integers move on to the threads' float accumulators; after the last one the sums go back to LDS as floats.
template <int GP, int THREADS, int CHUNKS, bool SIGNED>
__device__ __forceinline__ void wg_flush(uint32_t* s_grid, wg_f4 (&acc)[CHUNKS], const int used, const bool last)
{
    const int t = wg_again(threadIdx.x);
    uint4* g4 = reinterpret_cast<uint4*>(s_grid);
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
        const int q = t + i * THREADS;
        if (q < GP * WgGrid<GP>::ROWS * (WG_OBS / 4) && (GP == 1 ? q : q % (WgGrid<GP>::ROWS * (WG_OBS / 4))) < used * (WG_OBS / 4)) {
            acc[i] += wg_float4<SIGNED>(g4[q]);
            if (!last) g4[q] = make_uint4(0, 0, 0, 0);
            else reinterpret_cast<wg_f4*>(s_grid)[q] = acc[i];
        }
    }
}

// Bring the octaves together: node v = n_lo - 3 + p of a grid to its row WG_R0 + p, zeros in front and behind.
template <int GP, int THREADS, int CHUNKS, bool SIGNED>
__device__ __forceinline__ void wg_combine(uint32_t* s_grid, wg_f4 (&acc)[CHUNKS], const int n_lo, const int cells, const bool floats)
{
    const int nodes = cells + 5, e_lo = 31 - __builtin_clz(n_lo);
    const int t = wg_again(threadIdx.x);
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
        const int q = t + i * THREADS;
        const int pn = (GP == 1 ? q >> 2 : (q >> 2) % WgGrid<GP>::ROWS) - WG_R0;
        wg_f4 v = {0.f, 0.f, 0.f, 0.f};
        if (pn >= 0 && pn < nodes && (GP == 1 || q < GP * WgGrid<GP>::ROWS * (WG_OBS / 4))) {
            const int na = max(pn - 5, 0) + n_lo, nz = min(pn, cells - 1) + n_lo;       // sources that reach this node
            const int ea = 31 - __builtin_clz(na), ez = 31 - __builtin_clz(nz);
            for (int e = ea; e <= ez; ++e) {
                const int at = q + WG_OCT * (e - e_lo) * (WG_OBS / 4);
                const float sc = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
                if (floats) v += reinterpret_cast<const wg_f4*>(s_grid)[at] * sc;
                else        v += wg_float4<SIGNED>(reinterpret_cast<const uint4*>(s_grid)[at]) * sc;
            }
        }
        acc[i] = v;
    }
    __syncthreads();
    const int w = wg_again(threadIdx.x);
#pragma unroll
    for (int i = 0; i < CHUNKS; ++i) {
        const int q = w + i * THREADS;
        const int row = GP == 1 ? q >> 2 : (q >> 2) % WgGrid<GP>::ROWS;
        if (q < GP * WgGrid<GP>::ROWS * (WG_OBS / 4) && row < WG_R0 + nodes + 8) reinterpret_cast<wg_f4*>(s_grid)[q] = acc[i];
    }
}

// GR grids (`gs` floats apart) at KT tiles of 16 wavenumbers: rows j = 0 .. groups * 8 on both sides of the middle, E and O the sum
// and difference of the two sides: ec += E cos, os += O sin and (MOMENT) oc += y O cos, es += y E sin with y = j + 1/2.  The tiles
// share the grid values, the grids the tables, which come from L2, AHEAD groups of 8 rows ahead.  Of the groups those from `begin` on.
template <int KT, int AHEAD, bool MOMENT, int GR>
__device__ __forceinline__ void wg_product(const float* g, const int gs, const int mid, const int begin, const int groups, const float4* __restrict__ tb, const size_t ts, const int k2,
                                           wg_f4 (&ec)[GR][KT], wg_f4 (&os)[GR][KT], wg_f4 (&oc)[GR][KT], wg_f4 (&es)[GR][KT])
{
    const int lane = threadIdx.x & 63, obs = lane & 15, mm = lane >> 4;
    const float* gp = g + (WG_R0 + mid + mm) * WG_OBS + obs;
    const float* gm = g + (WG_R0 + mid - 1 - mm) * WG_OBS + obs;
#pragma unroll
    for (int r = 0; r < GR; ++r)
#pragma unroll
        for (int t = 0; t < KT; ++t) ec[r][t] = os[r][t] = oc[r][t] = es[r][t] = wg_f4{0.f, 0.f, 0.f, 0.f};
    float4 b[AHEAD][KT];
    auto fetch = [&](const int gr, float4 (&bb)[KT]) {
        const float4* at = tb + (size_t)min(gr, WG_GROUPS - 1) * ts;
#pragma unroll
        for (int t = 0; t < KT; ++t) bb[t] = at[t * k2];
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(begin + i, b[i]);
    float y = (float)(8 * begin + mm) + 0.5f;
    for (int g0 = begin; g0 < groups; g0 += AHEAD) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int gr = g0 + i;
            if (gr >= groups) break;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int off = (8 * gr + 4 * s) * WG_OBS;
#pragma unroll
                for (int r = 0; r < GR; ++r) {
                    const float a = gp[r * gs + off], m = gm[r * gs - off];
                    const float E = a + m, O = a - m;
                    const float Oy = O * y, Ey = E * y;
#pragma unroll
                    for (int t = 0; t < KT; ++t) {
                        const float bc = s ? b[i][t].z : b[i][t].x, bs = s ? b[i][t].w : b[i][t].y;
                        ec[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(E, bc, ec[r][t], 0, 0, 0);
                        os[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(O, bs, os[r][t], 0, 0, 0);
                        if (MOMENT) {
                            oc[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(Oy, bc, oc[r][t], 0, 0, 0);
                            es[r][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ey, bs, es[r][t], 0, 0, 0);
                        }
                    }
                }
                y += 4.0f;
            }
            fetch(gr + AHEAD, b[i]);
        }
    }
}

}  // namespace proteus_we_grid
