// Isotropic Wavefunction Embedding forward through distance grids, for gfx950 (MI355X).
//
// What it computes: the same sums as we_fwd.hip (weight 1/r),
//     F1(k) = sum_j e^(i k r_j) / r_j  (out: cos at even, sin at odd features),   F0(k) = sum_j e^(i k r_j)  (the sums)
// for every observer and every wavenumber.  For one observer F1 depends on nothing but its distances, so instead of
// evaluating every (source, wavenumber) pair the distances are first spread onto a uniform grid and the grid is then
// evaluated at the wavenumbers (a non-uniform Fourier transform of type 3; Dutt & Rokhlin 1993, Greengard & Lee 2004):
//     sum_l phi(a_l - x) e^(i theta a_l) = phihat(theta) e^(i theta x)   up to an aliasing error,   theta = k h,
// with 6 grid nodes around every distance.  Per pair of tokens that is a distance, six polynomial weights and six
// additions instead of 7 instructions per wavenumber; the rest is one small matrix product per observer,
// [nodes] x [nodes, 2 K], on the matrix cores.
//   - Grid: h = pi / (3.5 max|k|), nodes at half-integer multiples of h, so that the six nodes of a distance lie
//     symmetrically around the nearest integer multiple.
//   - phi: piecewise polynomial of degree 5 (an even and an odd part of degrees 4 and 5 for each pair of nodes), fitted by
//     least squares so that the relation above holds for all |theta| <= pi/3.5 with phihat the transform of phi itself:
//     relative error 2.2e-7 (rms over the position inside a cell, at the worst wavenumber), less than the error of a
//     single-precision phase at tens of revolutions.  1/phihat is an even polynomial in theta (WG_Q).
//   - F0 = -i dF1/dk comes from the same grid: two more products against node position x grid.
//   - Everything is summed in 32-bit integers (fixed point): LDS float atomics take 193 clocks per wave instruction on this
//     machine, integer ones 4.7 (conflict-free) to 6.2 (random cells); integer sums do not depend on their order, so
//     the waves of a workgroup share the grids and the result is the same from run to run.  A cell's octave e = floor(log2 n)
//     sets its scale: what is added is phi 2^e h / r < 2, so near and far sources keep the same relative precision (the
//     rounding of one addition is 2^-22 of the largest term); octaves have their own rows where they overlap.  After
//     2048 sources (what 32 bits hold at that scale) the integers are moved on to float accumulators.
//   - Pairs closer than h/2 (never the case for real structures) are summed directly, as are all pairs of a workgroup
//     whose distances would need too many windows of the grid or are not finite.
#include "we_grid.h"

namespace {

using namespace proteus_we_grid;

// Blocks [0, Z * L.blocks) compact the tokens of the batch items, the others fill the tables.
__global__ __launch_bounds__(256)
void we_grid_prepare_kernel(const float* __restrict__ coords, const int layout, const float* __restrict__ wavenumbers,
                            const uint8_t* __restrict__ mask, char* __restrict__ ws, const int Z, const int N, const int K)
{
    const WgLayout L = wg_layout(Z, N, K, false);
    const int blocks = Z * L.blocks;
    if ((int)blockIdx.x < blocks) {
        wg_compact(coords, layout, mask, ws, L, N, blockIdx.x);
        return;
    }
    const float inv_h = wg_cells_per_length(wg_block_max(wg_largest(wavenumbers, K)));
    const double h = 1.0 / (double)inv_h;
    const int unit = ((int)blockIdx.x - blocks) * 4 + (threadIdx.x >> 6);
    if (unit == 0 && (threadIdx.x & 63) == 0) { WgParams* p = reinterpret_cast<WgParams*>(ws); p->inv_h = inv_h; p->h = (float)h; }
    if (unit < WG_GROUPS * L.nkt) wg_fill_tables(wavenumbers, ws, L, K, h, unit);
}

// add(pair) for the pairs of one observer that are closer than h / 2, more of them than the lists hold (thousands of tokens in one place).
template <class Add>
__device__ __forceinline__ void wg_every_near(const float4* __restrict__ src, const int n, const float xi, const float yi, const float zi, const float inv_h,
                                              const int lane, Add add)
{
    float4 next = src[lane];
    for (int j0 = 0; j0 < n; j0 += 64) {
        const float4 q = next;
        next = src[j0 + 64 + lane];                            // (past the end: inside the list's padding)
        float r2, inv, r;
        wg_distance(xi - q.x, yi - q.y, zi - q.z, r2, inv, r);
        const bool near = __builtin_bit_cast(int, __builtin_fmaf(r, inv_h, WG_MAGIC)) == __builtin_bit_cast(int, WG_MAGIC);
        uint64_t todo = __builtin_amdgcn_ballot_w64(j0 + lane < n && r2 != 0.0f && near);
        while (todo) {
            const int b = __builtin_ctzll(todo);
            todo &= todo - 1;
            WgPair p;
            p.r = wg_lane(r, b); p.m = wg_lane(inv, b);
            add(p);
        }
    }
}

// Sums of four values over the four rows of 16 lanes: row i gets that of v_i.
__device__ __forceinline__ float wg_rows(const float v0, const float v1, const float v2, const float v3)
{
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    auto bits = [](const float v) { return __builtin_bit_cast(uint32_t, v); };
    auto sum  = [](const u2 v) { const uint32_t x = v.x, y = v.y; return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y); };
    const float a = sum(__builtin_bit_cast(u2, __builtin_amdgcn_permlane32_swap(bits(v0), bits(v2), false, false)));      // rows 0 + 2, 1 + 3 of v0 | of v2
    const float b = sum(__builtin_bit_cast(u2, __builtin_amdgcn_permlane32_swap(bits(v1), bits(v3), false, false)));
    return sum(__builtin_bit_cast(u2, __builtin_amdgcn_permlane16_swap(bits(a), bits(b), false, false)));
}

// All pairs of the workgroup's 16 observers summed directly, about as fast as the direct kernel does it (vector issue: a multiplication,
// fract, sine, cosine and two or four accumulations per pair and wavenumber; 1 x 4096, K = 256 1137 us bounded and 1305 unbounded against
// 1097 and 1188, K = 64 293 and 334 against 321 and 353; a wave per observer, its sources one by one, took 1225 at either K).  A lane holds an observer and a quarter of the
// wave's sources, 16 wavenumbers sit in scalar registers.  Tiles of 16 wavenumbers `first`, `first` + `step`, ...: as many waves as
// divide their number evenly take a tile each, the others of a tile share the sources and meet in LDS.
// BOUNDED: no phase leaves the +-256 revolutions that sine and cosine accept.
template <bool SUMS, int WAVES, bool BOUNDED>
__device__ __forceinline__ void wg_direct(uint32_t* s_grid, const int* s_tok, const float4* __restrict__ src, const int n, const int slot0, const float4& me,
                                          const float* __restrict__ wavenumbers, float* __restrict__ out, float* __restrict__ cos_sums,
                                          float* __restrict__ sin_sums, const size_t zN, const int K, const int first, const int step)
{
    constexpr int KT = 16, V = SUMS ? 4 : 2, BATCH = 8;       // V sums per observer and wavenumber
    static_assert(WAVES * WG_OBS * KT * V <= WG_ROWS * WG_OBS, "sums of the waves in LDS");
    const int tid = threadIdx.x, lane = tid & 63, obs = lane & 15, row = lane >> 4;
    const int wave  = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = ((K + KT - 1) / KT - first + step - 1) / step;
    const int kw = min(WAVES, tiles & -tiles), sw = WAVES / kw;          // tiles at a time, waves per tile
    const int kg = wave / sw, sg = wave % sw;
    typedef float Sums __attribute__((ext_vector_type(V)));
    Sums* red = reinterpret_cast<Sums*>(s_grid);              // [WAVES][WG_OBS][KT]
#pragma unroll 1
    for (int tile = 0; tile < tiles; tile += kw) {
        const int kl = (first + (tile + kg) * step) * KT + obs;
        const float krl = (float)((kl < K ? (double)wavenumbers[kl] : 0.0) * 0.15915494309189533577);
        float kr[KT], acc[V][KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            kr[t] = wg_lane(krl, t);
#pragma unroll
            for (int v = 0; v < V; ++v) acc[v][t] = 0.f;
        }
        float4 q = src[sg * 4 + row];                          // (reads past the end stay inside the list's padding)
#pragma unroll 1
        for (int j0 = sg * 4; j0 < n; j0 += sw * 4) {
            const float4 p = q;
            q = src[j0 + sw * 4 + row];
            float r2, inv, r;
            // (in units of length: the square of a scaled distance overflows from 4.5e15 on)
            wg_distance((me.x - p.x) * (1.0f / WG_UNIT), (me.y - p.y) * (1.0f / WG_UNIT), (me.z - p.z) * (1.0f / WG_UNIT), r2, inv, r);
            const bool use = j0 + row < n && r2 != 0.0f;
            inv = use ? inv : 0.f; r = use ? r : 0.f;
            const float one = use ? 1.f : 0.f;
            // phases, then sines and cosines, then accumulations, as in the direct kernel
#pragma unroll
            for (int t0 = 0; t0 < KT; t0 += BATCH) {
                float cs[BATCH], sn[BATCH];
#pragma unroll
                for (int t = 0; t < BATCH; ++t) sn[t] = BOUNDED ? r * kr[t0 + t] : __builtin_amdgcn_fractf(r * kr[t0 + t]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < BATCH; ++t) { cs[t] = __builtin_amdgcn_cosf(sn[t]); sn[t] = __builtin_amdgcn_sinf(sn[t]); }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < BATCH; ++t) {
                    acc[0][t0 + t] = __builtin_fmaf(cs[t], inv, acc[0][t0 + t]);
                    acc[1][t0 + t] = __builtin_fmaf(sn[t], inv, acc[1][t0 + t]);
                    if constexpr (SUMS) { acc[2][t0 + t] = __builtin_fmaf(cs[t], one, acc[2][t0 + t]); acc[3][t0 + t] = __builtin_fmaf(sn[t], one, acc[3][t0 + t]); }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();                                       // the previous tiles' sums are read
#pragma unroll
        for (int t = 0; t < KT; t += 4) {
            Sums v;
#pragma unroll
            for (int i = 0; i < V; ++i) v[i] = wg_rows(acc[i][t], acc[i][t + 1], acc[i][t + 2], acc[i][t + 3]);
            red[(wave * WG_OBS + obs) * KT + t + row] = v;
        }
        __syncthreads();
        for (int i = tid; i < kw * WG_OBS * KT; i += WAVES * 64) {
            const int g = i / (WG_OBS * KT), e = i % (WG_OBS * KT);
            const int tok = s_tok[e / KT], k = (first + (tile + g) * step) * KT + e % KT;
            Sums v = red[g * sw * WG_OBS * KT + e];
            for (int w = 1; w < sw; ++w) v += red[(g * sw + w) * WG_OBS * KT + e];
            if (tok >= 0 && k < K) {
                const bool keep = slot0 + e / KT < n;
                const size_t at = (zN + tok) * K + k;
                reinterpret_cast<float2*>(out)[at] = keep ? make_float2(v[0], v[1]) : make_float2(0.f, 0.f);
                if constexpr (SUMS) { cos_sums[at] = keep ? v[2] : 0.f; sin_sums[at] = keep ? v[3] : 0.f; }
            }
        }
    }
}

// WAVES  8: two workgroups share a compute unit, one's product under the other's spread; 16: twice the waves on the same
//        observers, for launches of at most one workgroup per compute unit
template <bool SUMS, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 4)
void we_grid_kernel(const char* __restrict__ ws, const float* __restrict__ wavenumbers,
                    float* __restrict__ out, float* __restrict__ cos_sums, float* __restrict__ sin_sums,
                    const int Z, const int N, const int K)
{
    constexpr int THREADS = WAVES * 64;
    constexpr int STEP    = WAVES * 16;           // sources per iteration: a wave takes 16 observers x 4 sources, four times
    constexpr int CHUNKS  = (WG_ROWS * WG_OBS / 4 + THREADS - 1) / THREADS;    // float4 pieces of the grid per thread
    constexpr int CELLS   = WgGrid<1>::CELLS;
    constexpr int KT      = 16 / WAVES;           // tiles of 16 wavenumbers a wave takes at a time
    constexpr int AHEAD   = WAVES == 16 ? 4 : 2;  // groups of the tables in flight: a lone workgroup has nothing else to cover their latency
    extern __shared__ __align__(16) uint32_t s_grid[];          // [WG_ROWS][WG_OBS]
    __shared__ float s_red[WAVES];
    __shared__ int   s_near[WG_OBS];
    __shared__ int   s_tok[WG_OBS];
    __shared__ int   s_cnt[WAVES];

    const WgLayout L = wg_layout(Z, N, K, false);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z = blockIdx.y;
    const size_t zN = (size_t)z * N;
    const int n = reinterpret_cast<const int*>(ws + L.counts)[z];
    const float4* __restrict__ src = reinterpret_cast<const float4*>(ws + L.sources) + (size_t)z * L.npad;
    const WgWave* __restrict__ waves = reinterpret_cast<const WgWave*>(ws + L.waves);
    const float4* __restrict__ table = reinterpret_cast<const float4*>(ws + L.table);
    const float inv_h = reinterpret_cast<const WgParams*>(ws)->inv_h * (1.0f / WG_UNIT), h = reinterpret_cast<const WgParams*>(ws)->h;

    // ---- the workgroup's slots: unpadded observers first, then padded tokens (zero rows), then nothing.  (Workgroups of every blockIdx.z
    //      have the same slots and, of the tiles of 16 wavenumbers, every gridDim.z-th.) ----
    const int slot0 = blockIdx.x * WG_OBS;
    const int obs   = lane & 15;
    const float4 me = src[slot0 + obs];
    const bool ok   = slot0 + obs < n;
    if (tid < WG_OBS) { s_tok[tid] = slot0 + tid < N ? __builtin_bit_cast(int, me.w) : -1; s_near[tid] = 0; }
    if (slot0 >= n) {
        // padded tokens only
        if (blockIdx.z) return;
        __syncthreads();
        for (int q = 0; q < WG_OBS; ++q) {
            const int t = s_tok[q];
            if (t < 0) continue;
            const size_t row = zN + t;
            for (int k = tid; k < 2 * K; k += THREADS) out[row * 2 * K + k] = 0.f;
            if (SUMS) for (int k = tid; k < K; k += THREADS) { cos_sums[row * K + k] = 0.f; sin_sums[row * K + k] = 0.f; }
        }
        return;
    }

    const float reach = wg_reach<WAVES>(me, ok, reinterpret_cast<const WgBox*>(ws + L.boxes) + (size_t)z * L.nbox, L.nbox, s_red) * inv_h + 2.0f;
    // Sums without the grid: where there is nothing to spread onto (values that are not finite, wavelengths below 0.11, more than 16
    // windows), where everything lies in a few cells and most pairs in none, and where the windows, each of which streams all sources
    // again, cost more.  Us with 16 waves: per window 7.5 + 0.005 n, its product 0.15 K, without the sums 0.085 K, all pairs directly 10 + 1.2e-3 n K and
    // 10 + 1.0e-3 n K, K being the workgroup's share of the wavenumbers; 8 waves, of which two workgroups share a compute unit: 16.6 + 0.0033 n per window and
    // workgroup, its product 0.095 K and 0.055 K, all pairs directly as before.  (Between the two, so that the choice and with it `out` do not
    // depend on whether the sums are wanted.)  Wavelengths from 3.7 on, grid / pairs / this choice (without the sums): 1 x 1024 over 3 windows, K = 64 47 / 31 / 31,
    // K = 128 51 / 50 / 50, K = 256 63 / 89 / 63, K = 512 89 / 168 / 89, over 5 windows 86 / 50 / 50, 109 / 89 / 89, 159 / 168 / 159; 1 x 2048, K = 64 3 windows 69 / 89 / 69, 6 133 / 89 / 89;
    // 1 x 4096, K = 64 6 windows 225 / 325 / 225, 12 451 / 324 / 324, K = 256 12 785 / 1266 / 785.  (The direct kernel: 1 x 4096, K = 64 321, K = 256 1097.)
    const bool far = !(reach < (float)(CELLS * WG_MAX_WINDOWS));
    const float windows = __builtin_ceilf(reach * (1.0f / (float)CELLS));
    const float mine    = (float)K / (float)gridDim.z;
    const float by_grid = windows * (WAVES == 16 ? 7.5f + 5.0e-3f * (float)n + 0.115f * mine : 16.6f + 3.3e-3f * (float)n + 0.075f * mine);
    const float by_pair = (WAVES == 16 ? 8.0f : 0.0f) + 1.1e-3f * (float)n * mine;
    const bool direct = __builtin_amdgcn_readfirstlane(far || reach < 4.0f || (windows > 1.0f && by_grid > by_pair)) != 0;
    if (direct) {
        // (a cell is at most pi / 3.5 of phase: 1750 of them are 250 revolutions)
        if (reach < 1750.0f) wg_direct<SUMS, WAVES, true>(s_grid, s_tok, src, n, slot0, me, wavenumbers, out, cos_sums, sin_sums, zN, K, blockIdx.z, gridDim.z);
        else                 wg_direct<SUMS, WAVES, false>(s_grid, s_tok, src, n, slot0, me, wavenumbers, out, cos_sums, sin_sums, zN, K, blockIdx.z, gridDim.z);
        return;
    }
    const int ncell = __builtin_amdgcn_readfirstlane((int)reach);

    {
        // ---- the spreading kernel's coefficients, in fixed point ----
        // A weight is made as a single-precision denormal: its bit pattern is the rounded integer, and no conversion is needed
        // (4.7 clocks each).  Of the 2^-149 that takes 2^-12 comes with 1/r (WG_UNIT) and the rest with the coefficients, so that
        // every factor is a normal number.  One unit is `scale` of a full weight: 2 scale (the largest weight) times the
        // sources between two flushes stays below 2^32.
        const int nit = (n + STEP - 1) / STEP, quarter = nit * (STEP / 4);
        const bool flushes = nit * STEP > WG_FLUSH;
        const int tiles = (L.nkt - (int)blockIdx.z + (int)gridDim.z - 1) / (int)gridDim.z;      // of this workgroup
        const float scale = flushes ? 1048000.0f : fminf(4190000.0f, 2147000000.0f / (float)(nit * STEP));
        const WgKernel kernel(scale * h * 0x1p-137f);
        const float magic = wg_vgpr(WG_MAGIC), inv_hv = wg_vgpr(inv_h);
        uint32_t emask = 0xff800000u;
        asm volatile("" : "+v"(emask));

        float lowest = 3.0e38f;                    // smallest n of any source, as magic + n

        for (int n_lo = 1; n_lo <= ncell; n_lo += CELLS) {
            const int cells = min(CELLS, ncell + 1 - n_lo);           // source cells n_lo .. n_lo + cells - 1
            const int e_lo  = 31 - __builtin_clz(n_lo);
            const int e_hi  = 31 - __builtin_clz(n_lo + cells - 1);
            const int used  = WG_R0 + cells + 5 + WG_OCT * (e_hi - e_lo);      // rows that hold anything
            wg_f4 facc[CHUNKS];
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) facc[i] = wg_f4{0.f, 0.f, 0.f, 0.f};

            __syncthreads();                                             // the previous window's product is done
            wg_clear<1, THREADS>(s_grid, used);
            __syncthreads();

            // LDS address of a source's first node: row (n - n_lo) + 8 (e - e_lo), with n and e taken from float bits.  Sources
            // that belong to no cell of this window go to the trash rows: with one window those are the observer itself and slots
            // past the end (n is NaN) and pairs closer than h / 2 (n = 0, whose exponent takes the address below zero), all of
            // which one unsigned minimum catches.
            uint32_t base = (uint32_t)(uintptr_t)(wg_lds_u32*)s_grid + (uint32_t)((WG_R0 - n_lo - WG_OCT * e_lo) * WG_OBS + obs) * 4u
                            - (WG_MAGIC_BITS << 6) - 127u * (WG_OCT * WG_OBS * 4u);
            uint32_t trash = (uint32_t)(uintptr_t)(wg_lds_u32*)s_grid + (uint32_t)(WgGrid<1>::TRASH * WG_OBS + obs) * 4u;
            asm volatile("" : "+v"(base), "+v"(trash));
            const uint32_t first = WG_MAGIC_BITS + (uint32_t)n_lo;

            // The four sources of a wave instruction come from four quarters of the sequence: neighbours in the chain lie in the
            // same cells, and additions to one address take turns.
            const float4* p = src + (lane >> 4) * quarter + wave * 2;
            auto spread = [&](const float4& q, auto multi) {
                float r2, inv, r;
                wg_distance(me.x - q.x, me.y - q.y, me.z - q.z, r2, inv, r);
                const float u  = __builtin_fmaf(r, inv_hv, magic);
                const float nf = u - magic;
                const float x  = __builtin_fmaf(r, inv_hv, -nf);
                const uint32_t ub = __builtin_bit_cast(uint32_t, u);
                const uint32_t eb = __builtin_bit_cast(uint32_t, nf) & emask;
                const float c  = inv * __builtin_bit_cast(float, eb);                      // 2^e / r
                float w[6];
                kernel.weights(x, c, w);
                uint32_t at = (ub << 6) + base + (eb >> 14);
                if (decltype(multi)::value) at = ub - first < (uint32_t)cells ? at : trash;
                else                        at = min(at, trash);
                wg_lds_u32* a = (wg_lds_u32*)(uintptr_t)at;
#pragma unroll
                for (int l = 0; l < 6; ++l)
                    __hip_atomic_fetch_add(a + l * WG_OBS, __builtin_bit_cast(uint32_t, w[l]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                lowest = __builtin_fminf(lowest, u);
            };
            float4 q0 = p[0], q1 = p[1], q2 = p[STEP / 8], q3 = p[STEP / 8 + 1];
            int until = flushes ? WG_FLUSH / STEP : nit;
            for (int it = 0;;) {
                auto stream = [&](auto multi) {
                    for (; it < until; ++it) {
                        p += STEP / 4;
                        spread(q0, multi); spread(q1, multi);
                        q0 = p[0]; q1 = p[1];
                        spread(q2, multi); spread(q3, multi);
                        q2 = p[STEP / 8]; q3 = p[STEP / 8 + 1];
                    }
                };
                if (ncell > CELLS) stream(wg_true{}); else stream(wg_false{});
                if (!flushes) break;
                __syncthreads();
                wg_flush<1, THREADS, CHUNKS, false>(s_grid, facc, used, it >= nit);
                __syncthreads();
                if (it >= nit) break;
                until = min(it + WG_FLUSH / STEP, nit);
            }
            if (!flushes) __syncthreads();

            wg_combine<1, THREADS, CHUNKS, false>(s_grid, facc, n_lo, cells, flushes);
            __syncthreads();

            // ---- the grid at the wavenumbers ----
            const int mid    = (cells + 6) / 2;
            const int groups = (mid + 7) / 8;
            const int vc     = n_lo - 3 + mid;                              // the middle lies at vc h
            const int mm     = lane >> 4;
            // rows `from` to `to` of a lane's four of a tile
            auto finish = [&](const int kt, const int from, const int to, const wg_f4& ec, const wg_f4& os, const wg_f4& oc, const wg_f4& es) {
                const int k = kt * 16 + obs;
                if (k >= K) return;
                const WgWave w = waves[k];
                const double ph = w.rev * (double)vc;
                const float f  = (float)(ph - __builtin_floor(ph));
                const float rc = __builtin_amdgcn_cosf(f), rs = __builtin_amdgcn_sinf(f);
                const float q1 = w.q / (scale * h), q0s = w.q / scale, dq = w.dq / scale;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (i < from || i >= to) continue;
                    const int  tok  = s_tok[mm * 4 + i];
                    if (tok < 0) continue;
                    const bool keep = slot0 + mm * 4 + i < n;
                    const size_t row = zN + tok;
                    float2 v = make_float2(q1 * (ec[i] * rc - os[i] * rs), q1 * (ec[i] * rs + os[i] * rc));
                    float2* po = reinterpret_cast<float2*>(out + row * 2 * K) + k;
                    if (n_lo > 1) { const float2 o = *po; v.x += o.x; v.y += o.y; }
                    *po = keep ? v : make_float2(0.f, 0.f);
                    if (SUMS) {
                        // F0 = rot [ q h (vc G + Gy) - i q' h G ] with G = ec + i os, Gy = oc + i es
                        const float gr_ = q0s * ((float)vc * ec[i] + oc[i]) + dq * os[i];
                        const float gi_ = q0s * ((float)vc * os[i] + es[i]) - dq * ec[i];
                        float c0 = gr_ * rc - gi_ * rs, s0 = gr_ * rs + gi_ * rc;
                        float* pc = cos_sums + row * K + k;
                        float* ps = sin_sums + row * K + k;
                        if (n_lo > 1) { c0 += *pc; s0 += *ps; }
                        *pc = keep ? c0 : 0.f;
                        *ps = keep ? s0 : 0.f;
                    }
                }
            };
            const float* grid = reinterpret_cast<const float*>(s_grid);
            // Fewer tiles than waves: `parts` waves share a tile's rows, at least four groups of 8 each (a wave's reads of the tables are then in flight
            // at once), and meet in LDS.  With the workgroups' shares, us, one workgroup and a wave a tile / so, with the sums and without: 1 x 700, K = 256
            // 27.7 / 22.5 and 24.0 / 22.5, 1 x 1024 30.3 / 24.7 and 26.0 / 23.2, 1 x 2000 40.4 / 36.3 and 33.2 / 31.3, 1 x 1200, K = 512 46.8 / 31.8 and
            // 36.0 / 28.1; with fewer rows than that the meeting costs what it saves (16 x 128, K = 256, without 20.9 / 22.1).
            int parts = 1;
            if (WAVES == 16) while (parts < 16 && tiles * parts * 2 <= 16 && groups >= 8 * parts) parts *= 2;
            if (parts == 1) {
                // (gridDim.z > 1 for one tile at a time only)
                for (int kp = KT * wave; kp < tiles; kp += KT * WAVES) {
                    const int kt = kp * (int)gridDim.z + (int)blockIdx.z;
                    wg_f4 ec[1][KT], os[1][KT], oc[1][KT], es[1][KT];
                    // (an odd number of tiles: the last one twice, written once)
                    wg_product<KT, AHEAD, SUMS, 1>(grid, 0, mid, 0, groups, table + (size_t)kt * 64 + lane, (size_t)L.nkt * 64, kp + 1 < tiles ? 64 : 0, ec, os, oc, es);
#pragma unroll
                    for (int t = 0; t < KT; ++t) finish(kt + t, 0, 4, ec[0][t], os[0][t], oc[0][t], es[0][t]);
                }
            } else {
                const int tile = wave / parts, part = wave % parts, kt = tile * (int)gridDim.z + (int)blockIdx.z;
                constexpr int V = SUMS ? 4 : 2;
                wg_f4* const red = reinterpret_cast<wg_f4*>(s_grid);              // [16 waves][V][64 lanes]
                static_assert(16 * V * 64 * 16 <= WG_ROWS * WG_OBS * 4, "sums of the waves in LDS");
                wg_f4 sum[V];
                if (tile < tiles) {
                    const int share = (groups + parts - 1) / parts, begin = min(part * share, groups);
                    wg_f4 ec[1][1], os[1][1], oc[1][1], es[1][1];
                    wg_product<1, AHEAD, SUMS, 1>(grid, 0, mid, begin, min(begin + share, groups), table + (size_t)kt * 64 + lane, (size_t)L.nkt * 64, 0, ec, os, oc, es);
                    sum[0] = ec[0][0]; sum[1] = os[0][0];
                    if (SUMS) { sum[V - 2] = oc[0][0]; sum[V - 1] = es[0][0]; }
                }
                __syncthreads();                                         // the grid is read
                if (tile < tiles)
#pragma unroll
                    for (int v = 0; v < V; ++v) red[(wave * V + v) * 64 + lane] = sum[v];
                __syncthreads();
                const int each = parts == 2 ? 2 : 1;                     // of the four rows for a wave
                if (tile < tiles && part * each < 4) {
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        sum[v] = red[(tile * parts * V + v) * 64 + lane];
                        for (int o = 1; o < parts; ++o) sum[v] += red[((tile * parts + o) * V + v) * 64 + lane];
                    }
                    finish(kt, part * each, part * each + each, sum[0], sum[1], sum[V - 2], sum[V - 1]);
                }
            }
        }
        if (lowest == WG_MAGIC && ok) s_near[obs] = 1;
    }

    // ---- pairs closer than h / 2 ----
    __syncthreads();
    const int at = wg_lane_id(), token = at & 15;
    const float4 own = src[slot0 + token];
    const uint32_t near = (uint32_t)__builtin_amdgcn_ballot_w64(at < WG_OBS && slot0 + token < n && s_near[token]);
    if (near == 0) return;
    const float closest = 0.5005f / inv_h;
    auto find = [&](int, float dx, float dy, float dz, WgPair& p) {
        float r2, inv, r;
        wg_distance(dx, dy, dz, r2, inv, r);
        p.r = r; p.m = inv; p.A = 0.f;
        return r2 != 0.0f && __builtin_bit_cast(int, __builtin_fmaf(r, inv_h, WG_MAGIC)) == __builtin_bit_cast(int, WG_MAGIC);
    };
    int lengths;
    const bool listed = wg_collect<WAVES>(s_grid, s_cnt, wave, near, src, n, own, closest * closest, lengths, find);
    const int zk = blockIdx.z, Zk = gridDim.z;
    wg_near_units<WAVES, 4>(wave, near, (L.nkt - zk + Zk - 1) / Zk, listed, [&](auto wide, const int q, const int first) {
        constexpr int U = decltype(wide)::value;
        int k[U];
        float kr[U], oc[U], os[U], c[U], s[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            k[u] = (zk + (first + 4 * u + (at >> 4)) * Zk) * 16 + token;             // a lane per wavenumber, of this workgroup's tiles
            kr[u] = (float)((k[u] < K ? (double)wavenumbers[k[u]] : 0.0) * 0.15915494309189533577) * (1.0f / WG_UNIT);
            oc[u] = os[u] = c[u] = s[u] = 0.f;
        }
        auto add = [&](const WgPair& p) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float ph = __builtin_amdgcn_fractf(p.r * kr[u]);
                const float cs = __builtin_amdgcn_cosf(ph), sn = __builtin_amdgcn_sinf(ph);
                oc[u] = __builtin_fmaf(cs, p.m, oc[u]);
                os[u] = __builtin_fmaf(sn, p.m, os[u]);
                if (SUMS) { c[u] += cs; s[u] += sn; }
            }
        };
        if (listed) wg_listed<WAVES>(s_grid, lengths, q, add);
        else wg_every_near(src, n, wg_lane(own.x, q), wg_lane(own.y, q), wg_lane(own.z, q), inv_h, at, add);
        const size_t row = zN + s_tok[q];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k[u] >= K) continue;
            float* o = out + row * 2 * K + 2 * k[u];
            o[0] += oc[u] * WG_UNIT; o[1] += os[u] * WG_UNIT;
            if (SUMS) { cos_sums[row * K + k[u]] += c[u]; sin_sums[row * K + k[u]] += s[u]; }
        }
    });
}

}  // namespace

// The grid pays from about 6e7 (pair, wavenumber) units on, below which two launches and the latency of one workgroup's
// phases are what a call costs, and from 64 wavenumbers on.  Measured, us, grid / direct kernel, with the sums and without: at 6.7e7 units
// 1 x 512 and K = 256 24.2 / 29.9 and 19.0 / 25.6, 16 x 128 and K = 256 21.3 / 26.8 and 17.0 / 22.1, 1 x 1000 and K = 64 23.3 / 36.6 and 21.1 / 31.6;
// at 3.4e7 4 x 256 and K = 128 18.2 / 18.0 and 15.2 / 15.4, 32 x 64 and K = 256 18.7 / 18.1 and 15.4 / 15.0, 1 x 512 and K = 128 19.2 / 21.2 and
// 17.1 / 18.3; 1 x 256 and K = 256 (1.7e7) 19.7 / 12.9 and 15.6 / 11.3.
static bool we_grid_wanted(int Z, int N, int K, int tuning)
{
    return tuning == 0 && K >= 64 && (double)Z * N * N * K >= 6.0e7;
}

extern "C" size_t proteus_we_fwd_workspace_bytes(int Z, int N, int K, int tuning)
{
    if (Z <= 0 || N <= 0 || K <= 0 || N > PROTEUS_WE_MAX_N || K > PROTEUS_WE_MAX_K || Z > 65535) return 0;
    return we_grid_wanted(Z, N, K, tuning) ? wg_layout(Z, N, K, false).bytes : 0;
}

extern "C" int proteus_we_fwd_ws(const float* coords, int coords_layout,
                                 const float* wavenumbers, const uint8_t* mask,
                                 float* out, float* cos_sums, float* sin_sums, void* workspace, size_t workspace_bytes,
                                 int Z, int N, int K, int tuning, void* stream)
{
    const int rc = proteus_we_fwd_check(coords, coords_layout, wavenumbers, mask, out, cos_sums, sin_sums, Z, N, K, tuning);
    if (rc != PROTEUS_OK) return rc;
    if (!workspace || tuning != 0 || workspace_bytes < wg_layout(Z, N, K, false).bytes)
        return proteus_we_fwd(coords, coords_layout, wavenumbers, mask, out, cos_sums, sin_sums, Z, N, K, tuning, stream);
    if ((uintptr_t)workspace & 255) return PROTEUS_ERR_BAD_ALIGNMENT;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const WgLayout L = wg_layout(Z, N, K, false);
    const unsigned prep = (unsigned)Z * (unsigned)L.blocks + (unsigned)((WG_GROUPS * L.nkt + 3) / 4);
    hipLaunchKernelGGL(we_grid_prepare_kernel, dim3(prep), dim3(256), 0, st, coords, coords_layout, wavenumbers, mask, (char*)workspace, Z, N, K);
    dim3 grid((N + WG_OBS - 1) / WG_OBS, Z);
    const size_t lds = (size_t)WG_ROWS * WG_OBS * 4;
    const bool few = (long)grid.x * Z <= 256;
    if (few) grid.z = min(L.nkt, 256 / (int)(grid.x * grid.y));        // (idle compute units spread the same pairs and share the wavenumbers out)
#define WG_GO(S_, W_) hipLaunchKernelGGL((we_grid_kernel<S_, W_>), grid, dim3(W_ * 64), lds, st, (const char*)workspace, wavenumbers, out, cos_sums, sin_sums, Z, N, K)
    if (cos_sums) { if (few) WG_GO(true, 16); else WG_GO(true, 8); }
    else          { if (few) WG_GO(false, 16); else WG_GO(false, 8); }
#undef WG_GO
    return (int)hipGetLastError();
}
