// Anisotropic (C-beta scaled) Wavefunction Embedding forward through distance grids, for gfx950 (MI355X).
//
// What it computes: the sums of we_aniso_fwd.hip, with R = a_i - a_j, r = |R|, A = (b_j . R)/r and phase k (r - cb_k A):
//     F(k, cb) = sum_j e^(i k (r_j - cb A_j)) / r_j (out: cos at even, sin at odd features), d_k = dF/dk, d_cb = dF/dcb.
// The grids are those of we_grid.hip (spreading kernel, octaves, fixed point, product), with two changes:
//   - Position: with c the middle of the scales, r_j - cb_k A_j = (r_j - c A_j) - (cb_k - c) A_j, and it is r - c A that is spread.
//     If all scales are equal, as the module constructs them, that is all there is to it: one grid, as in the isotropic case.
//   - Otherwise the rest of the phase is expanded in Chebyshev polynomials of A/b, b the longest C-beta vector:
//     e^(-i z t) = sum_p (2 - delta_p0) (-i)^p J_p(z) T_p(t),  z = k (cb_k - c) b,  t = A/b     (Jacobi-Anger)
//     with one grid per term, of the weights T_p(A_j/b) / r_j.  The terms come two at a time (two grids share the LDS and a pass
//     over the sources); (z/2)^P / P! < 1e-7 sets their number P: 2 with partial derivatives and equal scales, about 10 for
//     scales 1 +- 0.5 and wavelengths down to 3.7 A.
//   d_cb needs J_p' in place of J_p times k b, d_k that times (cb_k - c) b plus the k-derivative of the grids (we_grid.hip's F0).
// Per pair of tokens and pair of terms: about 40 vector instructions and twelve integer LDS additions, against 10 instructions per
// wavenumber in the direct kernel.
// Pairs that no cell takes (r - c A below h/2, or r so small against r - c A that the weight leaves its fixed-point range) are summed
// directly.  Where the expansion needs so many terms, or the distances so many windows of the grids, that the direct kernel is the faster
// one, and where something is not finite, which only the device can tell, that kernel does the work and this one returns at once.
#include "we_grid.h"
#include "we_aniso_direct.h"

namespace {

using namespace proteus_we_grid;

constexpr int WA_FLUSH = 1024;           // sources between two flushes: 1024 x 2 x 2^20 is what a signed cell holds

// Few enough workgroups of 16 observers for 16 waves each?  (A batch with a padding mask is taken to hold 0.6 of its tokens.)  With
// 8 and 16 waves, partial derivatives of 10 terms at K = 256: 252 workgroups 267 / 240 us, 250 with 4000 sources 549 / 449, 226 of
// 376 unpadded 389 / 349, 304 of 504 unpadded 337 / 356, 454 of 752 472 / 540.
__host__ __device__ inline bool wa_few(const int Z, const int N, const bool padded)
{
    return (padded ? 0.6f : 1.0f) * (float)Z * (float)((N + WG_OBS - 1) / WG_OBS) <= 256.0f;
}

// ---- preparation: one launch for the lists of sources, one for the tables, which need the longest C-beta vector ----

__global__ __launch_bounds__(256)
void we_aniso_grid_sources_kernel(const float* __restrict__ coordsA, const float* __restrict__ coordsB, const int layout,
                                  const uint8_t* __restrict__ mask, char* __restrict__ ws, const int Z, const int N, const int K)
{
    const WgLayout L = wg_layout(Z, N, K, true);
    const int z = blockIdx.x / L.blocks, j = (blockIdx.x % L.blocks) * 256 + threadIdx.x;
    const int slot = wg_compact(coordsA, layout, mask, ws, L, N, blockIdx.x);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (j < N && !(mask && mask[(size_t)z * N + j])) {
        const float* b = coordsB + (size_t)z * N * 3;
        if (layout == PROTEUS_COORDS_SOA) v = make_float4(b[j], b[(size_t)N + j], b[2 * (size_t)N + j], 0.f);
        else                              v = make_float4(b[3 * (size_t)j], b[3 * (size_t)j + 1], b[3 * (size_t)j + 2], 0.f);
    }
    if (slot < L.npad) reinterpret_cast<float4*>(ws + L.sources_b)[(size_t)z * L.npad + slot] = v;
    const float b2 = wg_block_max(v.x * v.x + v.y * v.y + v.z * v.z);
    if (threadIdx.x == 0) reinterpret_cast<float*>(ws + L.lengths)[blockIdx.x] = b2;
}

// Terms after which the series at z has a tail below `tail`; more than WG_MAX_TERMS if there is no such number.
__device__ __forceinline__ int wa_terms(const float z, const float tail)
{
    float t = 1.0f;
    int n = 1;
    for (; n <= WG_MAX_TERMS; ++n) { t *= 0.5f * z / (float)n; if (2.0f * t < tail) break; }
    return n;
}

// The batch items' boxes, read by a block of 256 threads: as many lanes share an item as it has boxes.  `fetch` sends off a thread's
// first two, `longest` returns the length of the longest diagonal of its items (infinite if one holds a token that is not finite).
struct WaBoxes {
    const WgBox* __restrict__ boxes;
    int Z, nbox, lanes, z, i;
    WgBox q[2];
    __device__ __forceinline__ void fetch(const WgBox* __restrict__ from, const int Z_, const int nbox_)
    {
        boxes = from; Z = Z_; nbox = nbox_;
        lanes = nbox > 32 ? 64 : nbox > 16 ? 32 : nbox > 8 ? 16 : nbox > 4 ? 8 : nbox > 2 ? 4 : nbox;
        z = (int)threadIdx.x / lanes; i = (int)threadIdx.x % lanes;
        const float inf = __builtin_inff();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            q[u] = WgBox{{inf, inf, inf}, {-inf, -inf, -inf}, 0.f, 0.f};                // (as of padded tokens only)
            if (z < Z && i + u * lanes < nbox) q[u] = boxes[(size_t)z * nbox + i + u * lanes];
        }
    }
    __device__ __forceinline__ float longest()
    {
        float far = 0.f;
        const int step = 256 / lanes;
        for (int item = z; item - z < Z; item += step) {                                // (all lanes of a wave meet in the exchanges)
            float lo[3], hi[3], bad = 0.f;
#pragma unroll
            for (int c = 0; c < 3; ++c) { lo[c] = 3.0e38f; hi[c] = -3.0e38f; }
            auto add = [&](const WgBox& w) {
                bad = fmaxf(bad, w.bad);
#pragma unroll
                for (int c = 0; c < 3; ++c) { lo[c] = fminf(lo[c], w.lo[c]); hi[c] = fmaxf(hi[c], w.hi[c]); }
            };
            if (item == z) { add(q[0]); add(q[1]); }
            for (int j = item == z ? i + 2 * lanes : i; item < Z && j < nbox; j += lanes) add(boxes[(size_t)item * nbox + j]);
#pragma unroll
            for (int o = 1; o < 64; o *= 2) {
                if (o >= lanes) break;
                bad = fmaxf(bad, __shfl_xor(bad, o));
#pragma unroll
                for (int c = 0; c < 3; ++c) { lo[c] = fminf(lo[c], __shfl_xor(lo[c], o)); hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], o)); }
            }
            const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
            if (lo[0] <= hi[0]) far = fmaxf(far, __builtin_sqrtf(dx * dx + dy * dy + dz * dz));
            far += bad;
        }
        return far;
    }
};

__global__ __launch_bounds__(256)
void we_aniso_grid_tables_kernel(const float* __restrict__ cb_magnitudes, const float* __restrict__ wavenumbers,
                                 char* __restrict__ ws, const int Z, const int N, const int K, const int partials, const int few)      // few: workgroups that share a batch's wavenumbers, 0 for the large launch
{
    const WgLayout L = wg_layout(Z, N, K, true);
    const int tid = threadIdx.x, lane = tid & 63;
    // Everything that needs no other answer meets in one reduction, the first values of every list loaded before any of them is
    // looked at: a list after the other cost a trip to memory each (8192 tokens with equal scales: this launch 5.8 us, 8.3 so and with
    // the tiles below for a single grid, which has no use for them).
    const float* lengths = reinterpret_cast<const float*>(ws + L.lengths);
    const int* counts = reinterpret_cast<const int*>(ws + L.counts);
    const bool first = blockIdx.x == 0;                                 // the block that estimates
    WaBoxes boxes;
    if (first) boxes.fetch(reinterpret_cast<const WgBox*>(ws + L.boxes), Z, L.nbox);
    int n0 = first && tid < Z ? counts[tid] : 0;
    float b2 = tid < Z * L.blocks ? lengths[tid] : 0.f;
    float hi = -3.0e38f, lo = -3.0e38f, km = 0.f;                       // lo: largest of -cb
    bool bad = false;
    const float c0 = tid < K ? cb_magnitudes[tid] : 0.f, w0 = tid < K ? wavenumbers[tid] : 0.f;
    for (int k = tid; k < K; k += 256) {
        const float c = k == tid ? c0 : cb_magnitudes[k], w = fabsf(k == tid ? w0 : wavenumbers[k]);
        bad |= !(fabsf(c) < 1.0e18f);
        hi = fmaxf(hi, c); lo = fmaxf(lo, -c); km = fmaxf(km, w < 3.0e38f ? w : __builtin_inff());
    }
    for (int i = tid + 256; i < Z * L.blocks; i += 256) b2 = fmaxf(b2, lengths[i]);
    float pairs = 0.f, nmax = 0.f, groups = 0.f, extent = 0.f;
    if (first) {
        for (int i = tid; i < Z; i += 256) {
            if (i > tid) n0 = counts[i];
            const float n = (float)n0;
            pairs += n * n; nmax = fmaxf(nmax, n); groups += __builtin_ceilf(n / WG_OBS);
        }
        extent = boxes.longest() * (1.0f / WG_UNIT);
    }
    float all[8] = {pairs, groups, km, bad ? __builtin_inff() : b2, hi, lo, nmax, extent};
    wg_block_reduce<2>(all);
    pairs = all[0]; groups = all[1]; nmax = all[6]; extent = all[7];
    const float inv_h = wg_cells_per_length(all[2]);
    const double h = 1.0 / (double)inv_h;
    const float mid = 0.5f * (all[4] - all[5]), b = __builtin_sqrtf(all[3]) * 1.0001f;
    float z = tid < K ? fabsf(w0 * (c0 - mid)) : 0.f;
    for (int k = tid + 256; k < K; k += 256) z = fmaxf(z, fabsf(wavenumbers[k] * (cb_magnitudes[k] - mid)));
    z = wg_block_max(z) * b;
    // number of terms: the tail of the series starts with 2 J_P(z) <= 2 (z/2)^P / P! (at the one wavenumber where z is largest), that of
    // its derivative with J_(P-1)(z)
    int terms = 0;
    if (b < 1.0e18f && z < 20.0f) {
        terms = wa_terms(z, 3.0e-7f) + partials;
        if (terms > WG_MAX_TERMS) terms = 0;
    }
    // (The first block answers, the others fill the tables.)
    if (terms > 0 && first) {
        // The direct kernel or the grids?  Estimated microseconds: the direct kernel takes 0.34 ps per pair and wavenumber with partial
        // derivatives (0.36 to 0.40 where it has few workgroups) and 0.24 without.  A pass over the sources (8 waves, K = 256, 1 x 1000 ... 8 x 2000 tokens, 4 to 12 terms) takes a round
        // of workgroups (two per compute unit) 22 us for its grids and products and 0.059 us per source, down to 0.026 for few workgroups.
        const bool  one     = terms == 1;                                // (a single grid: no partial derivatives)
        const int   most    = one ? WgGrid<1>::CELLS : WgGrid<2>::CELLS;
        const float cells   = 0.7f * extent * inv_h;
        const float windows = __builtin_ceilf(fmaxf(1.0f, cells / (float)most));
        const float rounds  = groups * (1.0f / 512.0f), share = fminf(1.0f, rounds);
        // (16 waves, 28 batches of 1 x 500 ... 2 x 2000 tokens, K = 128 and 256: a preparation of 37 to 53 us, and per pass 0.0128 us per source,
        // 0.3 ns per cell and wavenumber, half of that without partial derivatives, and 10 us for the flushes of more than 1024 sources.
        // Of the cells' part four fifths are shared by `few` workgroups, which takes 5 us: 1 x 1000, K = 512 203 us with the grids and 198 without.)
        const float passes  = (float)((terms + 1) / 2) * windows;
        float grid   = few ? (partials ? 53.0f : 37.0f) + (few > 1 ? 5.0f : 0.0f) + passes * (0.0128f * nmax + (partials ? 3.0e-4f : 1.4e-4f) * (float)K * (0.2f + 0.8f / (float)few) * cells / windows
                                                                    + (nmax > (float)WA_FLUSH ? 10.0f : 0.0f))
                           : passes * (22.0f + (0.026f + 0.033f * share) * nmax) * fmaxf(1.0f, rounds);
        float direct = pairs * (float)K * (partials ? (few ? 3.7e-7f : 3.4e-7f) : 2.4e-7f);
        if (one) {
            // A single grid, 60 batches of 1 x 1000 ... 32 x 500 tokens, K = 64 to 256, extents of up to 16 windows.  Grids / direct, us:
            // 1 x 2000 K = 64 1 window 43 / 172, 4 114 / 180, 7 212 / 179, 13 402 / 179; 1 x 4000 K = 64 5 234 / 350, 9 430 / 353; 1 x 4000 K = 256
            // 10 598 / 1074; 8 x 1000 K = 256 6 387 / 527, 11 742 / 529.  The direct kernel takes 0.086 us per source where its workgroups do not fill the chip.
            grid   = 12.0f + windows * (few ? 10.0f + 0.008f * nmax + 0.05f * (float)K
                                            : (6.0f + (0.5f + 0.5f * share) * (0.0118f * nmax + 0.18f * (float)K)) * fmaxf(1.0f, rounds));
            direct = fmaxf(direct, 0.086f * nmax);
        }
        if (!(grid < direct) || !(cells + fabsf(mid) * b * inv_h < (float)(most * WG_MAX_WINDOWS))) terms = 0;
    }
    if (blockIdx.x == 0 && tid == 0) {
        WgParams* p = reinterpret_cast<WgParams*>(ws);
        p->inv_h = inv_h; p->h = (float)h; p->cb_mid = mid; p->b_max = b; p->terms = terms;
    }
    // A tile of 16 wavenumbers takes part in the terms that its own z asks for (at a tenth of the tail above, which only the worst
    // wavenumber of all comes near): 267 -> 251 us at 4 x 1000 tokens, 10 terms, partial derivatives.
    if (blockIdx.x == 0) {
        for (int t = tid; terms > 1 && t < L.nkt; t += 256) {
            float zt = 0.f;
            for (int k = t * 16; k < min(t * 16 + 16, K); ++k) zt = fmaxf(zt, fabsf(wavenumbers[k] * (cb_magnitudes[k] - mid)));
            reinterpret_cast<int*>(ws + L.tiles)[t] = min(terms, wa_terms(zt * b, 3.0e-8f) + partials);
        }
        return;
    }
    const int unit = ((int)blockIdx.x - 1) * 4 + (tid >> 6);
    const int rows = WG_GROUPS * L.nkt;
    if (unit < rows) { wg_fill_tables(wavenumbers, ws, L, K, h, unit); return; }
    // (2 - delta_p0) J_p and its derivative: four orders of 16 wavenumbers per wave, by the power series in double precision (|z| <= 10)
    const int kt = (unit - rows) % L.nkt, p = (unit - rows) / L.nkt * 4 + (lane >> 4), k = kt * 16 + (lane & 15);
    if (p >= terms) return;
    const double x = k < K ? 0.5 * (double)(wavenumbers[k] * (cb_magnitudes[k] - mid)) * (double)b : 0.0;
    auto bessel = [&](const int n) {
        double term = 1.0;
        for (int i = 1; i <= n; ++i) term *= x / (double)i;
        double s = term;
        for (int m = 1; m <= 40; ++m) { term *= -x * x / ((double)m * (double)(m + n)); s += term; if (fabs(term) <= 1.0e-17 * fabs(s)) break; }
        return s;
    };
    const double j = bessel(p), jd = p ? 0.5 * (bessel(p - 1) - bessel(p + 1)) : -bessel(1);
    const double f = p ? 2.0 : 1.0;
    reinterpret_cast<float2*>(ws + L.terms)[(size_t)p * L.nkt * 16 + k] = make_float2((float)(f * j), (float)(f * jd));
}

// ---- main kernel ----

// What decides whether a pair has a cell: n = rint((r - c A)/h) >= 1 and 2^floor(log2 n) h / r <= 2.
struct Place { float A, r, inv, u, um, x, c; uint32_t eb; };

__device__ __forceinline__ Place wa_place(const float dx, const float dy, const float dz, const float4& b, const float mid, const float inv_h, const float magic, const uint32_t emask, float& r2)
{
    Place p;
    wg_distance(dx, dy, dz, r2, p.inv, p.r);
    p.A = (b.x * dx + b.y * dy + b.z * dz) * p.inv;
    const float s = __builtin_fmaf(-mid, p.A, p.r);
    p.u  = __builtin_fmaf(s, inv_h, magic);
    p.um = __builtin_fmaxf(p.u, magic);                       // magic + n (a value that is not a number becomes 0)
    const float nf = p.um - magic;
    p.x  = __builtin_fmaf(s, inv_h, -nf);
    p.eb = __builtin_bit_cast(uint32_t, nf) & emask;
    p.c  = p.inv * __builtin_bit_cast(float, p.eb);           // 2^e / r; 0 for n = 0
    return p;
}

// Source j's pair with an observer: has it no cell?
__device__ __forceinline__ bool wa_no_cell(const float4& b, const float dx, const float dy, const float dz, const float mid, const float inv_h, WgPair& p)
{
    float r2;
    const Place w = wa_place(dx, dy, dz, b, mid * WG_UNIT, inv_h, WG_MAGIC, 0xff800000u, r2);
    p.r = w.r * (1.0f / WG_UNIT); p.m = w.inv * WG_UNIT; p.A = w.A;
    return r2 != 0.0f && (!(w.u > WG_MAGIC) || w.c > 2.0f * inv_h);
}

// add(pair) for the pairs of one observer that have no cell, more of them than the lists hold.
template <class Add>
__device__ __forceinline__ void wa_every_near(const float4* __restrict__ src, const float4* __restrict__ srcb, const int n, const float xi, const float yi, const float zi,
                                              const float mid, const float inv_h, const int lane, Add add)
{
    float4 next = src[lane], nextb = srcb[lane];
    for (int j0 = 0; j0 < n; j0 += 64) {
        const float4 q = next, qb = nextb;
        next = src[j0 + 64 + lane]; nextb = srcb[j0 + 64 + lane];       // (past the end: inside the lists' padding)
        WgPair mine;
        uint64_t todo = __builtin_amdgcn_ballot_w64(wa_no_cell(qb, xi - q.x, yi - q.y, zi - q.z, mid, inv_h, mine) && j0 + lane < n);
        while (todo) {
            const int b = __builtin_ctzll(todo);
            todo &= todo - 1;
            WgPair p;
            p.r = wg_lane(mine.r, b); p.m = wg_lane(mine.m, b); p.A = wg_lane(mine.A, b);
            add(p);
        }
    }
}

// GP  grids per pass over the sources: 1 where the expansion has a single term (then its weights are those of the isotropic kernel,
//     unsigned denormals), 2 otherwise (signed weights, through the low bits of a magic sum)
template <bool GRADS, int GP, int WAVES, bool SHARED>
__device__ __forceinline__ void wa_grids(uint32_t* s_grid, int* s_near, const int* s_tok, const char* __restrict__ ws, const WgLayout& L,
                                         const float* __restrict__ cb_magnitudes, const float* __restrict__ wavenumbers,
                                         float* __restrict__ out, float* __restrict__ d_cb, float* __restrict__ d_k,
                                         const float4* __restrict__ src, const float4* __restrict__ srcb, const float4& me, const bool ok,
                                         const int n, const int slot0, const int ncell, const size_t zN, const int K)
{
    const int zk = SHARED ? blockIdx.z : 0, Zk = SHARED ? gridDim.z : 1;            // of the tiles of 16 wavenumbers, this workgroup's are zk, zk + Zk, ...
    constexpr int THREADS = WAVES * 64;
    constexpr int STEP   = WAVES * 8;                     // sources per iteration: a wave takes 16 observers x 4 sources, twice
    constexpr int CHUNKS = (WG_ROWS * WG_OBS / 4 + THREADS - 1) / THREADS;
    constexpr int CELLS  = WgGrid<GP>::CELLS;
    constexpr int FLUSH  = GP == 1 ? WG_FLUSH : WA_FLUSH;
    constexpr bool SIGNED = GP == 2;
    const int tid = threadIdx.x, lane = tid & 63, obs = lane & 15, mm = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const WgParams* __restrict__ params = reinterpret_cast<const WgParams*>(ws);
    const float inv_h = params->inv_h * (1.0f / WG_UNIT), h = params->h, mid_cb = params->cb_mid, bmax = params->b_max;
    const int terms = params->terms;
    const float4* __restrict__ table = reinterpret_cast<const float4*>(ws + L.table);
    const WgWave* __restrict__ waves = reinterpret_cast<const WgWave*>(ws + L.waves);
    const float2* __restrict__ coef = reinterpret_cast<const float2*>(ws + L.terms);

    const int nit = (n + STEP - 1) / STEP, quarter = nit * (STEP / 4);
    const bool flushes = nit * STEP > FLUSH;
    const float scale = GP == 1 ? (flushes ? 1048000.0f : fminf(4190000.0f, 2147000000.0f / (float)(nit * STEP)))
                                : (flushes ? 1048000.0f : fminf(2090000.0f, 1073000000.0f / (float)(nit * STEP)));
    const WgKernel kernel(GP == 1 ? scale * h * 0x1p-137f : scale * h * WG_UNIT);
    const float magic = wg_vgpr(WG_MAGIC), inv_hv = wg_vgpr(inv_h), midv = wg_vgpr(mid_cb * WG_UNIT), climit = wg_vgpr(2.0f * inv_h);
    const float inv_b = wg_vgpr(bmax > 0.f ? 1.0f / bmax : 0.f);
    uint32_t emask = 0xff800000u, mbits = WG_MAGIC_BITS;
    asm volatile("" : "+v"(emask), "+v"(mbits));
    float lowest = 3.0e38f, largest = 0.f;

    for (int p0 = 0; p0 < terms; p0 += GP) {
        for (int n_lo = 1; n_lo <= ncell; n_lo += CELLS) {
            const int cells = min(CELLS, ncell + 1 - n_lo);
            const int e_lo  = 31 - __builtin_clz(n_lo), e_hi = 31 - __builtin_clz(n_lo + cells - 1);
            const int used  = WG_R0 + cells + 5 + WG_OCT * (e_hi - e_lo);
            wg_f4 facc[CHUNKS];
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) facc[i] = wg_f4{0.f, 0.f, 0.f, 0.f};
            __syncthreads();
            wg_clear<GP, THREADS>(s_grid, used);
            __syncthreads();

            uint32_t base = (uint32_t)(uintptr_t)(wg_lds_u32*)s_grid + (uint32_t)((WG_R0 - n_lo - WG_OCT * e_lo) * WG_OBS + obs) * 4u
                            - (WG_MAGIC_BITS << 6) - 127u * (WG_OCT * WG_OBS * 4u);
            uint32_t trash = (uint32_t)(uintptr_t)(wg_lds_u32*)s_grid + (uint32_t)(WgGrid<GP>::TRASH * WG_OBS + obs) * 4u;
            asm volatile("" : "+v"(base), "+v"(trash));
            const uint32_t first = WG_MAGIC_BITS + (uint32_t)n_lo;

            const int from = (lane >> 4) * quarter + wave * 2;
            const float4* p = src + from;
            const float4* pb = srcb + from;
            float ua, ca;
            auto spread = [&](const float4& q, const float4& qb, auto second) {
                float r2;
                const Place w = wa_place(me.x - q.x, me.y - q.y, me.z - q.z, qb, midv, inv_hv, magic, emask, r2);
                float wt[6];
                kernel.template weights<GP == 1>(w.x, w.c, wt);
                const uint32_t ub = __builtin_bit_cast(uint32_t, w.um);
                uint32_t at = (ub << 6) + base + (w.eb >> 14);
                // (both conditions looked at: with && the compiler branches on the first, twice a pair)
                const bool in = (ub - first < (uint32_t)cells) & !(w.c > climit);
                at = in ? at : trash;
                // (the second of two pairs answers for both in instructions of three operands)
                if (decltype(second)::value) {
                    lowest  = __builtin_fminf(__builtin_fminf(ua, w.u), lowest);
                    largest = __builtin_fmaxf(__builtin_fmaxf(ca, w.c), largest);
                } else { ua = w.u; ca = w.c; }
                wg_lds_u32* a = (wg_lds_u32*)(uintptr_t)at;
                auto add = [&](const int row, const uint32_t v) { __hip_atomic_fetch_add(a + row * WG_OBS, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
                if (GP == 1) {
#pragma unroll
                    for (int l = 0; l < 6; ++l) add(l, __builtin_bit_cast(uint32_t, wt[l]));
                } else {
                    // T_p0 and T_(p0+1) of t = A/b by their recurrence, two orders at a time
                    const float t = w.A * inv_b, t2 = t + t;
                    float Ta = 1.0f, Tb = t;
                    for (int i = 0; i < p0; i += 2) { Ta = __builtin_fmaf(t2, Tb, -Ta); Tb = __builtin_fmaf(t2, Ta, -Tb); }
#pragma unroll
                    for (int l = 0; l < 6; ++l) {
                        add(l, __builtin_bit_cast(uint32_t, __builtin_fmaf(wt[l], Ta, magic)) - mbits);
                        add(l + WgGrid<GP>::ROWS, __builtin_bit_cast(uint32_t, __builtin_fmaf(wt[l], Tb, magic)) - mbits);
                    }
                }
            };
            float4 qa = p[0], qb = p[1], ba = pb[0], bb = pb[1];
            int until = flushes ? FLUSH / STEP : nit;
            for (int it = 0;;) {
                for (; it < until; ++it) {
                    p += STEP / 4; pb += STEP / 4;
                    spread(qa, ba, wg_false{});
                    qa = p[0]; ba = pb[0];
                    spread(qb, bb, wg_true{});
                    qb = p[1]; bb = pb[1];
                }
                if (!flushes) break;
                __syncthreads();
                wg_flush<GP, THREADS, CHUNKS, SIGNED>(s_grid, facc, used, it >= nit);
                __syncthreads();
                if (it >= nit) break;
                until = min(it + FLUSH / STEP, nit);
            }
            if (!flushes) __syncthreads();
            wg_combine<GP, THREADS, CHUNKS, SIGNED>(s_grid, facc, n_lo, cells, flushes);
            __syncthreads();

            const int mid    = (cells + 6) / 2;
            const int groups = (mid + 7) / 8;
            const int vc     = n_lo - 3 + mid;
            const bool more  = n_lo > 1 || p0 > 0;
            for (int kp = wave * Zk + zk; kp < L.nkt; kp += WAVES * Zk) {
                const int mine = GP == 1 ? 1 : __builtin_amdgcn_readfirstlane(reinterpret_cast<const int*>(ws + L.tiles)[kp]);
                if (p0 >= mine) continue;
                const int k = kp * 16 + obs;
                // (a tile that takes part in the first of two terms only runs the product of the second for nothing, every other pass)
                wg_f4 ec[GP][1], os[GP][1], oc[GP][1], es[GP][1];
                wg_product<1, WAVES == 16 ? 4 : 2, GRADS, GP>(reinterpret_cast<const float*>(s_grid), WgGrid<GP>::ROWS * WG_OBS, mid, 0, groups,
                                                              table + (size_t)kp * 64 + lane, (size_t)L.nkt * 64, 0, ec, os, oc, es);
                // (what earlier terms and windows left, all loads in flight at once; with the two grids sharing the reads of the tables 251 -> 240 us
                // at 4 x 1000 tokens, 10 terms, partial derivatives)
                int tok[4];
                float2 o[4], ob[4], okk[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    tok[i] = k < K ? s_tok[mm * 4 + i] : -1;
                    o[i] = ob[i] = okk[i] = make_float2(0.f, 0.f);
                    if (more && tok[i] >= 0) {
                        const size_t at = (zN + tok[i]) * K + k;
                        o[i] = reinterpret_cast<const float2*>(out)[at];
                        if (GRADS) { ob[i] = reinterpret_cast<const float2*>(d_cb)[at]; okk[i] = reinterpret_cast<const float2*>(d_k)[at]; }
                    }
                }
                const WgWave w = waves[k];
                const double ph = w.rev * (double)vc;
                const float f  = (float)(ph - __builtin_floor(ph));
                const float rc = __builtin_amdgcn_cosf(f), rs = __builtin_amdgcn_sinf(f);
                const float q1 = w.q / (scale * h), q0s = w.q / scale, dq = w.dq / scale;
                const float wn = k < K ? wavenumbers[k] : 0.f, kb = wn * bmax, db = k < K ? (cb_magnitudes[k] - mid_cb) * bmax : 0.f;
#pragma unroll
                for (int g = 0; g < GP; ++g) {
                    if (p0 + g >= mine) break;
                    const float2 J = coef[(size_t)(p0 + g) * L.nkt * 16 + k];
                    const int turn = (p0 + g) & 3;                                 // (-i)^p
                    auto turned = [&](const float x, const float y) {
                        return turn == 0 ? make_float2(x, y) : turn == 1 ? make_float2(y, -x) : turn == 2 ? make_float2(-x, -y) : make_float2(-y, x);
                    };
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float e = ec[g][0][i], s = os[g][0][i];
                        const float2 F = turned(q1 * (e * rc - s * rs), q1 * (e * rs + s * rc));
                        o[i].x += J.x * F.x; o[i].y += J.x * F.y;
                        if (GRADS) {
                            const float gr = q0s * ((float)vc * e + oc[g][0][i]) + dq * s;
                            const float gi = q0s * ((float)vc * s + es[g][0][i]) - dq * e;
                            const float2 D = turned(-(gr * rs + gi * rc), gr * rc - gi * rs);          // dF/dk = i F0
                            ob[i].x  += kb * J.y * F.x;                 ob[i].y  += kb * J.y * F.y;
                            okk[i].x += db * J.y * F.x + J.x * D.x;     okk[i].y += db * J.y * F.y + J.x * D.y;
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (tok[i] < 0) continue;
                    const bool keep = slot0 + mm * 4 + i < n;
                    const size_t at = (zN + tok[i]) * K + k;
                    const float2 zero = make_float2(0.f, 0.f);
                    reinterpret_cast<float2*>(out)[at] = keep ? o[i] : zero;
                    if (GRADS) { reinterpret_cast<float2*>(d_cb)[at] = keep ? ob[i] : zero; reinterpret_cast<float2*>(d_k)[at] = keep ? okk[i] : zero; }
                }
            }
        }
    }
    if (ok && (!(lowest > WG_MAGIC) || largest > climit)) s_near[obs] = 1;
}

// WAVES  8: two workgroups share a compute unit; 16: twice the waves on the same observers, for launches whose workgroups with
//        unpadded observers have a compute unit to themselves
// SHARED  workgroups of every blockIdx.z have the same slots and, of the tiles of 16 wavenumbers, every gridDim.z-th (of 16 waves, where compute
//        units would be idle; us, before / so, partial derivatives: 1 x 2000, K = 256, scales spread by 0.2 398 / 270, compact 271 / 236, 1 x 1500, K = 512
//        431 / 317, 2 x 1000, K = 256 206 / 198.  Launches of one share have kernels of their own: the two scalars cost registers, 4 x 1000 279 / 287)
template <bool GRADS, int WAVES, bool SHARED>
__global__ __launch_bounds__(WAVES * 64, 4)
void we_aniso_grid_kernel(const char* __restrict__ ws, const float* __restrict__ cb_magnitudes, const float* __restrict__ wavenumbers,
                          float* __restrict__ out, float* __restrict__ d_cb, float* __restrict__ d_k, const int Z, const int N, const int K)
{
    constexpr int THREADS = WAVES * 64;
    extern __shared__ __align__(16) uint32_t s_grid[];
    __shared__ float s_red[WAVES];
    __shared__ int   s_near[WG_OBS];
    __shared__ int   s_tok[WG_OBS];
    __shared__ int   s_cnt[WAVES];

    const WgLayout L = wg_layout(Z, N, K, true);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z = blockIdx.y;
    const size_t zN = (size_t)z * N;
    const int n = reinterpret_cast<const int*>(ws + L.counts)[z];
    const float4* __restrict__ src  = reinterpret_cast<const float4*>(ws + L.sources) + (size_t)z * L.npad;
    const float4* __restrict__ srcb = reinterpret_cast<const float4*>(ws + L.sources_b) + (size_t)z * L.npad;
    const WgParams* __restrict__ params = reinterpret_cast<const WgParams*>(ws);
    const float inv_h = params->inv_h * (1.0f / WG_UNIT), mid_cb = params->cb_mid;
    const int terms = params->terms;
    if (terms == 0) return;                                    // the direct kernel's

    const int slot0 = blockIdx.x * WG_OBS;
    const int obs   = lane & 15;
    const float4 me = src[slot0 + obs];
    const bool ok   = slot0 + obs < n;
    if (tid < WG_OBS) { s_tok[tid] = slot0 + tid < N ? __builtin_bit_cast(int, me.w) : -1; s_near[tid] = 0; }
    if (slot0 >= n) {
        __syncthreads();
        for (int q = 0; q < WG_OBS; ++q) {
            const int t = s_tok[q];
            if (t < 0) continue;
            const size_t row = (zN + t) * 2 * K;
            for (int k = tid; k < 2 * K; k += THREADS) { out[row + k] = 0.f; if (GRADS) { d_cb[row + k] = 0.f; d_k[row + k] = 0.f; } }
        }
        return;
    }

    // (The tables' launch has seen to it that 0.7 of an item's extent, and b, stay within WG_MAX_WINDOWS windows; the far corner and
    // the observers' own radius are at most twice that.)
    const int ncell = __builtin_amdgcn_readfirstlane((int)((wg_reach<WAVES>(me, ok, reinterpret_cast<const WgBox*>(ws + L.boxes) + (size_t)z * L.nbox, L.nbox, s_red)
                                                            + fabsf(mid_cb) * params->b_max * WG_UNIT) * inv_h + 2.0f));
    if (!GRADS && terms == 1) wa_grids<GRADS, 1, WAVES, SHARED>(s_grid, s_near, s_tok, ws, L, cb_magnitudes, wavenumbers, out, d_cb, d_k, src, srcb, me, ok, n, slot0, ncell, zN, K);
    else                      wa_grids<GRADS, 2, WAVES, SHARED>(s_grid, s_near, s_tok, ws, L, cb_magnitudes, wavenumbers, out, d_cb, d_k, src, srcb, me, ok, n, slot0, ncell, zN, K);

    // ---- pairs without a cell ----
    __syncthreads();
    const int at = wg_lane_id(), token = at & 15;
    const float4 own = src[slot0 + token];
    const uint32_t near = (uint32_t)__builtin_amdgcn_ballot_w64(at < WG_OBS && slot0 + token < n && s_near[token]);
    if (near == 0) return;
    // They lie within |c A| + h / 2: without a cell r - c A <= h/2 or 2^floor(log2 n) h / r > 2, and 2^floor(log2 n) h <= r - c A + h/2.
    const float closest = (fabsf(mid_cb) * WG_UNIT * params->b_max + 0.5f / inv_h) * 1.001f;
    auto find = [&](int j, float dx, float dy, float dz, WgPair& p) {
        return wa_no_cell(srcb[j], dx, dy, dz, mid_cb, inv_h, p);
    };
    int lengths;
    const bool listed = wg_collect<WAVES>(s_grid, s_cnt, wave, near, src, n, own, closest * closest, lengths, find);
    const int zk = SHARED ? blockIdx.z : 0, Zk = SHARED ? gridDim.z : 1;
    wg_near_units<WAVES, 2>(wave, near, (L.nkt - zk + Zk - 1) / Zk, listed, [&](auto wide, const int q, const int first) {
        constexpr int U = decltype(wide)::value;
        int k[U];
        float kr[U], cb[U], s[U][GRADS ? 6 : 2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            k[u] = (zk + (first + 4 * u + (at >> 4)) * Zk) * 16 + token;             // a lane per wavenumber, of this workgroup's tiles
            kr[u] = (float)((k[u] < K ? (double)wavenumbers[k[u]] : 0.0) * 0.15915494309189533577);
            cb[u] = k[u] < K ? cb_magnitudes[k[u]] : 0.f;
#pragma unroll
            for (int i = 0; i < (GRADS ? 6 : 2); ++i) s[u][i] = 0.f;
        }
        auto add = [&](const WgPair& p) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float ph = __builtin_amdgcn_fractf(__builtin_fmaf(-cb[u], p.A, p.r) * kr[u]);
                const float cs = __builtin_amdgcn_cosf(ph), sn = __builtin_amdgcn_sinf(ph);
                s[u][0] = __builtin_fmaf(cs, p.m, s[u][0]);
                s[u][1] = __builtin_fmaf(sn, p.m, s[u][1]);
                if constexpr (GRADS) {
                    s[u][2] += cs; s[u][3] += sn;
                    s[u][4] = __builtin_fmaf(cs, p.m * p.A, s[u][4]);
                    s[u][5] = __builtin_fmaf(sn, p.m * p.A, s[u][5]);
                }
            }
        };
        if (listed) wg_listed<WAVES>(s_grid, lengths, q, add);
        else wa_every_near(src, srcb, n, wg_lane(own.x, q), wg_lane(own.y, q), wg_lane(own.z, q), mid_cb, inv_h, at, add);
        const size_t row = (zN + s_tok[q]) * 2 * K;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k[u] >= K) continue;
            auto put = [&](float* to, float re, float im) { to[row + 2 * k[u]] += re; to[row + 2 * k[u] + 1] += im; };
            put(out, s[u][0], s[u][1]);
            if constexpr (GRADS) {
                put(d_k, -s[u][3] + cb[u] * s[u][5], s[u][2] - cb[u] * s[u][4]);
                put(d_cb, wavenumbers[k[u]] * s[u][5], -wavenumbers[k[u]] * s[u][4]);
            }
        }
    });
}

// What the grids need beside the direct kernel, two launches of preparation and one that finds nothing to do, costs 13 us.  Without
// partial derivatives the scales are likely to be equal, where the grid wins from about 1 x 512 tokens on (K = 256: 1 x 512 41 / 49 us,
// 1 x 2000 79 / 272, 8 x 1000 67 / 486); with them they are likely to differ, and the grids win where the direct kernel takes 400 us or more
// (4 x 1000 240 / 365, 1 x 2000 268 / 398, 8 x 1000 484 / 701, compact 1 x 8192 1.25 / 5.5 ms; below, 1 x 1500 305 / 238).  A batch with a padding mask is taken to hold 0.4 of its pairs.
bool we_aniso_grid_wanted(int Z, int N, int K, bool partials, bool padded, int tuning)
{
    return tuning == 0 && K >= 64 && (padded ? 0.4 : 1.0) * Z * N * N * K >= (partials ? 1.0e9 : 2.0e8);
}

}  // namespace

extern "C" size_t proteus_we_aniso_fwd_workspace_bytes(int Z, int N, int K, int partials, int padded, int tuning)
{
    if (Z <= 0 || N <= 0 || K <= 0 || N > PROTEUS_WE_MAX_N || K > PROTEUS_WE_MAX_K || Z > 65535) return 0;
    return we_aniso_grid_wanted(Z, N, K, partials != 0, padded != 0, tuning) ? wg_layout(Z, N, K, true).bytes : 0;
}

extern "C" int proteus_we_aniso_fwd_ws(const float* coordsA, const float* coordsB, int coords_layout,
                                       const float* cb_magnitudes, const float* wavenumbers, const uint8_t* mask,
                                       float* out, float* d_cb, float* d_k, void* workspace, size_t workspace_bytes,
                                       int Z, int N, int K, int tuning, void* stream)
{
    const int rc = proteus_we_aniso_fwd_check(coordsA, coordsB, coords_layout, cb_magnitudes, wavenumbers, mask, out, d_cb, d_k, Z, N, K, tuning);
    if (rc != PROTEUS_OK) return rc;
    const WgLayout L = wg_layout(Z, N, K, true);
    if (!workspace || tuning != 0 || workspace_bytes < L.bytes)
        return proteus_we_aniso_fwd(coordsA, coordsB, coords_layout, cb_magnitudes, wavenumbers, mask, out, d_cb, d_k, Z, N, K, tuning, stream);
    if ((uintptr_t)workspace & 255) return PROTEUS_ERR_BAD_ALIGNMENT;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    char* ws = (char*)workspace;
    hipLaunchKernelGGL(we_aniso_grid_sources_kernel, dim3((unsigned)Z * (unsigned)L.blocks), dim3(256), 0, st, coordsA, coordsB, coords_layout, mask, ws, Z, N, K);
    dim3 grid((N + WG_OBS - 1) / WG_OBS, Z);
    // (idle compute units spread the same pairs and share the wavenumbers out)
    const int few = wa_few(Z, N, mask != nullptr) ? max(1, min(L.nkt, 256 / (int)(grid.x * grid.y))) : 0;
    if (few) grid.z = few;
    const unsigned units = (unsigned)((WG_GROUPS + (WG_MAX_TERMS + 3) / 4) * L.nkt);
    hipLaunchKernelGGL(we_aniso_grid_tables_kernel, dim3((units + 3) / 4 + 1), dim3(256), 0, st, cb_magnitudes, wavenumbers, ws, Z, N, K, d_cb ? 1 : 0, few);
    const size_t lds = (size_t)WG_ROWS * WG_OBS * 4;
#define WA_GO(G_, W_, S_) hipLaunchKernelGGL((we_aniso_grid_kernel<G_, W_, S_>), grid, dim3(W_ * 64), lds, st, (const char*)ws, cb_magnitudes, wavenumbers, out, d_cb, d_k, Z, N, K)
    if (d_cb) { if (few > 1) WA_GO(true, 16, true); else if (few) WA_GO(true, 16, false); else WA_GO(true, 8, false); }
    else      { if (few > 1) WA_GO(false, 16, true); else if (few) WA_GO(false, 16, false); else WA_GO(false, 8, false); }
#undef WA_GO
    const int rl = (int)hipGetLastError();
    if (rl) return rl;
    return proteus_we_aniso_direct(coordsA, coordsB, coords_layout, cb_magnitudes, wavenumbers, mask, out, d_cb, d_k, Z, N, K, 0,
                                   &reinterpret_cast<const WgParams*>(ws)->terms, stream);
}
