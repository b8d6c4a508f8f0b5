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
//     single-precision phase at tens of revolutions.  1/phihat is an even polynomial in theta (kQ).
//   - F0 = -i dF1/dk comes from the same grid: two more products against node position x grid.
//   - Everything is summed in 32-bit integers (fixed point): LDS float atomics take 193 clocks per wave instruction on this
//     machine, integer ones 4.7 (conflict-free) to 6.2 (random cells); integer sums do not depend on their order, so
//     the waves of a workgroup share the grids and the result is the same from run to run.  A cell's octave e = floor(log2 n)
//     sets its scale: what is added is phi 2^e h / r < 2, so near and far sources keep the same relative precision (the
//     rounding of one addition is 2^-22 of the largest term); octaves have their own rows where they overlap.  After
//     1024 sources (what 32 bits hold at that scale) the integers are moved on to float accumulators.
//   - Pairs closer than h/2 (never the case for real structures) are summed directly, as are all pairs of a workgroup
//     whose distances would need too many windows of the grid or are not finite.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "proteus_hip.h"

namespace {

constexpr int WG_OBS     = 16;                    // observers per workgroup (one tile of the 16x16x4 product)
constexpr int WG_FLUSH   = 2048;                  // sources between two flushes
constexpr int WG_ROWS    = 1216;                  // rows of 16 cells in LDS: 77 824 bytes, two workgroups of 8 waves per compute unit
constexpr int WG_R0      = 8;                     // rows in front of the first node (zeros, read by the product)
constexpr int WG_OCT     = 8;                     // extra rows per octave: six nodes reach five rows into the next one (8: a shift in the address)
constexpr int WG_TRASH   = WG_ROWS - 6;           // the rows of sources that belong to no cell
constexpr int WG_CELLS   = WG_TRASH - WG_R0 - 5 - WG_OCT * 10;     // cells per window (n < 2^11)
constexpr int WG_MAX_WINDOWS = 16;
constexpr int WG_GROUPS  = (WG_CELLS + 5 + 1) / 2 / 8 + 1;         // groups of 8 rows of the tables

constexpr float WG_OVERSAMPLING = 3.5f;
constexpr float WG_UNIT  = 4096.0f;               // coordinates are scaled by this power of two (see the spread)
constexpr float WG_MAGIC = 12582912.0f;           // 1.5 x 2^23: t + WG_MAGIC holds rint(t) in its low bits
constexpr uint32_t WG_MAGIC_BITS = 0x4B400000u;

static_assert(WG_R0 + WG_CELLS - 1 + WG_OCT * 10 + 6 <= WG_TRASH, "rows of the spread");
static_assert(WG_R0 + 8 * WG_GROUPS * 2 + 8 <= WG_ROWS, "rows of the product");

struct WgParams {                 // head of the workspace, written by the preparation
    float inv_h, h;
    int   pad[62];
};
struct WgWave { double rev; float q, dq; };      // k h / 2 pi; 1/phihat and its derivative at theta = k h

// even polynomial 1/phihat(theta), relative error 3e-10 for |theta| <= pi/3.5
__device__ const double kQ[8] = {0.5144796916399992, 0.1467794687271181, 0.022356478641989086, 0.0024221529567290006,
                                 0.00020978467048036778, 1.54869506429115e-05, 9.95433626001851e-07, 7.199788952850109e-08};

struct WgBox { float lo[3], hi[3], bad, pad; };  // of 64 tokens, unpadded ones only; bad: one of them is not finite

struct WgLayout { size_t counts, waves, table, boxes, sources, bytes; int npad, nkt, nbox; };

__host__ __device__ inline WgLayout wg_layout(int Z, int N, int K)
{
    WgLayout l;
    l.nkt  = (K + 15) / 16;
    l.npad = (N + 63) / 64 * 64 + 512;            // the stream reads up to an iteration (256 sources) past the end
    l.nbox = (N + 63) / 64;
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    l.counts  = sizeof(WgParams);
    l.waves   = l.counts + up((size_t)Z * 4);
    l.table   = l.waves + up((size_t)l.nkt * 16 * sizeof(WgWave));
    l.boxes   = l.table + (size_t)WG_GROUPS * l.nkt * 64 * 16;
    l.sources = l.boxes + up((size_t)Z * l.nbox * sizeof(WgBox));
    l.bytes   = l.sources + up((size_t)Z * l.npad * 16);
    return l;
}

// ---------------------------------------------------------------------------------------------------------------
// Preparation: blocks [0, Z * ceil(npad / 256)) compact the tokens of the batch items (unpadded ones first, with their
// token index; padded and surplus slots get coordinates at infinity, which no cell takes), the others fill the tables.

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

__global__ __launch_bounds__(256)
void we_grid_prepare_kernel(const float* __restrict__ coords, const int layout, const float* __restrict__ wavenumbers,
                            const uint8_t* __restrict__ mask, char* __restrict__ ws, const int Z, const int N, const int K)
{
    const WgLayout L = wg_layout(Z, N, K);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per_item = (L.npad + 255) / 256;
    __shared__ int   s_cnt[3][4];
    __shared__ float s_max[4];

    if ((int)blockIdx.x < Z * per_item) {
        const int z = blockIdx.x / per_item, b = blockIdx.x % per_item;
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
        if (in) {
            src[valid ? before : n + (j - before)] = v;
        } else if (j < L.npad) {
            src[j] = v;
        }
        return;
    }

    // ---- tables ----
    float km = 0.f;
    bool bad = false;
    for (int k = tid; k < K; k += 256) { const float w = fabsf(wavenumbers[k]); bad |= !(w < 3.0e38f); km = fmaxf(km, w); }
    for (int o = 32; o > 0; o >>= 1) km = fmaxf(km, __shfl_xor(km, o));
    bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 0) s_max[wave] = bad ? __builtin_inff() : km;
    __syncthreads();
    km = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    // cells per unit of length, rounded to float once: h is its exact inverse from here on (a wavenumber beyond any use
    // gives an infinite value, which sends every workgroup to the direct sums)
    const float inv_h = fmaxf(km * (WG_OVERSAMPLING / 3.14159265f) * 1.000001f, 1.0e-6f);
    const double h = 1.0 / (double)inv_h;
    const int unit = ((int)blockIdx.x - Z * per_item) * 4 + wave;
    if (unit == 0 && lane == 0) { WgParams* p = reinterpret_cast<WgParams*>(ws); p->inv_h = inv_h; p->h = (float)h; }
    if (unit >= WG_GROUPS * L.nkt) return;
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
        for (int i = 7; i >= 0; --i) q = q * t2 + kQ[i];
#pragma unroll
        for (int i = 7; i >= 1; --i) dq = dq * t2 + 2 * i * kQ[i];
        WgWave w; w.rev = rev; w.q = (float)q; w.dq = (float)(dq * th);
        reinterpret_cast<WgWave*>(ws + L.waves)[k] = w;
    }
}

// ---------------------------------------------------------------------------------------------------------------

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

// The sources of `near` pairs of one observer (all of them if `all`), summed directly by one wave, a lane per wavenumber.
template <bool SUMS>
__device__ void wg_direct(const float4* __restrict__ src, const int n, const float xi, const float yi, const float zi, const float inv_h, const bool all,
                          const float* __restrict__ wavenumbers, float* __restrict__ o, float* __restrict__ pc, float* __restrict__ ps, const int K, const int lane)
{
    for (int kb = 0; kb < K; kb += 256) {
        float kr[4], oc[4], os[4], c[4], s[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = kb + 64 * u + lane;
            kr[u] = (float)((k < K ? (double)wavenumbers[k] : 0.0) * 0.15915494309189533577) * (1.0f / WG_UNIT);
            oc[u] = os[u] = c[u] = s[u] = 0.f;
        }
        for (int j0 = 0; j0 < n; j0 += 64) {
            const float4 q = src[j0 + lane];
            float r2, inv, r;
            wg_distance(xi - q.x, yi - q.y, zi - q.z, r2, inv, r);
            const bool near = __builtin_bit_cast(int, __builtin_fmaf(r, inv_h, WG_MAGIC)) == __builtin_bit_cast(int, WG_MAGIC);
            uint64_t todo = __builtin_amdgcn_ballot_w64(j0 + lane < n && r2 != 0.0f && (all || near));
            while (todo) {
                const int b = __builtin_ctzll(todo);
                todo &= todo - 1;
                const float rb = wg_lane(r, b), mb = wg_lane(inv, b);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float ph = __builtin_amdgcn_fractf(rb * kr[u]);
                    const float cs = __builtin_amdgcn_cosf(ph), sn = __builtin_amdgcn_sinf(ph);
                    oc[u] = __builtin_fmaf(cs, mb, oc[u]);
                    os[u] = __builtin_fmaf(sn, mb, os[u]);
                    if (SUMS) { c[u] += cs; s[u] += sn; }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = kb + 64 * u + lane;
            if (k >= K) continue;
            oc[u] *= WG_UNIT; os[u] *= WG_UNIT;
            if (!all) { oc[u] += o[2 * k]; os[u] += o[2 * k + 1]; }
            o[2 * k] = oc[u]; o[2 * k + 1] = os[u];
            if (SUMS) {
                if (!all) { c[u] += pc[k]; s[u] += ps[k]; }
                pc[k] = c[u]; ps[k] = s[u];
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
    constexpr int KT      = 16 / WAVES;           // tiles of 16 wavenumbers a wave takes at a time
    constexpr int AHEAD   = WAVES == 16 ? 4 : 2;  // groups of the tables in flight: a lone workgroup has nothing else to cover their latency
    extern __shared__ __align__(16) uint32_t s_grid[];          // [WG_ROWS][WG_OBS]
    __shared__ float s_red[WAVES];
    __shared__ int   s_near[WG_OBS];
    __shared__ int   s_tok[WG_OBS];

    const WgLayout L = wg_layout(Z, N, K);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z = blockIdx.y;
    const size_t zN = (size_t)z * N;
    const int n = reinterpret_cast<const int*>(ws + L.counts)[z];
    const float4* __restrict__ src = reinterpret_cast<const float4*>(ws + L.sources) + (size_t)z * L.npad;
    const WgWave* __restrict__ waves = reinterpret_cast<const WgWave*>(ws + L.waves);
    const float4* __restrict__ table = reinterpret_cast<const float4*>(ws + L.table);
    const float inv_h = reinterpret_cast<const WgParams*>(ws)->inv_h * (1.0f / WG_UNIT), h = reinterpret_cast<const WgParams*>(ws)->h;

    // ---- the workgroup's slots: unpadded observers first, then padded tokens (zero rows), then nothing ----
    const int slot0 = blockIdx.x * WG_OBS;
    const int obs   = lane & 15;
    const float4 me = src[slot0 + obs];
    const bool ok   = slot0 + obs < n;
    if (tid < WG_OBS) { s_tok[tid] = slot0 + tid < N ? __builtin_bit_cast(int, me.w) : -1; s_near[tid] = 0; }
    if (slot0 >= n) {
        // padded tokens only
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

    // ---- how far away can a source be?  Farthest source from the middle of the observers + their own radius ----
    bool direct;
    int  ncell;
    {
        float lo[3] = {3.0e38f, 3.0e38f, 3.0e38f}, hi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
        if (ok) { lo[0] = hi[0] = me.x; lo[1] = hi[1] = me.y; lo[2] = hi[2] = me.z; }
#pragma unroll
        for (int c = 0; c < 3; ++c)
            for (int o = 8; o > 0; o >>= 1) { lo[c] = fminf(lo[c], __shfl_xor(lo[c], o)); hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], o)); }
        const float mx = 0.5f * (lo[0] + hi[0]), my = 0.5f * (lo[1] + hi[1]), mz = 0.5f * (lo[2] + hi[2]);
        const float ex = hi[0] - mx, ey = hi[1] - my, ez = hi[2] - mz;
        // the corners of the boxes around every 64 tokens bound the distances (a thread has one box up to N = 64 THREADS)
        const WgBox* __restrict__ boxes = reinterpret_cast<const WgBox*>(ws + L.boxes) + (size_t)z * L.nbox;
        float far2 = 0.f;
        for (int b = tid; b < L.nbox; b += THREADS) {
            const WgBox q = boxes[b];
            const float dx = fmaxf(q.hi[0] - mx, mx - q.lo[0]), dy = fmaxf(q.hi[1] - my, my - q.lo[1]), dz = fmaxf(q.hi[2] - mz, mz - q.lo[2]);
            const float d2 = dx * dx + dy * dy + dz * dz + q.bad;
            if (q.lo[0] <= q.hi[0] || q.bad != 0.f) far2 = d2 < 3.0e38f ? fmaxf(far2, d2) : __builtin_inff();       // (NaN counts as infinity and stays)
        }
        for (int o = 32; o > 0; o >>= 1) far2 = fmaxf(far2, __shfl_xor(far2, o));
        if (lane == 0) s_red[wave] = far2;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) far2 = fmaxf(far2, s_red[w]);
        const float reach = (__builtin_sqrtf(far2) + __builtin_sqrtf(ex * ex + ey * ey + ez * ez)) * 1.00001f;
        const float cells = reach * inv_h + 2.0f;
        direct = !(cells < (float)(WG_CELLS * WG_MAX_WINDOWS));
        ncell  = direct ? 0 : (int)cells;
        ncell  = __builtin_amdgcn_readfirstlane(ncell);
        direct = __builtin_amdgcn_readfirstlane(direct ? 1 : 0) != 0;
    }

    if (!direct) {
        // ---- the spreading kernel's coefficients, in fixed point ----
        // A weight is made as a single-precision denormal: its bit pattern is the rounded integer, and no conversion is needed
        // (4.7 clocks each).  Of the 2^-149 that takes 2^-12 comes with 1/r (WG_UNIT) and the rest with the coefficients, so that
        // every factor is a normal number.  One unit is `scale` of a full weight: 2 scale (the largest weight) times the
        // sources between two flushes stays below 2^32.
        const int nit = (n + STEP - 1) / STEP, quarter = nit * (STEP / 4);
        const bool flushes = nit * STEP > WG_FLUSH;
        const float scale = flushes ? 1048000.0f : fminf(4190000.0f, 2147000000.0f / (float)(nit * STEP));
        const float fix = scale * h * 0x1p-137f;
        const float e00 = wg_vgpr(fix * 0.8198235f),    e01 = wg_vgpr(fix * -0.41093102f), e02 = wg_vgpr(fix * 0.08094943f);
        const float o00 = wg_vgpr(fix * 0.65685374f),   o01 = wg_vgpr(fix * -0.43981674f), o02 = wg_vgpr(fix * 0.14080364f);
        const float e10 = wg_vgpr(fix * 0.15015647f),   e11 = wg_vgpr(fix * 0.37342498f),  e12 = wg_vgpr(fix * -0.1214422f);
        const float o10 = wg_vgpr(fix * 0.40670425f),   o11 = wg_vgpr(fix * 0.057586372f), o12 = wg_vgpr(fix * -0.069855906f);
        const float e20 = wg_vgpr(fix * 0.0018756188f), e21 = wg_vgpr(fix * 0.037506126f), e22 = wg_vgpr(fix * 0.04049774f);
        const float o20 = wg_vgpr(fix * 0.013345578f),  o21 = wg_vgpr(fix * 0.05343353f),  o22 = wg_vgpr(fix * 0.01371953f);
        const float magic = wg_vgpr(WG_MAGIC), inv_hv = wg_vgpr(inv_h);
        uint32_t emask = 0xff800000u;
        asm volatile("" : "+v"(emask));

        float lowest = 3.0e38f;                    // smallest n of any source, as magic + n

        for (int n_lo = 1; n_lo <= ncell; n_lo += WG_CELLS) {
            const int cells = min(WG_CELLS, ncell + 1 - n_lo);           // source cells n_lo .. n_lo + cells - 1
            const int e_lo  = 31 - __builtin_clz(n_lo);
            const int e_hi  = 31 - __builtin_clz(n_lo + cells - 1);
            const int used  = WG_R0 + cells + 5 + WG_OCT * (e_hi - e_lo);      // rows that hold anything
            wg_f4 facc[CHUNKS];
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) facc[i] = wg_f4{0.f, 0.f, 0.f, 0.f};

            uint4* g4 = reinterpret_cast<uint4*>(s_grid);
            auto me_again = [&]() { int v = tid; asm volatile("" : "+v"(v)); return v; };     // (keeps the addresses of these passes out of registers between them)
            __syncthreads();                                             // the previous window's product is done
            for (int i = tid; i < used * (WG_OBS / 4); i += THREADS) g4[i] = make_uint4(0, 0, 0, 0);
            __syncthreads();

            // LDS address of a source's first node: row (n - n_lo) + 8 (e - e_lo), with n and e taken from float bits.  Sources
            // that belong to no cell of this window go to the trash rows: with one window those are the observer itself and slots
            // past the end (n is NaN) and pairs closer than h / 2 (n = 0, whose exponent takes the address below zero), all of
            // which one unsigned minimum catches.
            uint32_t base = (uint32_t)(uintptr_t)(wg_lds_u32*)s_grid + (uint32_t)((WG_R0 - n_lo - WG_OCT * e_lo) * WG_OBS + obs) * 4u
                            - (WG_MAGIC_BITS << 6) - 127u * (WG_OCT * WG_OBS * 4u);
            uint32_t trash = (uint32_t)(uintptr_t)(wg_lds_u32*)s_grid + (uint32_t)(WG_TRASH * WG_OBS + obs) * 4u;
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
                const float x2 = x * x, xc = x * c;
                const float E0 = __builtin_fmaf(__builtin_fmaf(e02, x2, e01), x2, e00), O0 = __builtin_fmaf(__builtin_fmaf(o02, x2, o01), x2, o00);
                const float E1 = __builtin_fmaf(__builtin_fmaf(e12, x2, e11), x2, e10), O1 = __builtin_fmaf(__builtin_fmaf(o12, x2, o11), x2, o10);
                const float E2 = __builtin_fmaf(__builtin_fmaf(e22, x2, e21), x2, e20), O2 = __builtin_fmaf(__builtin_fmaf(o22, x2, o21), x2, o20);
                const float t0 = E0 * c, t1 = E1 * c, t2 = E2 * c;
                uint32_t at = (ub << 6) + base + (eb >> 14);
                if (decltype(multi)::value) at = ub - first < (uint32_t)cells ? at : trash;
                else                        at = min(at, trash);
                wg_lds_u32* a = (wg_lds_u32*)(uintptr_t)at;
                auto add = [&](const int l, const float w) {
                    __hip_atomic_fetch_add(a + l * WG_OBS, __builtin_bit_cast(uint32_t, w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                };
                add(0, __builtin_fmaf(-O2, xc, t2));
                add(1, __builtin_fmaf(-O1, xc, t1));
                add(2, __builtin_fmaf(-O0, xc, t0));
                add(3, __builtin_fmaf(O0, xc, t0));
                add(4, __builtin_fmaf(O1, xc, t1));
                add(5, __builtin_fmaf(O2, xc, t2));
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
                if (ncell > WG_CELLS) stream(wg_true{}); else stream(wg_false{});
                if (!flushes) break;
                __syncthreads();
                const int tf = me_again();
#pragma unroll
                for (int i = 0; i < CHUNKS; ++i) {
                    const int q = tf + i * THREADS;
                    if (q < used * (WG_OBS / 4)) {
                        const uint4 v = g4[q];
                        facc[i] += wg_f4{(float)v.x, (float)v.y, (float)v.z, (float)v.w};
                        if (it < nit) g4[q] = make_uint4(0, 0, 0, 0);
                        else reinterpret_cast<wg_f4*>(s_grid)[q] = facc[i];
                    }
                }
                __syncthreads();
                if (it >= nit) break;
                until = min(it + WG_FLUSH / STEP, nit);
            }
            if (!flushes) __syncthreads();

            // ---- bring the octaves together: node v = n_lo - 3 + p to row WG_R0 + p, zeros behind the last ----
            const int nodes = cells + 5;
            const int tc = me_again();
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) {
                const int q = tc + i * THREADS;
                const int pn = (q >> 2) - WG_R0;
                wg_f4 v = {0.f, 0.f, 0.f, 0.f};
                if (pn >= 0 && pn < nodes) {
                    const int na = max(pn - 5, 0) + n_lo, nz = min(pn, cells - 1) + n_lo;       // sources that reach this node
                    const int ea = 31 - __builtin_clz(na), ez = 31 - __builtin_clz(nz);
                    for (int e = ea; e <= ez; ++e) {
                        const int at = q + WG_OCT * (e - e_lo) * (WG_OBS / 4);
                        const float sc = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23);
                        wg_f4 w;
                        if (flushes) w = reinterpret_cast<const wg_f4*>(s_grid)[at];
                        else { const uint4 b = g4[at]; w = wg_f4{(float)b.x, (float)b.y, (float)b.z, (float)b.w}; }
                        v += w * sc;
                    }
                }
                facc[i] = v;
            }
            __syncthreads();
            const int tw = me_again();
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) {
                const int q = tw + i * THREADS;
                if (q < (WG_R0 + nodes + 8) * (WG_OBS / 4)) reinterpret_cast<wg_f4*>(s_grid)[q] = facc[i];
            }
            __syncthreads();

            // ---- the grid at the wavenumbers: rows j = 0 .. on both sides of the middle ----
            // A wave's tiles share the grid values; the tables come from L2, AHEAD groups of rows ahead.
            const float* g = reinterpret_cast<const float*>(s_grid);
            const int mid    = (nodes + 1) / 2;
            const int groups = (mid + 7) / 8;
            const int vc     = n_lo - 3 + mid;                              // the middle lies at vc h
            const int mm     = lane >> 4;
            const float* gp  = g + (WG_R0 + mid + mm) * WG_OBS + obs;
            const float* gm  = g + (WG_R0 + mid - 1 - mm) * WG_OBS + obs;
            for (int kp = KT * wave; kp < L.nkt; kp += KT * WAVES) {
                wg_f4 ec[KT], os[KT], oc[KT], es[KT];
#pragma unroll
                for (int t = 0; t < KT; ++t) ec[t] = os[t] = oc[t] = es[t] = wg_f4{0.f, 0.f, 0.f, 0.f};
                const float4* tb = table + (size_t)kp * 64 + lane;
                const size_t  ts = (size_t)L.nkt * 64;
                const int     k2 = kp + 1 < L.nkt ? 64 : 0;                 // (an odd number of tiles: the last one twice, written once)
                float4 b[AHEAD][KT];
                auto fetch = [&](const int gr, float4 (&bb)[KT]) {
                    const float4* at = tb + (size_t)min(gr, WG_GROUPS - 1) * ts;
#pragma unroll
                    for (int t = 0; t < KT; ++t) bb[t] = at[t * k2];
                };
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) fetch(i, b[i]);
                float y = (float)mm + 0.5f;
                for (int g0 = 0; g0 < groups; g0 += AHEAD) {
#pragma unroll
                    for (int i = 0; i < AHEAD; ++i) {
                        const int gr = g0 + i;
                        if (gr >= groups) break;
#pragma unroll
                        for (int s = 0; s < 2; ++s) {
                            const int off = (8 * gr + 4 * s) * WG_OBS;
                            const float a = gp[off], m = gm[-off];
                            const float E = a + m, O = a - m;
                            const float Oy = O * y, Ey = E * y;
#pragma unroll
                            for (int t = 0; t < KT; ++t) {
                                const float bc = s ? b[i][t].z : b[i][t].x, bs = s ? b[i][t].w : b[i][t].y;
                                ec[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(E, bc, ec[t], 0, 0, 0);
                                os[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(O, bs, os[t], 0, 0, 0);
                                if (SUMS) {
                                    oc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(Oy, bc, oc[t], 0, 0, 0);
                                    es[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ey, bs, es[t], 0, 0, 0);
                                }
                            }
                            y += 4.0f;
                        }
                        fetch(gr + AHEAD, b[i]);
                    }
                }
#pragma unroll
                for (int t = 0; t < KT; ++t) {
                    const int k = (kp + t) * 16 + obs;
                    if (k >= K) continue;
                    const WgWave w = waves[k];
                    const double ph = w.rev * (double)vc;
                    const float f  = (float)(ph - __builtin_floor(ph));
                    const float rc = __builtin_amdgcn_cosf(f), rs = __builtin_amdgcn_sinf(f);
                    const float q1 = w.q / (scale * h), q0s = w.q / scale, dq = w.dq / scale;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int  tok  = s_tok[mm * 4 + i];
                        if (tok < 0) continue;
                        const bool keep = slot0 + mm * 4 + i < n;
                        const size_t row = zN + tok;
                        float2 v = make_float2(q1 * (ec[t][i] * rc - os[t][i] * rs), q1 * (ec[t][i] * rs + os[t][i] * rc));
                        float2* po = reinterpret_cast<float2*>(out + row * 2 * K) + k;
                        if (n_lo > 1) { const float2 o = *po; v.x += o.x; v.y += o.y; }
                        *po = keep ? v : make_float2(0.f, 0.f);
                        if (SUMS) {
                            // F0 = rot [ q h (vc G + Gy) - i q' h G ] with G = ec + i os, Gy = oc + i es
                            const float gr_ = q0s * ((float)vc * ec[t][i] + oc[t][i]) + dq * os[t][i];
                            const float gi_ = q0s * ((float)vc * os[t][i] + es[t][i]) - dq * ec[t][i];
                            float c0 = gr_ * rc - gi_ * rs, s0 = gr_ * rs + gi_ * rc;
                            float* pc = cos_sums + row * K + k;
                            float* ps = sin_sums + row * K + k;
                            if (n_lo > 1) { c0 += *pc; s0 += *ps; }
                            *pc = keep ? c0 : 0.f;
                            *ps = keep ? s0 : 0.f;
                        }
                    }
                }
            }
        }
        if (lowest == WG_MAGIC && ok) s_near[obs] = 1;
    }

    // ---- pairs closer than h / 2, and everything where the grid is of no use ----
    __syncthreads();
    for (int q = wave; q < WG_OBS; q += WAVES) {
        const int t = s_tok[q];
        if (t < 0) continue;
        const size_t row = zN + t;
        float* o  = out + row * 2 * K;
        float* pc = SUMS ? cos_sums + row * K : nullptr;
        float* ps = SUMS ? sin_sums + row * K : nullptr;
        if (slot0 + q >= n) {
            if (direct) {
                for (int k = lane; k < 2 * K; k += 64) o[k] = 0.f;
                if (SUMS) for (int k = lane; k < K; k += 64) { pc[k] = 0.f; ps[k] = 0.f; }
            }
            continue;
        }
        if (!direct && !s_near[q]) continue;
        wg_direct<SUMS>(src, n, wg_lane(me.x, q), wg_lane(me.y, q), wg_lane(me.z, q), inv_h, direct, wavenumbers, o, pc, ps, K, lane);
    }
}

}  // namespace

// The grid pays from about 6e7 (pair, wavenumber) units on, below which two launches and the latency of one workgroup's
// phases are what a call costs (measured, grid against direct kernel: 1 x 512 and K = 256 27 / 26 us, 16 x 128 and K = 256
// 20 / 23 us, 1 x 128 17.6 / 8.2 us, 1 x 256 and K = 64 14.7 / 11.4 us, 32 x 64 and K = 64 12.2 / 7.9 us), and from 64 wavenumbers on.
static bool we_grid_wanted(int Z, int N, int K, int tuning)
{
    return tuning == 0 && K >= 64 && (double)Z * N * N * K >= 6.0e7;
}

extern "C" size_t proteus_we_fwd_workspace_bytes(int Z, int N, int K, int tuning)
{
    if (Z <= 0 || N <= 0 || K <= 0 || N > PROTEUS_WE_MAX_N || K > PROTEUS_WE_MAX_K || Z > 65535) return 0;
    return we_grid_wanted(Z, N, K, tuning) ? wg_layout(Z, N, K).bytes : 0;
}

extern "C" int proteus_we_fwd_ws(const float* coords, int coords_layout,
                                 const float* wavenumbers, const uint8_t* mask,
                                 float* out, float* cos_sums, float* sin_sums, void* workspace, size_t workspace_bytes,
                                 int Z, int N, int K, int tuning, void* stream)
{
    const int rc = proteus_we_fwd_check(coords, coords_layout, wavenumbers, mask, out, cos_sums, sin_sums, Z, N, K, tuning);
    if (rc != PROTEUS_OK) return rc;
    if (!workspace || tuning != 0 || workspace_bytes < wg_layout(Z, N, K).bytes)
        return proteus_we_fwd(coords, coords_layout, wavenumbers, mask, out, cos_sums, sin_sums, Z, N, K, tuning, stream);
    if ((uintptr_t)workspace & 255) return PROTEUS_ERR_BAD_ALIGNMENT;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const WgLayout L = wg_layout(Z, N, K);
    const unsigned prep = (unsigned)Z * (unsigned)((L.npad + 255) / 256) + (unsigned)((WG_GROUPS * L.nkt + 3) / 4);
    hipLaunchKernelGGL(we_grid_prepare_kernel, dim3(prep), dim3(256), 0, st, coords, coords_layout, wavenumbers, mask, (char*)workspace, Z, N, K);
    const dim3 grid((N + WG_OBS - 1) / WG_OBS, Z);
    const size_t lds = (size_t)WG_ROWS * WG_OBS * 4;
    const bool few = (long)grid.x * Z <= 256;
#define WG_GO(S_, W_) hipLaunchKernelGGL((we_grid_kernel<S_, W_>), grid, dim3(W_ * 64), lds, st, (const char*)workspace, wavenumbers, out, cos_sums, sin_sums, Z, N, K)
    if (cos_sums) { if (few) WG_GO(true, 16); else WG_GO(true, 8); }
    else          { if (few) WG_GO(false, 16); else WG_GO(false, 8); }
#undef WG_GO
    return (int)hipGetLastError();
}
