// The encoder's training step between its matrix products (fp32 tensors, gfx950): residual add + LayerNorm with what
// its backward needs, that backward, column sums (bias gradients), the laying-out of the attention's per-head weights for
// plain products and of their gradients back, and the gradient of a small embedding table.  (GELU and its derivative are
// epilogues of products, gemm_f32.hip.)
//
// All of it is streaming work of a few MB per call, so a call's time is its launch and one trip through memory; what
// these kernels remove is launches and trips.  A training step of 4 x 512 tokens (d_model 512, 3 layers) ran 178
// launches, 2.14 ms on the device; with these it ran 108, 1.69 ms on the device, and with a layer's launches issued by the library
// (encoder_layer.hip) it takes 1.54 ms in all.  At the kernels: device times of torch's kernels and of these at that size.
//
// Sums over tokens are taken in a fixed order (partial sums per workgroup, then one pass over them): the same bits on
// every call.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "proteus_hip.h"
#include "train_internal.h"

namespace {

constexpr int LN_WAVES  = 4;
constexpr int LN_MAX_D  = 2048;
using namespace proteus_train;
constexpr int EB_TOKENS = 128;          // tokens of an embedding-gradient workgroup
constexpr int EB_MAX_V  = 64;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// y = x + res, out = LayerNorm(y) * gamma + beta, stat[row] = (mean, 1 / sqrt(var + eps)).  A wave owns a row, CH chunks
// of 256 elements.  torch's add and layer_norm 4.4 + 5.6 us, this 5.8.
template <int CH>
__global__ __launch_bounds__(LN_WAVES * 64)
void add_layernorm_train_kernel(const float* __restrict__ x, const float* __restrict__ res, const float* __restrict__ gamma,
                                const float* __restrict__ beta, float* __restrict__ out, float* __restrict__ ysum,
                                float2* __restrict__ stat, const long rows, const int D, const float eps)
{
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * LN_WAVES + (threadIdx.x >> 6);
    if (row >= rows) return;                       // (whole waves leave: no barrier follows)
    const size_t base = (size_t)row * D;
    float4 y[CH];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e0 = (c * 64 + lane) * 4;
        y[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e0 < D) {
            const float4 a = *reinterpret_cast<const float4*>(x + base + e0);
            const float4 b = *reinterpret_cast<const float4*>(res + base + e0);
            y[c] = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
            *reinterpret_cast<float4*>(ysum + base + e0) = y[c];
            sum += (y[c].x + y[c].y) + (y[c].z + y[c].w);
        }
    }
    const float mean = wave_sum(sum) / (float)D;
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        if ((c * 64 + lane) * 4 < D) {
            const float4 t = make_float4(y[c].x - mean, y[c].y - mean, y[c].z - mean, y[c].w - mean);
            sq += (t.x * t.x + t.y * t.y) + (t.z * t.z + t.w * t.w);
        }
    }
    const float rstd = 1.0f / __builtin_sqrtf(wave_sum(sq) / (float)D + eps);
    if (lane == 0) stat[row] = make_float2(mean, rstd);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e0 = (c * 64 + lane) * 4;
        if (e0 < D) {
            const float4 g = *reinterpret_cast<const float4*>(gamma + e0);
            const float4 b = *reinterpret_cast<const float4*>(beta + e0);
            *reinterpret_cast<float4*>(out + base + e0) =
                make_float4(__builtin_fmaf((y[c].x - mean) * rstd, g.x, b.x), __builtin_fmaf((y[c].y - mean) * rstd, g.y, b.y),
                            __builtin_fmaf((y[c].z - mean) * rstd, g.z, b.z), __builtin_fmaf((y[c].w - mean) * rstd, g.w, b.w));
        }
    }
}

// dx = rstd (t - mean(t) - n mean(t n)) with t = dout gamma, n = (y - mean) rstd; part[workgroup] = its rows' share of
// (dgamma, dbeta) = (sum dout n, sum dout).  A wave takes every gridDim.x * LN_WAVES-th row and keeps its columns' sums in
// registers, so y and dout are read once for all three gradients (torch reads them twice: 8.2 + 5.7 + 3.9 us; this 6.9 + 3.0).
template <int CH>
__global__ __launch_bounds__(LN_WAVES * 64)
void layernorm_bwd_kernel(const float* __restrict__ dout, const float* __restrict__ ysum, const float2* __restrict__ stat,
                          const float* __restrict__ gamma, float* __restrict__ dx, float* __restrict__ part,
                          const long rows, const int D)
{
    __shared__ float red[2][CH * 256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float g[CH][4], ag[CH][4], ab[CH][4];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int e0 = (c * 64 + lane) * 4;
        const float4 t = e0 < D ? *reinterpret_cast<const float4*>(gamma + e0) : make_float4(0.f, 0.f, 0.f, 0.f);
        g[c][0] = t.x; g[c][1] = t.y; g[c][2] = t.z; g[c][3] = t.w;
#pragma unroll
        for (int e = 0; e < 4; ++e) ag[c][e] = ab[c][e] = 0.f;
    }
    const float inv = 1.0f / (float)D;
    for (long row = (long)blockIdx.x * LN_WAVES + wave; row < rows; row += (long)gridDim.x * LN_WAVES) {
        const size_t base = (size_t)row * D;
        const float2 st = stat[row];
        float t[CH][4], n[CH][4];
        float s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int e0 = (c * 64 + lane) * 4;
            if (e0 < D) {
                const float4 d4 = *reinterpret_cast<const float4*>(dout + base + e0);
                const float4 y4 = *reinterpret_cast<const float4*>(ysum + base + e0);
                const float d[4] = {d4.x, d4.y, d4.z, d4.w}, y[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    n[c][e] = (y[e] - st.x) * st.y;
                    t[c][e] = d[e] * g[c][e];
                    ag[c][e] = __builtin_fmaf(d[e], n[c][e], ag[c][e]);
                    ab[c][e] += d[e];
                    s1 += t[c][e];
                    s2 = __builtin_fmaf(t[c][e], n[c][e], s2);
                }
            }
        }
        s1 = wave_sum(s1) * inv;
        s2 = wave_sum(s2) * inv;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const int e0 = (c * 64 + lane) * 4;
            if (e0 < D) {
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = st.y * (t[c][e] - s1 - n[c][e] * s2);
                *reinterpret_cast<float4*>(dx + base + e0) = make_float4(o[0], o[1], o[2], o[3]);
            }
        }
    }
    for (int w = 0; w < LN_WAVES; ++w) {           // the waves add their sums up in turn
        if (wave == w) {
#pragma unroll
            for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int i = (c * 64 + lane) * 4 + e;
                    red[0][i] = w ? red[0][i] + ag[c][e] : ag[c][e];
                    red[1][i] = w ? red[1][i] + ab[c][e] : ab[c][e];
                }
        }
        __syncthreads();
    }
    float* p = part + (size_t)blockIdx.x * 2 * D;
    for (int i = threadIdx.x; i < D; i += LN_WAVES * 64) { p[i] = red[0][i]; p[D + i] = red[1][i]; }
}

// sums[slab][c] = sum over the slab's rows of a[row][c].
__global__ __launch_bounds__(CS_BLOCK)
void colsum_kernel(const float* __restrict__ a, float* __restrict__ sums, const long rows, const int C, const long slab_rows)
{
    __shared__ float red[CS_BLOCK / 64][CS_COLS];
    const long r0 = (long)blockIdx.y * slab_rows, r1 = r0 + slab_rows < rows ? r0 + slab_rows : rows;
    column_sums(a, sums + (size_t)blockIdx.y * C, r0, r1, C, blockIdx.x, red);
}

int colsum(const float* a, float* out, float* ws, long rows, int C, hipStream_t st) {
    const long slabs = (rows + CS_ROWS - 1) / CS_ROWS;
    const dim3 grid((unsigned)((C + CS_COLS - 1) / CS_COLS), (unsigned)slabs);
    hipLaunchKernelGGL(colsum_kernel, grid, dim3(CS_BLOCK), 0, st, a, slabs > 1 ? ws : out, rows, C, (long)CS_ROWS);
    if (slabs > 1)
        hipLaunchKernelGGL(colsum_kernel, dim3(grid.x), dim3(CS_BLOCK), 0, st, ws, out, slabs, C, slabs);
    return (int)hipGetLastError();
}

// Per-head projections [H][dm][dk] (three of them) <-> one matrix W [dm][3][H][dk]; output projection [dm][dk][H] <->
// Wo [dm][H][dk]; biases; sigma = min_spread + exp(w), with a copy of w.  torch: two cat, two copies, two elementwise launches forward;
// copies and additions of views backward (some 12).  One launch each way, 5 us.
struct HeadTensors {
    float *q_w, *k_w, *v_w, *q_b, *k_b, *v_b, *spread, *out_w;
};

template <bool BACK>
__global__ __launch_bounds__(256)
void heads_layout_kernel(const HeadTensors t, float* __restrict__ W, float* __restrict__ b, float* __restrict__ Wo,
                         float* __restrict__ sigma, const float* __restrict__ spread_w, const int dm, const int H, const int dk,
                         const float min_spread)
{
    const int row4 = 3 * H * dk / 4;                   // float4 of a row of W
    const long nW = (long)dm * row4, nO = (long)dm * dm, nB = 3 * H * dk;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < nW + nO + nB + H; i += (long)gridDim.x * 256) {
        if (i < nW) {
            const int m = (int)(i / row4), c = (int)(i % row4) * 4;
            const int p = c / (H * dk), h = (c / dk) % H, j = c % dk;
            float* src = p == 0 ? t.q_w : p == 1 ? t.k_w : t.v_w;
            if (!src) continue;                        // (backward: a projection that needs no gradient)
            float4* s = reinterpret_cast<float4*>(src + ((size_t)h * dm + m) * dk + j);
            float4* w = reinterpret_cast<float4*>(W + (size_t)m * 3 * H * dk + c);
            if (BACK) *s = *w; else *w = *s;
        } else if (i < nW + nO) {
            const long e = i - nW;
            const int o = (int)(e / dm), c = (int)(e % dm);
            float* w = Wo + e;
            if (t.out_w) {
                float* s = t.out_w + (size_t)o * dm + (c % dk) * H + c / dk;
                if (BACK) *s = *w; else *w = *s;
            }
        } else if (i < nW + nO + nB) {
            const int c = (int)(i - nW - nO), p = c / (H * dk), e = c % (H * dk);
            float* s = p == 0 ? t.q_b : p == 1 ? t.k_b : t.v_b;
            if (s) { if (BACK) s[e] = b[c]; else b[c] = s[e]; }
        } else {
            const int h = (int)(i - nW - nO - nB);
            if (!BACK) {
                const float w = spread_w[h];
                sigma[h] = min_spread + expf(w);
                if (t.spread) t.spread[h] = w;
            } else if (t.spread) t.spread[h] = sigma[h] * expf(spread_w[h]);        // sigma: its gradient
        }
    }
}

// part[slab][v][c] = sum over the slab's tokens with index v of dout[token][c].  A wave has a table of its own in LDS
// (its 64 columns, one per lane: no two lanes share a cell, so there are no atomics) and walks through its tokens in
// order.  torch: 106.8 us at 2048 tokens, 33 rows, 512 columns; this 8.2 and
// the sum over the slabs 3.
__global__ __launch_bounds__(256)
void embedding_bwd_kernel(const float* __restrict__ dout, const int64_t* __restrict__ tokens, float* __restrict__ part,
                          const long T, const int V, const int D)
{
    extern __shared__ float table[];                   // [4][V][64]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* tb = table + (size_t)wave * V * 64;
    for (int v = 0; v < V; ++v) tb[v * 64 + lane] = 0.f;
    const int col = blockIdx.x * 64 + lane;
    const bool in = col < D;
    const long t0 = (long)blockIdx.y * EB_TOKENS + wave * (EB_TOKENS / 4);
    const long t1 = t0 + EB_TOKENS / 4 < T ? t0 + EB_TOKENS / 4 : T;
    for (long t = t0; t < t1; t += 8) {
        float v[8];
        int64_t k[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool ok = t + u < t1;
            k[u] = ok ? tokens[t + u] : -1;
            v[u] = ok && in ? dout[(size_t)(t + u) * D + col] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k[u] >= 0 && k[u] < V) tb[(int)k[u] * 64 + lane] += v[u];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < V * 64; i += 256) {
        const int c = blockIdx.x * 64 + (i & 63);
        if (c < D) part[((size_t)blockIdx.y * V + (i >> 6)) * D + c] =
            (table[i] + table[V * 64 + i]) + (table[2 * V * 64 + i] + table[3 * V * 64 + i]);
    }
}

int ln_groups(long rows) { const long g = (rows + LN_WAVES - 1) / LN_WAVES; return (int)(g < 256 ? g : 256); }

bool misaligned(const void* p) { return ((uintptr_t)p & 15) != 0; }

}  // namespace

extern "C" size_t proteus_train_workspace_bytes(long rows, int C)
{
    if (rows <= 0 || C <= 0) return 0;
    const size_t slabs = (size_t)((rows + CS_ROWS - 1) / CS_ROWS);
    return (slabs > 1 ? slabs : 0) * (size_t)C * 4;
}

extern "C" size_t proteus_layernorm_bwd_workspace_bytes(long rows, int D)
{
    return rows <= 0 || D <= 0 ? 0 : (size_t)ln_groups(rows) * 2 * D * 4;
}

extern "C" size_t proteus_embedding_bwd_workspace_bytes(long T, int V, int D)
{
    if (T <= 0 || V <= 0 || D <= 0) return 0;
    const long slabs = (T + EB_TOKENS - 1) / EB_TOKENS;
    return (size_t)slabs * V * D * 4 + proteus_train_workspace_bytes(slabs, V * D);
}

extern "C" int proteus_add_layernorm_train_fwd(const float* x, const float* res, const float* gamma, const float* beta, float* out,
                                               float* ysum, float* stat, long rows, int D, float eps, void* stream)
{
    if (!x || !res || !gamma || !beta || !out || !ysum || !stat) return PROTEUS_ERR_NULL_POINTER;
    if (rows <= 0 || rows > ((1L << 31) - 1) * LN_WAVES || D <= 0 || D % 4 || D > LN_MAX_D || !(eps >= 0.0f)) return PROTEUS_ERR_BAD_SHAPE;
    if (misaligned(x) || misaligned(res) || misaligned(gamma) || misaligned(beta) || misaligned(out) || misaligned(ysum) || misaligned(stat))
        return PROTEUS_ERR_BAD_ALIGNMENT;
    const dim3 grid((unsigned)((rows + LN_WAVES - 1) / LN_WAVES)), block(LN_WAVES * 64);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define LN_GO(CH_) hipLaunchKernelGGL((add_layernorm_train_kernel<CH_>), grid, block, 0, st, x, res, gamma, beta, out, ysum, \
                                      (float2*)stat, rows, D, eps)
    switch ((D + 255) / 256) {
        case 1: LN_GO(1); break;
        case 2: LN_GO(2); break;
        case 3: case 4: LN_GO(4); break;
        default: LN_GO(8); break;
    }
#undef LN_GO
    return (int)hipGetLastError();
}

int proteus_train::layernorm_bwd_begin(const float* dout, const float* ysum, const float* stat, const float* gamma, float* dx, float* dgamma_dbeta, void* ws, size_t ws_bytes,
                                       long rows, int D, ColumnSums& sums, void* stream)
{
    if (!dout || !ysum || !stat || !gamma || !dx || !ws) return PROTEUS_ERR_NULL_POINTER;
    if (rows <= 0 || D <= 0 || D % 4 || D > LN_MAX_D || ws_bytes < proteus_layernorm_bwd_workspace_bytes(rows, D)) return PROTEUS_ERR_BAD_SHAPE;
    if (misaligned(dout) || misaligned(ysum) || misaligned(stat) || misaligned(gamma) || misaligned(dx) || misaligned(dgamma_dbeta) || misaligned(ws))
        return PROTEUS_ERR_BAD_ALIGNMENT;
    const int groups = ln_groups(rows);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define LN_GO(CH_) hipLaunchKernelGGL((layernorm_bwd_kernel<CH_>), dim3(groups), dim3(LN_WAVES * 64), 0, st, dout, ysum, \
                                      (const float2*)stat, gamma, dx, (float*)ws, rows, D)
    switch ((D + 255) / 256) {
        case 1: LN_GO(1); break;
        case 2: LN_GO(2); break;
        case 3: case 4: LN_GO(4); break;
        default: LN_GO(8); break;
    }
#undef LN_GO
    sums = {(const float*)ws, dgamma_dbeta, groups, 2 * D};      // (at most CS_ROWS groups)
    return (int)hipGetLastError();
}

extern "C" int proteus_layernorm_bwd(const float* dout, const float* ysum, const float* stat, const float* gamma, float* dx,
                                     float* dgamma_dbeta, void* ws, size_t ws_bytes, long rows, int D, void* stream)
{
    if (!dgamma_dbeta) return PROTEUS_ERR_NULL_POINTER;
    ColumnSums sums;
    const int rc = layernorm_bwd_begin(dout, ysum, stat, gamma, dx, dgamma_dbeta, ws, ws_bytes, rows, D, sums, stream);
    if (rc != PROTEUS_OK) return rc;
    return colsum(sums.a, sums.out, nullptr, sums.rows, sums.cols, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int proteus_colsum(const float* a, float* sums, void* ws, size_t ws_bytes, long rows, int C, void* stream)
{
    if (!a || !sums) return PROTEUS_ERR_NULL_POINTER;
    if (rows <= 0 || C <= 0 || C % 4 || rows > 65535L * CS_ROWS) return PROTEUS_ERR_BAD_SHAPE;
    const size_t need = proteus_train_workspace_bytes(rows, C);
    if (need && !ws) return PROTEUS_ERR_NULL_POINTER;
    if (ws_bytes < need) return PROTEUS_ERR_BAD_SHAPE;
    if (misaligned(a) || misaligned(sums) || misaligned(ws)) return PROTEUS_ERR_BAD_ALIGNMENT;
    return colsum(a, sums, (float*)ws, rows, C, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int proteus_heads_layout(float* const* tensors, float* W, float* b, float* Wo, float* sigma, const float* spread_w,
                                    int d_model, int H, int d_head, float min_spread, int backward, void* stream)
{
    if (!tensors || !W || !b || !Wo || !sigma || !spread_w) return PROTEUS_ERR_NULL_POINTER;
    if (d_model <= 0 || H <= 0 || d_head <= 0 || d_head % 4 || d_model != H * d_head || d_model > 16384) return PROTEUS_ERR_BAD_SHAPE;
    for (int i = 0; i < 8; ++i) {
        if (!backward && i != 6 && !tensors[i]) return PROTEUS_ERR_NULL_POINTER;
        if (i < 3 && misaligned(tensors[i])) return PROTEUS_ERR_BAD_ALIGNMENT;
    }
    if (misaligned(W)) return PROTEUS_ERR_BAD_ALIGNMENT;
    const HeadTensors t = {tensors[0], tensors[1], tensors[2], tensors[3], tensors[4], tensors[5], tensors[6], tensors[7]};
    const long n = (long)d_model * (3 * H * d_head / 4) + (long)d_model * d_model + 3 * H * d_head + H;
    const dim3 grid((unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096));
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (backward) hipLaunchKernelGGL((heads_layout_kernel<true>), grid, dim3(256), 0, st, t, W, b, Wo, sigma, spread_w, d_model, H, d_head, min_spread);
    else          hipLaunchKernelGGL((heads_layout_kernel<false>), grid, dim3(256), 0, st, t, W, b, Wo, sigma, spread_w, d_model, H, d_head, min_spread);
    return (int)hipGetLastError();
}

extern "C" int proteus_embedding_bwd(const float* dout, const int64_t* tokens, float* dW, void* ws, size_t ws_bytes, long T, int V, int D, void* stream)
{
    if (!dout || !tokens || !dW || !ws) return PROTEUS_ERR_NULL_POINTER;
    if (T <= 0 || V <= 0 || V > EB_MAX_V || D <= 0 || D % 4 || D > 16384 || T > 65535L * EB_TOKENS) return PROTEUS_ERR_BAD_SHAPE;
    if (ws_bytes < proteus_embedding_bwd_workspace_bytes(T, V, D)) return PROTEUS_ERR_BAD_SHAPE;
    if (misaligned(dout) || ((uintptr_t)tokens & 7) || misaligned(dW) || misaligned(ws)) return PROTEUS_ERR_BAD_ALIGNMENT;
    const long slabs = (T + EB_TOKENS - 1) / EB_TOKENS;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    float* part = (float*)ws;
    hipLaunchKernelGGL(embedding_bwd_kernel, dim3((unsigned)((D + 63) / 64), (unsigned)slabs), dim3(256), (size_t)4 * V * 64 * 4, st,
                       dout, tokens, part, T, V, D);
    return colsum(part, dW, part + (size_t)slabs * V * D, slabs, V * D, st);
}
