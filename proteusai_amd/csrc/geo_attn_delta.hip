// D = rowsum(O * dO) for the attention backward, gfx950.
//
// The reference's backward wrapper takes it with torch before its kernel runs (old/old_scripts/attn/geometric_attn.py:618:
// `D = torch.sum(O*dO, dim=3)`); the backward kernels subtract it from dP.  Here: one pass over O (fp32) and dO (fp32,
// bf16 or fp16, as autograd hands it over), products and sum in fp32, D [Z,H,N] fp32.  HBM-bound streaming work:
// (4 + sizeof(dO element)) bytes per element read, 4 bytes per row written.  d / 4 lanes share a row, every lane
// loads 4 consecutive elements of both tensors (16 / 8 bytes), the lanes of a row meet by shuffles.
//
// The backward also needs dO in the operands' 16-bit type and its per-head sums cleared.  Both are done here on request
// (proteus_geo_attn_prepare_bwd): dO is in registers anyway, so its cast costs the 2 bytes that are written instead of a
// launch that reads 4 and writes 2.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "proteus_hip.h"
#include "geo_attn_ops.h"

namespace {

constexpr int GD_THREADS = 256;

struct GdStrides { long o[3], g[3], c[3]; };      // (batch, head, token) element strides of O, dO and the cast of dO
struct GdExtra { uint16_t* cast; float* zero_a; float* zero_b; };      // any of them may be NULL

template <int DTYPE> struct Grad;
template <> struct Grad<PROTEUS_DTYPE_F32> {
    typedef float T;
    static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
        const float4 t = *reinterpret_cast<const float4*>(p);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    }
};
template <> struct Grad<PROTEUS_DTYPE_BF16> {
    typedef uint16_t T;
    static __device__ __forceinline__ void load(const uint16_t* p, float (&v)[4]) {
        const uint2 t = *reinterpret_cast<const uint2*>(p);
        v[0] = __builtin_bit_cast(float, t.x << 16); v[1] = __builtin_bit_cast(float, t.x & 0xffff0000u);
        v[2] = __builtin_bit_cast(float, t.y << 16); v[3] = __builtin_bit_cast(float, t.y & 0xffff0000u);
    }
};
template <> struct Grad<PROTEUS_DTYPE_F16> {
    typedef uint16_t T;
    static __device__ __forceinline__ void load(const uint16_t* p, float (&v)[4]) {
        typedef _Float16 half2v __attribute__((ext_vector_type(2)));
        const uint2 t = *reinterpret_cast<const uint2*>(p);
        const half2v a = __builtin_bit_cast(half2v, t.x), b = __builtin_bit_cast(half2v, t.y);
        v[0] = (float)a[0]; v[1] = (float)a[1]; v[2] = (float)b[0]; v[3] = (float)b[1];
    }
};

// LPR = d / 4 lanes per row (8, 16, 32); F16: the cast is to fp16, otherwise to bf16
template <int DTYPE, int LPR, bool F16>
__global__ __launch_bounds__(GD_THREADS)
void geo_attn_delta_kernel(const float* __restrict__ O, const typename Grad<DTYPE>::T* __restrict__ dO, float* __restrict__ D,
                           const long rows, const int H, const int N, const GdStrides st, const GdExtra ex)
{
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < H; i += GD_THREADS) {
            if (ex.zero_a) ex.zero_a[i] = 0.f;
            if (ex.zero_b) ex.zero_b[i] = 0.f;
        }
    constexpr int RPW = GD_THREADS / LPR;                    // rows per workgroup
    const int  sub = threadIdx.x % LPR;
    const long row = (long)blockIdx.x * RPW + threadIdx.x / LPR;
    float s = 0.f;
    if (row < rows) {
        const long n = row % N, zh = row / N;
        const long h = zh % H, z = zh / H;
        float a[4], b[4];
        const float* po = O + z * st.o[0] + h * st.o[1] + n * st.o[2] + 4 * sub;
        Grad<DTYPE>::load(dO + z * st.g[0] + h * st.g[1] + n * st.g[2] + 4 * sub, b);
        const float4 t = *reinterpret_cast<const float4*>(po);
        a[0] = t.x; a[1] = t.y; a[2] = t.z; a[3] = t.w;
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_fmaf(a[e], b[e], s);
        typedef proteus_ops::Operand<F16> Op;
        if (ex.cast) *reinterpret_cast<uint2*>(ex.cast + z * st.c[0] + h * st.c[1] + n * st.c[2] + 4 * sub) = make_uint2(Op::pack(b[0], b[1]), Op::pack(b[2], b[3]));
    }
    // (rows of a wave all take part: a row past the end adds zeros among its own lanes)
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (row < rows && sub == 0) D[row] = s;
}

template <int DTYPE, bool F16>
int launch(const float* O, const void* dO, float* D, int Z, int H, int N, int d, const GdStrides& st, const GdExtra& ex, hipStream_t stream)
{
    typedef typename Grad<DTYPE>::T T;
    const long rows = (long)Z * H * N;
    const int  lpr = d / 4;
    const dim3 grid((unsigned)((rows + GD_THREADS / lpr - 1) / (GD_THREADS / lpr)));
    if (lpr == 8)       hipLaunchKernelGGL((geo_attn_delta_kernel<DTYPE, 8, F16>), grid, dim3(GD_THREADS), 0, stream, O, (const T*)dO, D, rows, H, N, st, ex);
    else if (lpr == 16) hipLaunchKernelGGL((geo_attn_delta_kernel<DTYPE, 16, F16>), grid, dim3(GD_THREADS), 0, stream, O, (const T*)dO, D, rows, H, N, st, ex);
    else                hipLaunchKernelGGL((geo_attn_delta_kernel<DTYPE, 32, F16>), grid, dim3(GD_THREADS), 0, stream, O, (const T*)dO, D, rows, H, N, st, ex);
    return (int)hipGetLastError();
}

int check(const float* O, const void* dO, const int64_t* strides, const float* D, int Z, int H, int N, int d_head, int dtype, GdStrides& st)
{
    if (!O || !dO || !D) return PROTEUS_ERR_NULL_POINTER;
    if (d_head != 32 && d_head != 64 && d_head != 128) return PROTEUS_ERR_BAD_HEAD_DIM;
    if (dtype != PROTEUS_DTYPE_F32 && dtype != PROTEUS_DTYPE_BF16 && dtype != PROTEUS_DTYPE_F16) return PROTEUS_ERR_BAD_OPERAND_TYPE;
    if (Z <= 0 || H <= 0 || N <= 0 || N > PROTEUS_ATTN_MAX_N || (long)Z * H > 65535) return PROTEUS_ERR_BAD_SHAPE;
    if ((long)Z * H * N / (GD_THREADS / (d_head / 4)) >= (1L << 31) - 1) return PROTEUS_ERR_BAD_SHAPE;      // grid.x below 2^31
    const int gbytes = dtype == PROTEUS_DTYPE_F32 ? 4 : 2;
    if (((uintptr_t)O & 15) || ((uintptr_t)dO & (uintptr_t)(4 * gbytes - 1)) || ((uintptr_t)D & 3)) return PROTEUS_ERR_BAD_ALIGNMENT;
    if (!strides) {
        st.o[0] = st.g[0] = (long)H * N * d_head; st.o[1] = st.g[1] = (long)N * d_head; st.o[2] = st.g[2] = d_head;
        return PROTEUS_OK;
    }
    for (int i = 0; i < 3; ++i) { st.o[i] = (long)strides[i]; st.g[i] = (long)strides[3 + i]; }
    for (int i = 0; i < 3; ++i) {
        // rows of d elements must not overlap and every row must start on a 16-byte (O) / 4-element (dO) boundary
        if (st.o[i] < 0 || st.g[i] < 0) return PROTEUS_ERR_BAD_LAYOUT;
        if ((st.o[i] & 3) || (st.g[i] & 3)) return PROTEUS_ERR_BAD_ALIGNMENT;
    }
    if (st.o[2] < d_head || st.g[2] < d_head) return PROTEUS_ERR_BAD_LAYOUT;
    return PROTEUS_OK;
}

// strides[9]: of O, dO and the cast of dO, whose rows start on multiples of 16 bytes as the backward wants its operands
int check_prepare(const float* O, const void* dO, const int64_t* strides, const float* D, const uint16_t* cast,
                  int Z, int H, int N, int d_head, int dtype, int operand_type, GdStrides& st)
{
    const int rc = check(O, dO, strides, D, Z, H, N, d_head, dtype, st);
    if (rc != PROTEUS_OK) return rc;
    if (operand_type != PROTEUS_OPERAND_BF16 && operand_type != PROTEUS_OPERAND_F16) return PROTEUS_ERR_BAD_OPERAND_TYPE;
    if ((uintptr_t)cast & 15) return PROTEUS_ERR_BAD_ALIGNMENT;
    for (int i = 0; i < 3; ++i) st.c[i] = strides && cast ? (long)strides[6 + i] : st.o[i];
    if (strides && cast) {
        for (int i = 0; i < 3; ++i) {
            if (st.c[i] < 0) return PROTEUS_ERR_BAD_LAYOUT;
            if (st.c[i] & 7) return PROTEUS_ERR_BAD_ALIGNMENT;
        }
        if (st.c[2] < d_head || (Z > 1 && st.c[0] == 0) || (H > 1 && st.c[1] == 0)) return PROTEUS_ERR_BAD_LAYOUT;
    }
    return PROTEUS_OK;
}

int launch_any(bool f16, const float* O, const void* dO, float* D, int Z, int H, int N, int d, int dtype, const GdStrides& st, const GdExtra& ex, hipStream_t s)
{
#define GD_GO(T_) (f16 ? launch<T_, true>(O, dO, D, Z, H, N, d, st, ex, s) : launch<T_, false>(O, dO, D, Z, H, N, d, st, ex, s))
    if (dtype == PROTEUS_DTYPE_F32)  return GD_GO(PROTEUS_DTYPE_F32);
    if (dtype == PROTEUS_DTYPE_BF16) return GD_GO(PROTEUS_DTYPE_BF16);
    return GD_GO(PROTEUS_DTYPE_F16);
#undef GD_GO
}

}  // namespace

extern "C" int proteus_geo_attn_delta_check(const float* O, const void* dO, const int64_t* strides, const float* D,
                                            int Z, int H, int N, int d_head, int dO_dtype)
{
    GdStrides st;
    return check(O, dO, strides, D, Z, H, N, d_head, dO_dtype, st);
}

extern "C" int proteus_geo_attn_delta(const float* O, const void* dO, const int64_t* strides, float* D,
                                      int Z, int H, int N, int d_head, int dO_dtype, void* stream)
{
    GdStrides st;
    const int rc = check(O, dO, strides, D, Z, H, N, d_head, dO_dtype, st);
    if (rc != PROTEUS_OK) return rc;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    return launch_any(false, O, dO, D, Z, H, N, d_head, dO_dtype, st, GdExtra{nullptr, nullptr, nullptr}, s);
}

extern "C" int proteus_geo_attn_prepare_bwd_check(const float* O, const void* dO, const int64_t* strides, const float* D, const uint16_t* dO_cast,
                                                  const float* d_sigma, const float* d_beta, int Z, int H, int N, int d_head, int dO_dtype, int operand_type)
{
    (void)d_sigma; (void)d_beta;
    GdStrides st;
    return check_prepare(O, dO, strides, D, dO_cast, Z, H, N, d_head, dO_dtype, operand_type, st);
}

extern "C" int proteus_geo_attn_prepare_bwd(const float* O, const void* dO, const int64_t* strides, float* D, uint16_t* dO_cast,
                                            float* d_sigma, float* d_beta, int Z, int H, int N, int d_head, int dO_dtype, int operand_type, void* stream)
{
    GdStrides st;
    const int rc = check_prepare(O, dO, strides, D, dO_cast, Z, H, N, d_head, dO_dtype, operand_type, st);
    if (rc != PROTEUS_OK) return rc;
    return launch_any(operand_type == PROTEUS_OPERAND_F16, O, dO, D, Z, H, N, d_head, dO_dtype, st, GdExtra{dO_cast, d_sigma, d_beta},
                      reinterpret_cast<hipStream_t>(stream));
}
