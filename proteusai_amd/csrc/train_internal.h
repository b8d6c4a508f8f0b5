// Column sums of the training step (encoder_train.hip), which a launch that adds up other things may do as well (gemm_f32.hip).
#pragma once

#include <hip/hip_runtime.h>
#include "proteus_hip.h"

namespace proteus_train {

constexpr int CS_COLS   = 16;           // columns of a column-sum workgroup: 64 bytes of a row
constexpr int CS_BLOCK  = 512;          // 4 threads of 16 bytes x 128 rows
constexpr int CS_ROWS   = 2048;         // rows a column-sum workgroup takes before the rows are cut into slabs

struct ColumnSums { const float* a; float* out; int rows, cols; };      // out[c] = sum over the rows of a[row][c]

// out[c] = sum over rows r0 to r1 of a[row][c] for the 16 columns from `block` * 16 on.  torch's reduction 10.8 - 14.1 us with a clearing launch in front, a launch
// of this 5.6 - 6.3 (2048 columns).
__device__ __forceinline__ void column_sums(const float* __restrict__ a, float* __restrict__ out, const long r0, const long r1, const int C, const int block,
                                            float (&red)[CS_BLOCK / 64][CS_COLS])
{
    const int q = threadIdx.x & 3, r = threadIdx.x >> 2;
    const int col = block * CS_COLS + q * 4;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (col < C) {
#pragma unroll 4
        for (long row = r0 + r; row < r1; row += CS_BLOCK / 4) {
            const float4 v = *reinterpret_cast<const float4*>(a + (size_t)row * C + col);
            s[0] += v.x; s[1] += v.y; s[2] += v.z; s[3] += v.w;
        }
    }
#pragma unroll
    for (int o = 4; o < 64; o <<= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += __shfl_xor(s[e], o);
    if ((threadIdx.x & 63) < 4)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[threadIdx.x >> 6][q * 4 + e] = s[e];
    __syncthreads();
    const int c = block * CS_COLS + threadIdx.x;
    if (threadIdx.x < CS_COLS && c < C) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < CS_BLOCK / 64; ++w) t += red[w][threadIdx.x];
        out[c] = t;
    }
}

// proteus_layernorm_bwd without its last launch: `sums` is what that has yet to do.
__attribute__((visibility("hidden")))
int layernorm_bwd_begin(const float* dout, const float* ysum, const float* stat, const float* gamma, float* dx, float* dgamma_dbeta, void* ws, size_t ws_bytes, long rows, int D,
                        ColumnSums& sums, void* stream);

}  // namespace proteus_train
