// Gradients of weights of one layer: each may leave the sums of its shares of K to a launch that does all of them (gemm_f32.hip).
#pragma once

#include <hip/hip_runtime.h>
#include "proteus_hip.h"

namespace proteus_gemm {

struct GemmArgs {
    const float *A, *B, *bias, *h;
    void  *C;
    float *H;
    int M, N, K, lda, ldb, ldc, tiles_n, tiles, per_xcd;
    float *part;                                    // sums of the shares of K, where a product is cut
    int shares, steps;                              // their number, and the steps of each
};

// Products whose shares are not added up yet, and the workgroups of the launch that does it: first[i] to first[i + 1] for product i.
struct PendingSums {
    static constexpr int MOST = 4;
    GemmArgs product[MOST];
    int first[MOST + 1] = {0};
    int count = 0;
};

// C = A^T B as proteus_gemm_f32_ws gives it, or, where it is cut, once gemm_sums has run; until then `ws` is the product's own, and A and B
// stay as they are (elements that are not finite are summed again from them).
__attribute__((visibility("hidden")))
int gemm_begin(const float* A, const float* B, float* C, int M, int N, int K, int lda, int ldb, int ldc, void* ws, size_t ws_bytes, PendingSums& sums, void* stream);
__attribute__((visibility("hidden")))
int gemm_sums(PendingSums& sums, void* stream);

}  // namespace proteus_gemm
