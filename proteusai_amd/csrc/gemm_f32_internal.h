// Gradients of weights of one layer: each may leave the sums of its shares of K to a launch that does all of them (gemm_f32.hip).
#pragma once

#include <hip/hip_runtime.h>
#include "proteus_hip.h"
#include "train_internal.h"

namespace proteus_gemm {

struct GemmArgs {
    const float *A, *B, *bias, *h;
    void  *C;
    float *H;
    int M, N, K, lda, ldb, ldc, tiles_n, tiles, per_xcd;
    float *part;                                    // sums of the shares of K, where a product is cut
    int shares, steps;                              // their number, and the steps of each
};

// Products whose shares are not added up yet and column sums that are yet to be made, for the launch that does it: tiles first[i] to first[i + 1] are product i's,
// workgroups first_column[i] to first_column[i + 1] behind those of the tiles column sum i's.
struct PendingSums {
    static constexpr int MOST = 4;
    GemmArgs product[MOST];
    int first[MOST + 1] = {0};
    int count = 0;
    proteus_train::ColumnSums columns[MOST];
    int first_column[MOST + 1] = {0};
    int column_count = 0;
    // Takes column sums on where one workgroup does all rows.
    bool add(const proteus_train::ColumnSums& c)
    {
        if (column_count == MOST || c.rows > proteus_train::CS_ROWS) return false;
        columns[column_count] = c;
        first_column[column_count + 1] = first_column[column_count] + (c.cols + proteus_train::CS_COLS - 1) / proteus_train::CS_COLS;
        ++column_count;
        return true;
    }
};

// C = A^T B as proteus_gemm_f32_ws gives it, or, where it is cut, once gemm_sums has run; until then `ws` is the product's own, and A and B
// stay as they are (elements that are not finite are summed again from them).
__attribute__((visibility("hidden")))
int gemm_begin(const float* A, const float* B, float* C, int M, int N, int K, int lda, int ldb, int ldc, void* ws, size_t ws_bytes, PendingSums& sums, void* stream);
// (what the column sums are of stays as it is until then, too)
__attribute__((visibility("hidden")))
int gemm_sums(PendingSums& sums, void* stream);

}  // namespace proteus_gemm
