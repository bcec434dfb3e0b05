// Internal interface of the split-operand kernels (gemm_split.hip): fp32 matrix
// products and convolutions on the bf16 matrix cores, every fp32 operand taken
// as the exact sum of three bf16 values.
#pragma once

#include <cstddef>
#include <cstdint>

namespace camel_hip {

struct SplitGemm {
    const float *A;    // [M, lda] row-major, or At [K, lda] (a_trans)
    const float *B;    // [K, ldb] row-major; conv: x
    float *C;          // [M, ldc] row-major; conv: y
    const float *bias; // per column (conv: per row), or null
    float *partial;    // split-K partial sums [split][M][N], or null
    int M, N, K;
    int lda, ldb, ldc;
    int k_per_split; // set by the launch
    int flags;       // CAMEL_EPI_*, conv: CAMEL_CONV_Y_NCHW4
};

// How the split kernels run a GEMM: the tile and the K splits.
enum class SplitTile { None, T256, T128 };
struct SplitPlan {
    SplitTile tile = SplitTile::None;
    int splits = 1;
    size_t partial_bytes = 0;
};

// The plan for C[M, N] = A[M, K] B[K, N]; SplitTile::None where the fp32 MFMA
// kernels are faster or the kernels' 32-bit offsets do not reach.
// `unaligned`: A transposed or an operand without 16-byte aligned rows.
SplitPlan split_gemm_plan(int64_t M, int64_t N, int64_t K, bool unaligned, int64_t lda, int64_t ldb,
                          int cus);
// Runs it on the library stream; `partial`: plan.partial_bytes of scratch.
int split_gemm(SplitGemm g, bool a_trans, const SplitPlan &plan, float *partial);

} // namespace camel_hip
