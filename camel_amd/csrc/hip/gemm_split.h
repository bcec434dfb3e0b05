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

// A convolution as that GEMM: M = output channels, N = pixels (batch OH OW, or
// 4 per pool window), K = taps x channels padded to a multiple of 8 (see `unit`).
struct SplitConv {
    typedef uint32_t chunk __attribute__((ext_vector_type(4)));
    // set by split_conv, with kpad, unit, taps, shift, the multipliers, patch
    // and per_image
    const chunk *w_split;
    int kpad;
    int C, H, W, KH, KW, stride, pad;
    int unit, taps; // K as runs of `unit` channels of one of the taps
    int P, OW;    // output pixels per image, width
    int PW, PP;   // pool windows per row, per image (pooled)
    int CHW, HW;  // input elements per image, per plane
    int pxs, cqs; // distance of pixels and (quads) of channel quads
    int shift;    // elements before x that the first window reaches back
    uint32_t bytes;          // of x and the shift before it
    uint32_t mul_unit;                   // floor(k / unit) = k mul_unit >> 32
    uint32_t mul_kw, mul_taps;           // tap_mul of KW and taps
    int patch, per_image;    // positions of a patch (0: not that kernel), tiles per image
    int w_packed;            // weights [Co][KH][KW][C], else [Co][C][KH][KW]
};

// How the split kernels run a GEMM: the tile and the K splits.
enum class SplitTile { None, T256, T128, T64 };
struct SplitPlan {
    SplitTile tile = SplitTile::None;
    int splits = 1;
    size_t partial_bytes = 0;
};

// The plan for C[M, N] = A[M, K] B[K, N]; SplitTile::None where the fp32 MFMA
// kernels are faster or the kernels' 32-bit offsets do not reach.
// `a_unaligned`, `b_unaligned`: an operand without 16-byte aligned rows.
SplitPlan split_gemm_plan(int64_t M, int64_t N, int64_t K, bool a_trans, bool a_unaligned, bool b_unaligned,
                          int64_t lda, int64_t ldb, int cus);
// Runs it on the library stream; `partial`: plan.partial_bytes of scratch.
int split_gemm(SplitGemm g, bool a_trans, const SplitPlan &plan, float *partial);

// True when split_conv serves the geometry (any layout): c's C, H, W, KH, KW,
// stride and pad, N images, `pixels` of output in all.
bool split_conv_serves(const SplitConv &c, int64_t N, int64_t pixels, int64_t Co, int cus);
// The kernel and K splits of a convolution and its scratch: the split weights,
// then the partial sums.
struct SplitConvPlan {
    int blocked = 0, patch = 0;
    int per_image = 0;
    int splits = 1;
    size_t weight_bytes = 0, partial_bytes = 0;
};
// (g.N: the pixels of the unpooled output, here and below.)
SplitConvPlan split_conv_plan(const SplitGemm &g, const SplitConv &c, bool pool, int cus);
// Runs it (`quads`: x in NHWC or NCHW4, else NCHW; `pool`: the 2x2 pooled
// output); `scratch`: weight_bytes + partial_bytes.
int split_conv(SplitGemm g, SplitConv c, bool quads, bool pool, const SplitConvPlan &plan, void *scratch);

// y = maxpool2x2(conv2(conv1(x))), x [N, 1, H, 28], conv1 1 -> 32 and conv2 32 ->
// Co2, both 3x3, stride 1, unpadded.
constexpr int PAIR_C1 = 32;
struct SplitPair {
    const float *x, *w1, *b1, *w2, *b2;
    float *y;
    int H, Co2, bands; // bands: set by split_pair
    int flags1, flags2, w2_packed;
};
bool split_pair_serves(int64_t H, int64_t W, int64_t C1, int64_t Co2);
size_t split_pair_bytes(int64_t Co2); // scratch for conv2's split weights
int split_pair(SplitPair p, int N, void *scratch);

} // namespace camel_hip
