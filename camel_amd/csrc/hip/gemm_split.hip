// fp32 GEMM on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16), which run 16
// times the fp32 MFMA rate.
//
// Every fp32 operand x is scaled by 2^24 and taken as hi + mid + lo, three bf16
// values: hi = x and mid = x - hi rounded to nearest, lo = the rest.
// 24 significant bits make three 8-bit parts, so the sum is x exactly: the last
// bit of a scaled value is at least 2^-125, inside the bf16 range, for
// subnormal x too.  The results are scaled back by 2^-48.  A product of two such
// operands is the six part products hi hi, hi mid, mid hi, mid mid, hi lo, lo
// hi, each exact in fp32.  The three others are dropped: |mid| <= 2^-8 and |lo| <=
// 2^-17 of the leading bit, so they are at most 2^-24 (1 + 2^-9) of the product.
//
// Sums: the 6 MFMAs of a 16 x 16 block and 32 k start from zero, smallest
// products first, and their sum is added to the block's fp32 accumulator on
// the vector ALU (round to nearest).  An accumulator is rounded once per 32 k:
// error against fp64 at 4096^3, U(-1, 1): 2.1e-7 (2-norm), against 1.1e-6 for
// the fp32 MFMA chain, which rounds every 2 k.  (The 6 MFMAs on the
// accumulator itself: 1.03e-6, 4% faster.)
//
// One product by itself: the MFMA cuts its sum where an fp32 product rounds, so
// a sum of one term is off by up to 1.5 units of its last place (the cut 1, the
// dropped products 0.5; measured 1.46, 2-norm 3.1e-8 against 2.5e-8 of a rounded
// product).  With hi hi in a sum of its own, added on the vector ALU, it is 1.0
// (measured 0.96, 2-norm 2.5e-8); the 64 x 64 tile, whose three chains need that
// add anyway, does so, the others would run 3 to 7% longer (4096^3 537 -> 567 us,
// conv 64 x 64 x 56 x 56 140 -> 150).  With the two products mid lo and lo mid as
// well it is 0.51 (measured), at 4096^3 537 -> 685.  Sums of more terms are
// more exact than the fp32 chain's in all forms: 64 terms 4.5e-8 against 1.4e-7.
//
// The top of the range: |x| >= 2^104, infinities and NaN make hi infinite or NaN
// and mid NaN, and a sum can pass 2^80 (the fp32 maximum, scaled).  Either way
// the output is not finite, and non-finite outputs, each by itself, are formed
// again in fp32 MFMA: special values and the ends of the range give what they
// give in fp32, and no output depends on another row or column.
// That takes time only where such values are: 4096^3 550 us (fp32 kernels 960),
// with one infinity 1560, with all sums past 2^80 2510.
//
// Tile: waves as WM x WN, each FM x FN blocks of 16 x 16; A goes from global
// memory straight into the registers of the waves that multiply it (lane (r,
// o) of a block: 8 k of row r, 32 bytes), B through LDS, converted once per
// work-group: three planes per stage of 32 k, [part][octet][column] chunks of
// 8 bf16, so that stores (64 columns of an octet) and operand reads (16
// columns of each of 4 octets; BN % 16 == 0 chunks per octet) touch every bank
// once.  Global loads run one stage ahead of their conversion, a stage of B is
// stored while the one before is multiplied, one barrier a stage.  The MFMA
// operands are exchanged (D = B^T A^T), so a lane's 4 results are 4
// consecutive columns: one 16-byte store.
#include "common.h"
#include "gemm_split.h"

#include <algorithm>
#include <type_traits>

namespace camel_hip {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4))); // 16-byte access, 4-byte aligned
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int BK = 32;     // k per stage: one 16x16x32 MFMA
constexpr int GROUP_M = 4; // tile rows per group of the XCD-aware order

// The scale of each operand, and of the result back.
constexpr float SCALE = 0x1p24f, UNSCALE = 0x1p-48f;

// The upper halves of two floats, x0 in the lower half.
__device__ __forceinline__ uint32_t upper_pair(float x0, float x1) {
    return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}

// Pair c of f[0..7] (split8: all four) into three chunks of 8 bf16 (hi, mid,
// lo).  (v_dot2_f32_bf16 with a -1 forms x - hi in one operation instead of two,
// but its results may not be read for 3 wait states: 4096^3 557 -> 578 us.)
__device__ __forceinline__ void split_pair(const float *f, int c, u4 *out) {
    // (The factor in a scalar register instead of a literal: half the size of the
    // multiplication; 16 x 96 x 55 x 55 stride 2 60.8 -> 56.7 us.)
    float scale = SCALE;
    asm("" : "+s"(scale));
    float x0 = f[2 * c] * scale, x1 = f[2 * c + 1] * scale;
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){x0, x1}, bf2));
    x0 = x0 - __uint_as_float(h << 16);
    x1 = x1 - __uint_as_float(h & 0xffff0000u);
    const uint32_t m = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){x0, x1}, bf2));
    out[0][c] = h;
    out[1][c] = m;
    out[2][c] = upper_pair(x0 - __uint_as_float(m << 16), x1 - __uint_as_float(m & 0xffff0000u));
}
__device__ __forceinline__ void split8(const float *f, u4 *out) {
#pragma unroll
    for (int c = 0; c < 4; ++c) split_pair(f, c, out);
}

// Operands of the part products, smallest first: (lo hi), (hi lo), (mid mid),
// (mid hi), (hi mid), (hi hi).
constexpr int PRODUCTS = 6;
constexpr int PA[PRODUCTS] = {2, 0, 1, 1, 0, 0}, PB[PRODUCTS] = {0, 2, 1, 0, 1, 0};

// Adds the scaled products of 32 k to a block's accumulator.
__device__ __forceinline__ void add_products(f4 &acc, f4 t) {
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(t[v], UNSCALE, acc[v]);
}

// WM x WN waves of FM x FN blocks; WK groups of them take alternate stages of
// K, and their sums meet in LDS in group order.
template <int FM_, int FN_, int WM_, int WN_, int WK_> struct STile {
    static constexpr int FM = FM_, FN = FN_, WM = WM_, WN = WN_, WK = WK_;
    static constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN;
    static constexpr int GW = WM * WN; // waves of a group
    static constexpr int THREADS = 64 * GW * WK;
    static constexpr int SB = BK * WK;     // k per step of all groups
    static constexpr int B_ST = 12 * BN;   // chunks per stage
    static constexpr int B_IT = BN / 16 / GW; // (64 columns, octet) items per wave and stage
    static constexpr int LDS = 2 * WK * B_ST;
    static_assert(BN % 64 == 0 && BN / 16 % GW == 0, "whole column items per wave");
    static_assert((WK - 1) * FM * FN * GW * 64 <= LDS, "group sums fit the stage buffers");
    static_assert(FN >= 4, "the stage's store, barrier and next reads fall on different columns");
};

// Logical tile id -> (tm, tn), grouped GROUP_M tile rows deep.
__device__ __forceinline__ void split_tile_of(int id, int tiles_m, int tiles_n, int &tm, int &tn) {
    const int per_group = GROUP_M * tiles_n;
    const int g = id / per_group;
    const int first_m = g * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = id - g * per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// Where the A operand comes from: row-major fp32, transposed fp32, or already
// split ([stage][16-row block][part][64 lanes] chunks, the conv weights).
enum ASource { A_ROWS, A_COLS, A_SPLIT };
enum Output { OUT_MATRIX, OUT_CONV, OUT_POOL };

// B as a row-major matrix: lane = column, octet o of a stage = rows 8 o .. +7,
// 256 contiguous bytes of a row per load.
template <class T> struct MatrixB {
    const float *base;
    int ld;
    uint32_t off[T::B_IT];
    __device__ __forceinline__ MatrixB(const SplitGemm &g, const SplitConv &) : base(g.B), ld(g.ldb) {}
    __device__ __forceinline__ void column(const SplitGemm &g, const SplitConv &, int i, int n) {
        off[i] = (uint32_t)min(n, g.N - 1) * 4u;
    }
    // 8 rows from k (all inside [0, K))
    __device__ __forceinline__ void load(int i, int k, float *f) const {
        const char *q = reinterpret_cast<const char *>(base + (size_t)k * ld);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            f[j] = *reinterpret_cast<const float *>(q + off[i]);
            q += (size_t)ld * sizeof(float);
        }
    }
    // rows below 0 are zero
    __device__ __forceinline__ void load_ragged(int i, int k, float *f) const {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            f[j] = k + j < 0 ? 0.f
                             : *reinterpret_cast<const float *>(
                                   reinterpret_cast<const char *>(base + (size_t)(k + j) * ld) + off[i]);
    }
    __device__ __forceinline__ static float at(const SplitGemm &g, const SplitConv &, int k, int n) {
        return g.B[(size_t)k * g.ldb + n];
    }
};

// Image, row and column of GEMM column n of a convolution: pixels in order, or
// (POOL) 4 per window of the 2x2 pool, ((0,0), (0,1), (1,0), (1,1)).
template <bool POOL>
__device__ __forceinline__ void conv_pixel(const SplitConv &c, int n, int &img, int &oh, int &ow) {
    if constexpr (POOL) {
        img = n / (4 * c.PP);
        const int r = n - img * 4 * c.PP, win = r >> 2, d = r & 3, ph = win / c.PW;
        oh = 2 * ph + (d >> 1);
        ow = 2 * (win - ph * c.PW) + (d & 1);
    } else {
        img = n / c.P;
        const int r = n - img * c.P;
        oh = r / c.OW;
        ow = r - oh * c.OW;
    }
}

// Tap and channel of k: runs of `unit` channels of one tap, tap after tap, then
// the next `unit` channels (unit: all channels padded to 8, or 32).
__device__ __forceinline__ void conv_k(const SplitConv &c, int k, int &tap, int &ch) {
    const int run = k / c.unit, blk = run / c.taps;
    tap = run - blk * c.taps;
    ch = blk * c.unit + k - run * c.unit;
}

// floor(n / d) for d <= 32 taps and n < 8192 runs of channels as a product: the
// multiplier 2^18 / d + 1 fits 32 bits for d = 1 too, and the product as well.
// (A branch for d = 1 in the stage loop: 16 x 96 x 55 x 55 stride 2 60 -> 68 us.)
constexpr uint32_t tap_mul(uint32_t d) { return (1u << 18) / d + 1; }
__host__ __device__ __forceinline__ constexpr uint32_t tap_quotient(uint32_t n, uint32_t mul) {
    return n * mul >> 18;
}
constexpr bool tap_quotients_hold() {
    for (uint32_t d = 1; d <= 32; ++d)
        for (uint32_t n = d; n <= 8192; n += d) // both ends of each quotient
            if (tap_quotient(n - 1, tap_mul(d)) != n / d - 1 || (n < 8192 && tap_quotient(n, tap_mul(d)) != n / d))
                return false;
    return true;
}
static_assert(tap_quotients_hold(), "divisions of the convolution's k");

// Element (k, n) of the im2col matrix.
template <bool QUADS, bool POOL>
__device__ __forceinline__ float conv_input(const SplitGemm &g, const SplitConv &c, int k, int n) {
    int tap, ch;
    conv_k(c, k, tap, ch);
    const int kh = tap / c.KW, kw = tap - kh * c.KW;
    int img, oh, ow;
    conv_pixel<POOL>(c, n, img, oh, ow);
    const int ih = oh * c.stride - c.pad + kh, iw = ow * c.stride - c.pad + kw;
    if (ch >= c.C || (unsigned)ih >= (unsigned)c.H || (unsigned)iw >= (unsigned)c.W) return 0.f;
    const size_t px = (size_t)img * c.CHW + (size_t)(ih * c.W + iw) * c.pxs;
    return QUADS ? g.B[px + (size_t)(ch >> 2) * c.cqs + (ch & 3)] : g.B[px + (size_t)ch * c.HW];
}

// B as the im2col matrix of a convolution, K ordered as conv_k: an octet is 8 channels of one tap, the
// same for a whole wave, so its offset is scalar, and a lane's pixel gives the
// vector offset.  Buffer loads: a lane whose tap lies in the padding (a bit
// per tap, decoded once) or a channel past C takes an offset past the end of
// the buffer, which reads zero.  QUADS: channel quads 16 bytes apart in
// memory or side by side (NHWC, NCHW4), two 16-byte loads; else 8 planes, 256
// contiguous bytes of one each (for a stride of 1).
constexpr uint32_t NO_ELEMENT = 1u << 31; // buffers and scalar offsets stay below 2^31 bytes
template <class T, bool QUADS, bool POOL> struct ConvB {
    const SplitConv &c;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t off[T::B_IT], taps[T::B_IT];
    __device__ __forceinline__ ConvB(const SplitGemm &g, const SplitConv &cv) : c(cv) {
        // offsets count from `shift` elements before x, so that the window of
        // the first pixel starts at 0
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.B - c.shift), 0, c.bytes, 0x00027000);
    }
    __device__ __forceinline__ void column(const SplitGemm &g, const SplitConv &, int i, int n) {
        int img, oh, ow;
        conv_pixel<POOL>(c, min(n, g.N - 1), img, oh, ow);
        const int ih = oh * c.stride - c.pad, iw = ow * c.stride - c.pad;
        off[i] = (uint32_t)(img * c.CHW + (ih * c.W + iw) * c.pxs + c.shift) * 4u;
        uint32_t m = 0;
        for (int kh = 0, t = 0; kh < c.KH; ++kh)
            for (int kw = 0; kw < c.KW; ++kw, ++t)
                m |= ((unsigned)(ih + kh) < (unsigned)c.H && (unsigned)(iw + kw) < (unsigned)c.W) ? 1u << t : 0u;
        taps[i] = m;
    }
    __device__ __forceinline__ void load(int i, int k, float *f) const {
        const int run = (int)__umulhi((uint32_t)k, c.mul_unit), blk = (int)tap_quotient(run, c.mul_taps);
        const int tap = run - blk * c.taps, c0 = blk * c.unit + k - run * c.unit;
        const int kh = (int)tap_quotient(tap, c.mul_kw), kw = tap - kh * c.KW;
        const uint32_t v = (taps[i] >> tap) & 1 ? off[i] : NO_ELEMENT;
        const uint32_t s = (uint32_t)((kh * c.W + kw) * c.pxs) * 4u;
        if constexpr (QUADS) {
            const uint32_t so = s + (uint32_t)((c0 >> 2) * c.cqs) * 4u;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u4 q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, c0 + 4 * h < c.C ? v : NO_ELEMENT,
                                                                   so + (uint32_t)(h * c.cqs) * 4u, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) f[4 * h + j] = __uint_as_float(q[j]);
            }
        } else {
            uint32_t so = s + (uint32_t)(c0 * c.HW) * 4u;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                f[j] = __uint_as_float(
                    __builtin_amdgcn_raw_buffer_load_b32(rsrc, c0 + j < c.C ? v : NO_ELEMENT, so, 0));
                so += (uint32_t)c.HW * 4u;
            }
        }
    }
    // an octet is wholly below 0 or not at all
    __device__ __forceinline__ void load_ragged(int i, int k, float *f) const {
        load(i, max(k, 0), f);
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = k < 0 ? 0.f : f[j];
    }
    __device__ __forceinline__ static float at(const SplitGemm &g, const SplitConv &c, int k, int n) {
        return conv_input<QUADS, POOL>(g, c, k, n);
    }
};

// Weight (row, k) of a convolution.
__device__ __forceinline__ float conv_weight(const SplitGemm &g, const SplitConv &c, int row, int k) {
    int tap, ch;
    conv_k(c, k, tap, ch);
    if (ch >= c.C) return 0.f;
    return g.A[c.w_packed ? ((size_t)row * c.taps + tap) * c.C + ch : ((size_t)row * c.C + ch) * c.taps + tap];
}

// The weights of a convolution as the MFMA operand, split: stage blockIdx.x,
// 16-row block blockIdx.y, lane (r16, oct) its 8 k.  Rows past Co repeat the
// last one.
__global__ __launch_bounds__(64) void split_weights_kernel(SplitGemm g, SplitConv c, u4 *dst) {
    const int lane = threadIdx.x, stage = blockIdx.x, blk = blockIdx.y;
    const int kpad = gridDim.x * BK - g.K;
    const int row = min(16 * blk + (lane & 15), g.M - 1), k0 = stage * BK - kpad + 8 * (lane >> 4);
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = k0 < 0 ? 0.f : conv_weight(g, c, row, k0 + j);
    u4 out[3];
    split8(f, out);
    u4 *d = dst + ((size_t)stage * gridDim.y + blk) * 192 + lane;
#pragma unroll
    for (int q = 0; q < 3; ++q) d[64 * q] = out[q];
}

// Lane (r16, oct) holds columns nw + 16 j + 4 oct .. +3 of rows mw + 16 i (mw
// and nw include the lane): bias and relu, or the split's partial sums.
template <int FM, int FN>
__device__ __forceinline__ void store_matrix(const SplitGemm &g, f4 (*acc)[FN], int split, int mw, int nw) {
    const bool part = g.partial != nullptr;
    const bool has_bias = (g.flags & CAMEL_EPI_BIAS) != 0 && !part;
    const bool has_relu = (g.flags & CAMEL_EPI_RELU) != 0 && !part;
    float *out = part ? g.partial + (size_t)split * g.M * g.N : g.C;
    const size_t ldo = part ? (size_t)g.N : (size_t)g.ldc;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int col = nw + 16 * j;
        f4 bv = f4{0.f, 0.f, 0.f, 0.f};
        if (has_bias)
#pragma unroll
            for (int v = 0; v < 4; ++v) bv[v] = col + v < g.N ? g.bias[col + v] : 0.f;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int row = mw + 16 * i;
            if (row >= g.M) continue;
            f4 x = acc[i][j];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (has_bias) x[v] = x[v] + bv[v];
                if (has_relu) x[v] = relu_idiom(x[v]);
            }
            float *o = out + (size_t)row * ldo + col;
            if (col + 3 < g.N)
                *reinterpret_cast<f4u *>(o) = x;
            else
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (col + v < g.N) o[v] = x[v];
        }
    }
}

// Image and place in it of GEMM column n of a convolution's output (per = P, or
// 4 PP columns per image when pooled).
struct ConvColumn {
    int img, p;
    __device__ __forceinline__ ConvColumn(int n, int per) : img(n / per), p(n - img * per) {}
    __device__ __forceinline__ void advance(int by, int per) {
        for (p += by; p >= per; p -= per) ++img;
    }
};

// 4 columns (from n, at col) of output channel `row` of a convolution: bias and
// relu, then NCHW, NCHW4, or (POOL: the columns are a window) the window's
// maximum by the pool's rule, first then strict '>'.
template <bool POOL>
__device__ __forceinline__ void store_conv_quad(const SplitGemm &g, const SplitConv &c, f4 x, int row, int n,
                                                ConvColumn col, float bias) {
    const bool q4 = (g.flags & CAMEL_CONV_Y_NCHW4) != 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (g.flags & CAMEL_EPI_BIAS) x[v] = x[v] + bias;
        if (g.flags & CAMEL_EPI_RELU) x[v] = relu_idiom(x[v]);
    }
    if constexpr (POOL) {
        float mx = x[0];
#pragma unroll
        for (int v = 1; v < 4; ++v)
            if (x[v] > mx) mx = x[v];
        g.C[((size_t)col.img * g.M + row) * c.PP + (col.p >> 2)] = mx;
        return;
    }
    if (!q4 && col.p + 3 < c.P) {
        *reinterpret_cast<f4u *>(g.C + ((size_t)col.img * g.M + row) * c.P + col.p) = x;
        return;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (n + v < g.N)
            g.C[q4 ? (size_t)col.img * g.M * c.P + (size_t)(row & ~3) * c.P + 4 * (size_t)col.p + (row & 3)
                   : ((size_t)col.img * g.M + row) * c.P + col.p] = x[v];
        col.advance(1, c.P);
    }
}

// The lanes' results (as store_matrix) of a convolution, rows = output
// channels; or the split's partial sums.
template <int FM, int FN, bool POOL>
__device__ __forceinline__ void store_conv(const SplitGemm &g, const SplitConv &c, f4 (*acc)[FN], int split,
                                           int mw, int nw) {
    if (g.partial) {
        SplitGemm part = g;
        part.flags = 0;
        store_matrix<FM, FN>(part, acc, split, mw, nw);
        return;
    }
    float bias[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i)
        bias[i] = (g.flags & CAMEL_EPI_BIAS) ? g.bias[min(mw + 16 * i, g.M - 1)] : 0.f;
    const int per = POOL ? 4 * c.PP : c.P;
    ConvColumn col(nw, per);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        if (nw + 16 * j >= g.N) break;
#pragma unroll
        for (int i = 0; i < FM; ++i)
            if (mw + 16 * i < g.M) store_conv_quad<POOL>(g, c, acc[i][j], mw + 16 * i, nw + 16 * j, col, bias[i]);
        col.advance(16, per);
    }
}

// Forms a wave's non-finite sums, and no others, again
// in fp32 (v_mfma_f32_16x16x4_f32, the same result layout): JW columns of blocks
// at a time, where any of them holds one.  a(i, k), b(j, k): this lane's
// operand of block row i, column j; a lane's k of 32 are 8 consecutive ones,
// loaded together.
template <int FM, int FN, int JW, int S, class A, class B>
__device__ __forceinline__ void finish_sums(f4 (*acc)[FN], int kbeg, int kend, int oct, A a, B b) {
    static_assert(FN % JW == 0, "columns in groups");
#pragma unroll
    for (int j0 = 0; j0 < FN; j0 += JW) {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = j0; j < j0 + JW; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) bad |= !(__builtin_fabsf(acc[i][j][v]) < INFINITY);
        if (!__any(bad)) continue;
        f4 y[FM][JW];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < JW; ++j) y[i][j] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int k0 = kbeg; k0 < kend; k0 += 4 * S) {
            float fa[FM][S], fb[JW][S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int k = min(k0 + S * oct + s, kend - 1);
#pragma unroll
                for (int i = 0; i < FM; ++i) fa[i][s] = a(i, k);
#pragma unroll
                for (int j = 0; j < JW; ++j) fb[j][s] = b(j0 + j, k);
            }
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const bool in = k0 + S * oct + s < kend; // past the end both are zero
#pragma unroll
                for (int j = 0; j < JW; ++j) fb[j][s] = in ? fb[j][s] : 0.f;
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    fa[i][s] = in ? fa[i][s] : 0.f;
#pragma unroll
                    for (int j = 0; j < JW; ++j)
                        y[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][s], fa[i][s], y[i][j], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < JW; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (!(__builtin_fabsf(acc[i][j0 + j][v]) < INFINITY)) acc[i][j0 + j][v] = y[i][j][v];
    }
}

// Stride-1 convolution with the input converted once per work-group instead
// of once per tap: a tile's output pixels read a contiguous range of the
// zero-padded image (position (img Hp + ih) Wp + iw; tap (kh, kw) adds kh Wp +
// kw), at most PATCH positions.  For 32 channels at a time that range goes to
// LDS as split chunks [part][octet][position]; all taps then multiply from it
// with no conversion, store or barrier between them, and the next 32 channels'
// loads are in flight meanwhile.  16 output pixels read 16 nearly always
// consecutive positions (an eighth of the LDS cycles are bank conflicts, where
// they straddle rows).  Weights come split, straight into registers, a tap ahead.
// 64 x 64 x 56 x 56 -> 128 3x3: 262 us on the fp32 MFMA implicit GEMM, 206 with
// the im2col loads above, 140 so (211 TFLOP/s; the matrix pipe busy for 68% of
// the kernel's cycles, the rest the patch's conversion, tile ends and 3.1 rounds).
template <int FM_, int FN_, int WM_, int WN_> struct PatchTile {
    static constexpr int FM = FM_, FN = FN_, WM = WM_, WN = WN_;
    static constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN;
    static constexpr int THREADS = 64 * WM * WN;
    static_assert(WM * WN == 4, "a wave per octet loads the patch");
};
constexpr int PATCH = 320;               // positions: 60 KiB, two work-groups per CU
constexpr int PATCH_IT = (PATCH + 63) / 64;

template <class T, bool QUADS, bool POOL>
__global__ __launch_bounds__(T::THREADS, 2) void conv_patch_kernel(SplitGemm g, SplitConv c) {
    __shared__ u4 patch[12 * PATCH];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / T::WN, wn = wave - wm * T::WN;
    const int r16 = lane & 15, oct = lane >> 4;
    const int per = POOL ? 4 * c.PP : c.P; // columns per image
    const int tiles_m = (g.M + T::BM - 1) / T::BM, tiles_i = (per + T::BN - 1) / T::BN;
    const int nt = gridDim.x; // tiles_m x (tiles of an image x images, or of all columns)
    int bid = blockIdx.x;
    if ((nt & 7) == 0) bid = (bid & 7) * (nt >> 3) + (bid >> 3);
    const int tn = bid / tiles_m, tm = bid - tn * tiles_m;
    const int m0 = tm * T::BM;
    // columns n0 .. nend - 1 (a tile of its image, or of all)
    const int n0 = c.per_image ? tn / tiles_i * per + tn % tiles_i * T::BN : tn * T::BN;
    const int nend = c.per_image ? (tn / tiles_i + 1) * per : g.N;
    const int Hp = c.H + 2 * c.pad, Wp = c.W + 2 * c.pad, taps = c.taps;
    auto position = [&](int n) {
        int img, oh, ow;
        conv_pixel<POOL>(c, min(n, nend - 1), img, oh, ow);
        return (img * Hp + oh) * Wp + ow;
    };
    // Columns past the tile's end repeat the last one.  (Pool order: a
    // window's first column has the least position, but windows of one pool
    // row come before the row below it, so the tile's least is column n0's.)
    const int q0 = position(n0);

    // This lane's patch items: position lane + 64 i, octet `wave`.
    uint32_t off[PATCH_IT];
    {
        const int last = g.N / per * Hp * Wp; // positions of all images
#pragma unroll
        for (int i = 0; i < PATCH_IT; ++i) {
            const int q = q0 + lane + 64 * i, row = q / Wp, iw = q - row * Wp - c.pad;
            const int img = row / Hp, ih = row - img * Hp - c.pad;
            const bool in = q < last && (unsigned)ih < (unsigned)c.H && (unsigned)iw < (unsigned)c.W;
            off[i] = in ? (uint32_t)(img * c.CHW + (ih * c.W + iw) * c.pxs) * 4u : NO_ELEMENT;
        }
    }
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(g.B), 0, c.bytes, 0x00027000);
    float raw[PATCH_IT][8];
    auto load_patch = [&](int blk) {
        const int c0 = blk * BK + 8 * wave;
#pragma unroll
        for (int i = 0; i < PATCH_IT; ++i) {
            if (64 * i >= c.patch) break;
            if constexpr (QUADS) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const u4 q = __builtin_amdgcn_raw_buffer_load_b128(
                        rsrc, c0 + 4 * h < c.C ? off[i] : NO_ELEMENT, (uint32_t)(((c0 >> 2) + h) * c.cqs) * 4u, 0);
#pragma unroll
                    for (int j = 0; j < 4; ++j) raw[i][4 * h + j] = __uint_as_float(q[j]);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    raw[i][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rsrc, c0 + j < c.C ? off[i] : NO_ELEMENT, (uint32_t)((c0 + j) * c.HW) * 4u, 0));
            }
        }
    };
    auto store_patch = [&]() {
#pragma unroll
        for (int i = 0; i < PATCH_IT; ++i) {
            if (64 * i >= c.patch) break;
            u4 d[3];
            split8(raw[i], d);
            if (64 * i + lane < PATCH)
#pragma unroll
                for (int q = 0; q < 3; ++q) patch[(q * 4 + wave) * PATCH + 64 * i + lane] = d[q];
        }
    };
    // Operand chunks of the lane's columns: at[j] + tap offset.
    int at[T::FN];
#pragma unroll
    for (int j = 0; j < T::FN; ++j)
        at[j] = oct * PATCH + position(n0 + (wn * T::FN + j) * 16 + r16) - q0;
    const int a_blocks = (g.M + 15) / 16;
    const u4 *a_src[T::FM];
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
        a_src[i] = c.w_split + (size_t)min(m0 / 16 + wm * T::FM + i, a_blocks - 1) * 192 + lane;
    const int blocks = (c.C + BK - 1) / BK, stages = blocks * taps;
    u4 an[T::FM][3];
    auto load_a = [&](int stage) { // past the end the last one again
        const size_t o = (size_t)min(stage, stages - 1) * a_blocks * 192;
#pragma unroll
        for (int i = 0; i < T::FM; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q) an[i][q] = a_src[i][o + 64 * q];
    };
    f4 acc[T::FM][T::FN];
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
        for (int j = 0; j < T::FN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    load_patch(0);
    load_a(0);
    bf8 b[2][3], a[T::FM][3];
    f4 t[2][T::FM];
    auto fetch = [&](int j, int tap_off, bf8 *d) {
#pragma unroll
        for (int q = 0; q < 3; ++q)
            d[q] = __builtin_bit_cast(bf8, patch[q * 4 * PATCH + at[j] + tap_off]);
    };
    int stage = 0;
    for (int blk = 0; blk < blocks; ++blk) {
        if (blk > 0) __syncthreads(); // the block before is multiplied
        store_patch();
        __syncthreads();
        if (blk + 1 < blocks) load_patch(blk + 1);
        fetch(0, 0, b[0]);
        int kw = 0, tap_off = 0;
        for (int tap = 0; tap < taps; ++tap, ++stage) {
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q) a[i][q] = __builtin_bit_cast(bf8, an[i][q]);
            load_a(stage + 1);
            // next tap's offset (after the last one this tap's again)
            int next_off = tap_off + 1;
            if (++kw == c.KW) {
                kw = 0;
                next_off = tap_off + 1 + Wp - c.KW;
            }
            if (tap + 1 == taps) next_off = tap_off;
#pragma unroll
            for (int j = 0; j < T::FN; ++j) {
                fetch((j + 1) % T::FN, j + 1 < T::FN ? tap_off : next_off, b[(j + 1) & 1]);
#pragma unroll
                for (int i = 0; i < T::FM; ++i) t[j & 1][i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = 0; p < PRODUCTS; ++p)
#pragma unroll
                    for (int i = 0; i < T::FM; ++i)
                        t[j & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j & 1][PB[p]], a[i][PA[p]],
                                                                              t[j & 1][i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < T::FM; ++i)
                    if (j > 0) add_products(acc[i][j - 1], t[(j + 1) & 1][i]);
#pragma unroll
                for (int r = 0; r < PRODUCTS * T::FM; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (r % T::FM == T::FM - 1 && r < 3 * T::FM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if (r >= T::FM) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < T::FM; ++i) add_products(acc[i][T::FN - 1], t[(T::FN - 1) & 1][i]);
            tap_off = next_off;
        }
    }

    const int mw = m0 + wm * T::FM * 16 + r16, nw = n0 + wn * T::FN * 16;
    finish_sums<T::FM, T::FN, 4, 2>(
        acc, 0, g.K, oct, [&](int i, int k) { return conv_weight(g, c, min(mw + 16 * i, g.M - 1), k); },
        [&](int j, int k) { return conv_input<QUADS, POOL>(g, c, k, min(nw + 16 * j + r16, nend - 1)); });
    SplitGemm tile = g;
    tile.N = nend;
    tile.partial = nullptr;
    store_conv<T::FM, T::FN, POOL>(tile, c, acc, 0, mw, nw + 4 * oct);
}

// ---- the first two convolutions of an image CNN, fused with the pool -----------
//
// y = maxpool2x2(conv2(conv1(x))) (each conv with its optional bias and relu)
// for a one-channel input: conv1 1 -> PAIR_C1 channels, 3x3, then conv2 PAIR_C1
// -> Co2, 3x3, both stride 1 and unpadded, then the 2x2 stride-2 pool.  conv1's
// output (PAIR_C1 x 26 x 26 per 28 x 28 image, 44 MB at batch 512) never
// reaches HBM: a work-group computes the rows of it that its band of conv2
// rows reads, splits them into LDS as the patch kernel's chunks, and multiplies
// all nine taps from there.
//   * work-group = (image, band of PAIR_BR pooled rows = 2 PAIR_BR conv2 rows) x
//     64 output channels; 4 waves as 2 (channels) x 2 (column halves) of 2 x 6
//     blocks; columns in pool order, a window per lane quad of results, 16
//     columns a 2 x 2 block of windows (pair_window);
//   * conv1: a wave an octet of channels, a lane a pixel, the weights scalar;
//     the direct kernel's FMA chain (k ascending, then bias and x * (x > 0)), so
//     the patch splits exactly the values the conv1 kernel stores;
//   * the MFMA sequence and the epilogue are those of the pooled split
//     convolution of 32 channels, so the result equals the two conv calls and
//     the pool bit for bit.
// The 16 pixels of 16 columns, (2 py + r, 2 px + c) for r, c in 0..3, lie on 16
// chunks that differ mod 16 at a row pitch of 28 (28 r = 0, 12, 8, 4 mod 16), so
// by the model of 16 lanes a clock the reads do not conflict; the conflict
// counter reads 43% of the LDS cycles all the same, which is not explained.  CNN
// forward at batch 512: 119.0 us with the pair in fp32 MFMA (98 us of it), 75.2 so
// (51 us, the matrix pipe busy for 58% of its cycles).
constexpr int PAIR_W = 28, PAIR_OW1 = PAIR_W - 2, PAIR_PW = (PAIR_OW1 - 2) / 2;
constexpr int PAIR_BR = 4;                     // pooled rows per work-group
constexpr int PAIR_R1 = 2 * PAIR_BR + 2;       // conv1 rows a band reads
constexpr int PAIR_IR = PAIR_R1 + 2;           // input rows a band reads
constexpr int PAIR_POS = PAIR_R1 * PAIR_W;     // chunk positions of a plane (row pitch 28)
constexpr int PAIR_COLS = PAIR_BR * PAIR_PW * 4;
constexpr int PAIR_FN = PAIR_COLS / 32;        // column blocks per wave
static_assert(PAIR_W % 16 == 12, "conflict-free patch row pitch");
static_assert(PAIR_COLS % 32 == 0 && PAIR_BR % 2 == 0 && PAIR_PW % 2 == 0, "windows in 2 x 2 blocks");

// The pool window (row py of the band, column px) of GEMM column col.
__device__ __forceinline__ void pair_window(int col, int &py, int &px) {
    const int g = col >> 4, w4 = (col >> 2) & 3;
    py = 2 * (g / (PAIR_PW / 2)) + (w4 >> 1);
    px = 2 * (g % (PAIR_PW / 2)) + (w4 & 1);
}

// conv1's finished value from its 9 inputs.
__device__ __forceinline__ float pair_conv1(const float *x, const float *w, float bias, bool has_bias,
                                            bool has_relu) {
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < 9; ++k) v = __builtin_fmaf(w[k], x[k], v);
    if (has_bias) v = v + bias;
    if (has_relu) v = relu_idiom(v);
    return v;
}

__global__ __launch_bounds__(256, 2) void conv_pair_kernel(SplitPair p, const u4 *w2_split) {
    constexpr int FM = 2, FN = PAIR_FN;
    __shared__ u4 patch[12 * PAIR_POS];
    __shared__ __attribute__((aligned(16))) float img[PAIR_IR * PAIR_W];
    const bool bias1 = p.flags1 & CAMEL_EPI_BIAS, relu1 = p.flags1 & CAMEL_EPI_RELU;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1, r16 = lane & 15, oct = lane >> 4;
    const int n = blockIdx.x / p.bands, band = blockIdx.x - n * p.bands;
    const int m0 = blockIdx.y * 64, PH = p.bands * PAIR_BR;
    const int Y0 = band * 2 * PAIR_BR; // first conv2 (and conv1) row of the band
    const float *xi = p.x + ((size_t)n * p.H + Y0) * PAIR_W;
    const int a_blocks = p.Co2 / 16;
    const u4 *a_src[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) a_src[i] = w2_split + (size_t)(m0 / 16 + wm * FM + i) * 192 + lane;
    u4 an[FM][3];
    auto load_a = [&](int tap) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q) an[i][q] = a_src[i][(size_t)tap * a_blocks * 192 + 64 * q];
    };
    load_a(0);
    // The band's input rows, 16 bytes per thread (zeros past the image: never
    // read by a valid output).
    if (tid < PAIR_IR * PAIR_W / 4) {
        const int r = Y0 + tid / (PAIR_W / 4);
        reinterpret_cast<f4 *>(img)[tid] =
            r < p.H ? reinterpret_cast<const f4 *>(xi)[tid] : f4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();
    const float *w1 = p.w1 + 8 * wave * 9;
#pragma unroll 1
    for (int q = lane; q < PAIR_POS; q += 64) {
        const int r = q / PAIR_W, c = min(q - r * PAIR_W, PAIR_OW1 - 1); // the pitch's last two repeat
        float xv[9], f[8];
#pragma unroll
        for (int k = 0; k < 9; ++k) xv[k] = img[(r + k / 3) * PAIR_W + c + k % 3];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            f[e] = pair_conv1(xv, w1 + 9 * e, bias1 ? p.b1[8 * wave + e] : 0.f, bias1, relu1);
        u4 d[3];
        split8(f, d);
#pragma unroll
        for (int h = 0; h < 3; ++h) patch[(h * 4 + wave) * PAIR_POS + q] = d[h];
    }
    __syncthreads();

    int at[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int col = (wn * FN + j) * 16 + r16, d = col & 3;
        int py, px;
        pair_window(col, py, px);
        at[j] = oct * PAIR_POS + (2 * py + (d >> 1)) * PAIR_W + 2 * px + (d & 1);
    }
    f4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    bf8 b[2][3], a[FM][3];
    f4 t[2][FM];
    auto fetch = [&](int j, int off, bf8 *d) {
#pragma unroll
        for (int q = 0; q < 3; ++q) d[q] = __builtin_bit_cast(bf8, patch[q * 4 * PAIR_POS + at[j] + off]);
    };
    fetch(0, 0, b[0]);
#pragma unroll 1
    for (int kh = 0; kh < 3; ++kh) {
#pragma unroll
        for (int kw = 0; kw < 3; ++kw) {
            const int off = kh * PAIR_W + kw, next = kw < 2 ? off + 1 : min(kh + 1, 2) * PAIR_W;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q) a[i][q] = __builtin_bit_cast(bf8, an[i][q]);
            load_a(min(3 * kh + kw + 1, 8));
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int u = (kw * FN + j) & 1;
                fetch((j + 1) % FN, j + 1 < FN ? off : next, b[u ^ 1]);
#pragma unroll
                for (int i = 0; i < FM; ++i) t[u][i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < PRODUCTS; ++q)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
                        t[u][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[u][PB[q]], a[i][PA[q]], t[u][i], 0,
                                                                          0, 0);
                if (j > 0)
#pragma unroll
                    for (int i = 0; i < FM; ++i) add_products(acc[i][j - 1], t[u ^ 1][i]);
#pragma unroll
                for (int r = 0; r < PRODUCTS * FM; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (r % FM == FM - 1 && r < 3 * FM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if (r >= FM) __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < FM; ++i) add_products(acc[i][FN - 1], t[(kw * FN + FN - 1) & 1][i]);
        }
    }

    SplitGemm g2{};
    SplitConv c2{};
    g2.A = p.w2;
    c2.C = c2.unit = PAIR_C1;
    c2.taps = 9;
    c2.w_packed = p.w2_packed;
    finish_sums<FM, FN, 2, 2>(
        acc, 0, 9 * PAIR_C1, oct,
        [&](int i, int k) { return conv_weight(g2, c2, m0 + (wm * FM + i) * 16 + r16, k); },
        [&](int j, int k) {
            const int col = (wn * FN + j) * 16 + r16, d = col & 3, tap = k / PAIR_C1, ch = k % PAIR_C1;
            int py, px;
            pair_window(col, py, px);
            const int r = 2 * py + (d >> 1) + tap / 3, c = 2 * px + (d & 1) + tap % 3;
            float xv[9];
            for (int e = 0; e < 9; ++e) xv[e] = img[(r + e / 3) * PAIR_W + c + e % 3];
            return pair_conv1(xv, p.w1 + 9 * ch, bias1 ? p.b1[ch] : 0.f, bias1, relu1);
        });
    // bias, relu, then the window's maximum: first, then strict '>'
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int row = m0 + (wm * FM + i) * 16 + r16;
        const float bias = (p.flags2 & CAMEL_EPI_BIAS) ? p.b2[row] : 0.f;
        float *out = p.y + ((size_t)n * p.Co2 + row) * PH * PAIR_PW + (size_t)band * PAIR_BR * PAIR_PW;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            int py, px;
            pair_window((wn * FN + j) * 16 + 4 * oct, py, px);
            f4 v = acc[i][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (p.flags2 & CAMEL_EPI_BIAS) v[e] = v[e] + bias;
                if (p.flags2 & CAMEL_EPI_RELU) v[e] = relu_idiom(v[e]);
            }
            float mx = v[0];
#pragma unroll
            for (int e = 1; e < 4; ++e)
                if (v[e] > mx) mx = v[e];
            out[py * PAIR_PW + px] = mx;
        }
    }
}

// (The conv kernels' first stage below k = 0 is stage 0 of the split weights.)
template <class T, int ASRC, class BSrc, int OUT>
__global__ __launch_bounds__(T::THREADS, 2) void split_gemm_kernel(SplitGemm g, SplitConv cv) {
    constexpr bool AT = ASRC == A_COLS;
    __shared__ u4 smem[T::LDS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = T::WK > 1 ? wave / T::GW : 0, w = wave - kg * T::GW;
    const int wm = w / T::WN, wn = w - wm * T::WN;
    const int r16 = lane & 15, oct = lane >> 4;
    const int tiles_m = (g.M + T::BM - 1) / T::BM, tiles_n = (g.N + T::BN - 1) / T::BN;
    // XCD x (work-groups are dispatched round-robin) takes a contiguous range
    // of (split, tile) positions, so that its L2 holds a compact block.
    const int nt = gridDim.x, nb = nt * gridDim.y;
    int bid = blockIdx.x + nt * blockIdx.y;
    if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    const int split = bid / nt;
    int tm, tn;
    split_tile_of(bid - split * nt, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * T::BM, n0 = tn * T::BN;
    // K in whole steps; a ragged one comes first, starting below k = 0.
    const int kpad = (T::SB - g.K % T::SB) % T::SB;
    const int ks0 = split * g.k_per_split - kpad, kend = min(g.K, ks0 + g.k_per_split);
    const int ns = (kend - ks0) / T::SB;
    const int kbeg = ks0 + kg * BK;
    u4 *const bufs = smem + kg * 2 * T::B_ST;

    // Rows and columns past the problem repeat the last one (never stored).
    const int mw = m0 + wm * T::FM * 16 + r16;
    const float *a_base = ASRC == A_ROWS ? g.A + (size_t)m0 * g.lda : g.A;
    uint32_t a_off[T::FM];
    const int a_blocks = (g.M + 15) / 16; // A_SPLIT
#pragma unroll
    for (int i = 0; i < T::FM; ++i) {
        if constexpr (ASRC == A_SPLIT) {
            a_off[i] = (uint32_t)min(m0 / 16 + wm * T::FM + i, a_blocks - 1) * 192u + lane;
            continue;
        }
        const int row = min(mw + 16 * i, g.M - 1);
        a_off[i] = AT ? (uint32_t)row * 4u + (uint32_t)(8 * oct) * (uint32_t)g.lda * 4u
                      : (uint32_t)(row - m0) * (uint32_t)g.lda * 4u + 32u * oct;
    }
    // A's stage at k0: 8 fp32 values a block, or (A_SPLIT) its three chunks.
    struct ARegs {
        float f[ASRC == A_SPLIT ? 1 : T::FM][8];
        u4 c[ASRC == A_SPLIT ? T::FM : 1][3];
    };
    auto load_a = [&](int k0, int i, ARegs &r) {
        if constexpr (ASRC == A_SPLIT) {
            const u4 *q = cv.w_split + (size_t)((k0 + cv.kpad) / BK) * a_blocks * 192 + a_off[i];
#pragma unroll
            for (int p = 0; p < 3; ++p) r.c[i][p] = q[64 * p];
        } else if constexpr (!AT) {
            const char *q = reinterpret_cast<const char *>(a_base + k0) + a_off[i];
            const f4 v0 = *reinterpret_cast<const f4u *>(q);
            const f4 v1 = *reinterpret_cast<const f4u *>(q + 16);
#pragma unroll
            for (int c = 0; c < 4; ++c) r.f[i][c] = v0[c], r.f[i][4 + c] = v1[c];
        } else {
            const char *q = reinterpret_cast<const char *>(a_base + (size_t)k0 * g.lda);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                r.f[i][j] = *reinterpret_cast<const float *>(q + a_off[i]);
                q += (size_t)g.lda * sizeof(float);
            }
        }
    };
    auto load_all_a = [&](int k0, ARegs &r) {
#pragma unroll
        for (int i = 0; i < T::FM; ++i) load_a(k0, i, r);
    };
    BSrc bsrc(g, cv);
    int b_slot[T::B_IT], b_oct[T::B_IT];
#pragma unroll
    for (int i = 0; i < T::B_IT; ++i) {
        const int wi = w + i * T::GW, c = (wi >> 2) * 64 + lane;
        b_oct[i] = wi & 3;
        b_slot[i] = b_oct[i] * T::BN + c;
        bsrc.column(g, cv, i, n0 + c);
    }
    auto load_b = [&](int k0, float (*f)[8]) {
#pragma unroll
        for (int i = 0; i < T::B_IT; ++i) bsrc.load(i, k0 + 8 * b_oct[i], f[i]);
    };
    auto store_b = [&](u4 *lds, float (*f)[8]) {
#pragma unroll
        for (int i = 0; i < T::B_IT; ++i) {
            u4 c[3];
            split8(f[i], c);
#pragma unroll
            for (int q = 0; q < 3; ++q) lds[q * 4 * T::BN + b_slot[i]] = c[q];
        }
    };
    bf8 a[T::FM][3];
    auto split_a = [&](const ARegs &r) {
#pragma unroll
        for (int i = 0; i < T::FM; ++i) {
            u4 c[3];
            if constexpr (ASRC == A_SPLIT) {
#pragma unroll
                for (int q = 0; q < 3; ++q) c[q] = r.c[i][q];
            } else {
                split8(r.f[i], c);
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) a[i][q] = __builtin_bit_cast(bf8, c[q]);
        }
    };
    // k of this group's stage s; past the end the last one again (in bounds,
    // never used)
    auto k_of = [&](int s) { return max(kbeg + min(s, ns - 1) * T::SB, 0); };

    f4 acc[T::FM][T::FN];
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
        for (int j = 0; j < T::FN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    ARegs ra;
    float rb[T::B_IT][8];
    if (kbeg >= 0) {
        load_all_a(kbeg, ra);
        load_b(kbeg, rb);
    } else {
        if constexpr (ASRC == A_SPLIT) load_all_a(kbeg, ra);
#pragma unroll
        for (int i = 0; i < (ASRC == A_SPLIT ? 0 : T::FM); ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = kbeg + 8 * oct + j;
                const size_t row = min(mw + 16 * i, g.M - 1);
                ra.f[i][j] = k >= 0 ? (AT ? g.A[(size_t)k * g.lda + row] : g.A[row * g.lda + k]) : 0.f;
            }
#pragma unroll
        for (int i = 0; i < T::B_IT; ++i) bsrc.load_ragged(i, kbeg + 8 * b_oct[i], rb[i]);
    }
    split_a(ra);
    store_b(bufs, rb);
    load_b(k_of(1), rb);
    load_all_a(k_of(1), ra);
    __syncthreads();
    const int b_rd = oct * T::BN + wn * T::FN * 16 + r16;
    bf8 b[2][3];
    // A wave of one block row runs its six products as three chains, so that no
    // MFMA waits for the one before; hi hi is one of its own, which the vector
    // ALU adds rounded.
    constexpr int NC = T::FM == 1 ? 3 : 1;
    f4 t[2][T::FM * NC];
    auto add_t = [&](int j) {
        if constexpr (NC == 3)
            add_products(acc[0][j], (t[j & 1][0] + t[j & 1][1]) + t[j & 1][2]);
        else
#pragma unroll
            for (int i = 0; i < T::FM; ++i) add_products(acc[i][j], t[j & 1][i]);
    };
    auto fetch = [&](const u4 *Bs, int j, bf8 *d) {
#pragma unroll
        for (int q = 0; q < 3; ++q)
            d[q] = __builtin_bit_cast(bf8, Bs[q * 4 * T::BN + b_rd + 16 * j]);
    };
    fetch(bufs, 0, b[0]);
    // SPREAD: the conversions of the next stage, a pair of values at a time,
    // over the columns, so that they run in the shadow of the MFMAs: B's pairs
    // in the first half (before the barrier column), A's in the second, each
    // item's next loads when its last pair is done (128 x 128 tiles: 128 x 4096
    // x 4096 in 8 splits 42.5 -> 36.5 us, 1000 x 3001 x 2047 99 -> 80).  The
    // 256 x 256 tile has no registers for A's converted next stage (9 spilled,
    // 536 -> 564 us at 4096^3): B's are converted together during one column,
    // A's after the last.
    constexpr bool SPREAD = T::FM * T::FN <= 16;
    constexpr int J_ST = SPREAD ? -1 : 2;
    constexpr int NB = 4 * T::B_IT, NA = ASRC == A_SPLIT ? 0 : 4 * T::FM;
    constexpr int B_COLS = NA ? T::FN / 2 : T::FN - 2, REST = T::FN - B_COLS;
    u4 cb[3], an[T::FM][3];
    for (int s = 0; s < ns; ++s) {
        const u4 *Bc = bufs + (s & 1) * T::B_ST;
        u4 *Bn = bufs + ((s + 1) & 1) * T::B_ST;
        const int k2 = k_of(s + 2);
#pragma unroll
        for (int j = 0; j < T::FN; ++j) {
            // (the last column's reads for the next stage come after the
            // barrier in the one before)
            fetch(j + 1 < T::FN ? Bc : Bn, (j + 1) % T::FN, b[(j + 1) & 1]);
#pragma unroll
            for (int i = 0; i < T::FM * NC; ++i) t[j & 1][i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < PRODUCTS; ++p)
#pragma unroll
                for (int i = 0; i < T::FM; ++i) {
                    f4 &c = t[j & 1][i + (NC == 1 ? 0 : p + 1 < PRODUCTS ? p % 2 : 2)];
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j & 1][PB[p]], a[i][PA[p]], c, 0, 0, 0);
                }
            if (j > 0) add_t(j - 1);
            if (j == J_ST) {
                store_b(Bn, rb);
                load_b(k2, rb);
            }
#pragma unroll
            for (int u = 0; u < (SPREAD ? NB : 0); ++u) {
                if (u * B_COLS / NB != j) continue;
                split_pair(rb[u / 4], u % 4, cb);
                if (u % 4 == 3) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) Bn[q * 4 * T::BN + b_slot[u / 4]] = cb[q];
                    bsrc.load(u / 4, k2 + 8 * b_oct[u / 4], rb[u / 4]);
                }
            }
#pragma unroll
            for (int u = 0; u < (SPREAD ? NA : 0); ++u) {
                if (B_COLS + u * REST / (NA ? NA : 1) != j) continue;
                split_pair(ra.f[u / 4], u % 4, an[u / 4]);
                if (u % 4 == 3) load_a(k2, u / 4, ra);
            }
            if (j == T::FN - 2) __syncthreads();
            // Operand reads between the first MFMAs, vector operations (the
            // adds of the column before, conversions) after each of the
            // others (masks: 0x8 MFMA, 0x100 LDS read, 0x2 VALU): 4096^3 580 ->
            // 570 us against the compiler's order.
            if constexpr (SPREAD) {
#pragma unroll
                for (int r = 0; r < PRODUCTS * T::FM; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (r % T::FM == T::FM - 1 && r < 3 * T::FM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if (r >= T::FM) __builtin_amdgcn_sched_group_barrier(0x002, (NC == 1 ? 2 : 3), 0);
                }
            } else if (j != J_ST) {
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, T::FM, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
#pragma unroll
                for (int r = 0; r < 2 * T::FM; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x008, T::FM, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (SPREAD && ASRC != A_SPLIT) {
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q) a[i][q] = __builtin_bit_cast(bf8, an[i][q]);
        } else {
            split_a(ra);
            load_all_a(k2, ra);
        }
        add_t(T::FN - 1);
    }

    if constexpr (T::WK > 1) {
        __syncthreads(); // the last operand reads
        f4 *red = reinterpret_cast<f4 *>(smem);
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
#pragma unroll
                for (int j = 0; j < T::FN; ++j)
                    red[(((kg - 1) * T::GW + w) * T::FM * T::FN + i * T::FN + j) * 64 + lane] = acc[i][j];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int q = 0; q < T::WK - 1; ++q)
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
#pragma unroll
                for (int j = 0; j < T::FN; ++j)
                    acc[i][j] += red[((q * T::GW + w) * T::FM * T::FN + i * T::FN + j) * 64 + lane];
    }
    const int nw = n0 + wn * T::FN * 16;
    finish_sums<T::FM, T::FN, 4, (ASRC == A_SPLIT ? 2 : T::FM * T::FN > 16 ? 4 : 8)>(
        acc, max(ks0, 0), kend, oct,
        [&](int i, int k) {
            const size_t m = min(mw + 16 * i, g.M - 1);
            if constexpr (ASRC == A_SPLIT) return conv_weight(g, cv, (int)m, k);
            return AT ? g.A[(size_t)k * g.lda + m] : g.A[m * g.lda + k];
        },
        [&](int j, int k) { return BSrc::at(g, cv, k, min(nw + 16 * j + r16, g.N - 1)); });
    if constexpr (OUT == OUT_MATRIX)
        store_matrix<T::FM, T::FN>(g, acc, split, mw, nw + 4 * oct);
    else
        store_conv<T::FM, T::FN, OUT == OUT_POOL>(g, cv, acc, split, mw, nw + 4 * oct);
}

// C = sum of the K splits' partials [split][M][N] in split order, then bias
// and relu; VEC: 4 columns per thread (N % 4 == 0, C 16-byte aligned).
template <bool VEC>
__global__ __launch_bounds__(256) void split_reduce_kernel(SplitGemm g, int splits) {
    constexpr int W = VEC ? 4 : 1;
    typedef float vec __attribute__((ext_vector_type(W)));
    const size_t total = (size_t)g.M * g.N, step = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total / W; q += step) {
        const size_t idx = q * W;
        vec s = *reinterpret_cast<const vec *>(g.partial + idx);
        for (int z0 = 1; z0 < splits; z0 += 8) {
            vec t[8]; // up to 8 loads in flight
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (z0 + u < splits) t[u] = *reinterpret_cast<const vec *>(g.partial + (z0 + u) * total + idx);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (z0 + u < splits) s = s + t[u];
        }
        const int row = (int)(idx / g.N), col = (int)(idx - (size_t)row * g.N);
#pragma unroll
        for (int v = 0; v < W; ++v) {
            float x = s[v];
            if (g.flags & CAMEL_EPI_BIAS) x = x + g.bias[col + v];
            if (g.flags & CAMEL_EPI_RELU) x = relu_idiom(x);
            s[v] = x;
        }
        *reinterpret_cast<vec *>(g.C + (size_t)row * g.ldc + col) = s;
    }
}

// The splits' partials of a convolution, in split order, then its epilogue; a
// thread per 4 columns of a channel.
template <bool POOL>
__global__ __launch_bounds__(256) void split_conv_reduce_kernel(SplitGemm g, SplitConv c, int splits) {
    const int quads = (g.N + 3) / 4;
    const size_t total = (size_t)g.M * g.N;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < (size_t)g.M * quads;
         q += (size_t)gridDim.x * blockDim.x) {
        const int row = (int)(q / quads), n = 4 * (int)(q - (size_t)row * quads);
        const float *src = g.partial + (size_t)row * g.N + n;
        const bool whole = n + 3 < g.N;
        f4 s = {0.f, 0.f, 0.f, 0.f};
        for (int z0 = 0; z0 < splits; z0 += 8) {
            f4 t[8]; // up to 8 loads in flight
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (z0 + u >= splits) continue;
                const float *p = src + (z0 + u) * total;
                if (whole)
                    t[u] = *reinterpret_cast<const f4u *>(p);
                else
                    for (int v = 0; v < 4; ++v) t[u][v] = n + v < g.N ? p[v] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (z0 + u < splits) s = z0 + u ? s + t[u] : t[u];
        }
        store_conv_quad<POOL>(g, c, s, row, n, ConvColumn(n, POOL ? 4 * c.PP : c.P),
                              (g.flags & CAMEL_EPI_BIAS) ? g.bias[row] : 0.f);
    }
}

// 256 x 256: 8 waves of 32 x 256.  128 x 128 and 64 x 64: 8 waves, 4 of 32 x 128
// or 16 x 64 on each of two k groups (64 x 64 with the six products of a block
// as two MFMA chains: 21.1 -> 20.2 us at 1024^3, 14.1 -> 14.5 at 68 x 192 x 8021;
// as three, hi hi by itself: 1500^3 66.7 -> 68.0; four k groups of two 32 x 64
// waves: 300 x 3000 x 800 18.8 -> 20.6).
using T256 = STile<2, 16, 8, 1, 1>;
using T128 = STile<2, 8, 4, 1, 2>;
using T64 = STile<1, 4, 4, 1, 2>;

// Convolutions: 4 waves of 32 channels x 128 pixels (two work-groups share a
// CU, so one's first loads and stores overlap the other's products), 2 x 2 of
// 32 x 64 for up to 64 channels.
using C128 = STile<2, 8, 4, 1, 1>;
using C64 = STile<2, 4, 2, 2, 1>;

// K per split and the splits a request really gives: whole steps, none empty.
template <class T> void split_k(int64_t K, int splits, int &k_per_split, int &used) {
    const int steps = (int)((K + T::SB - 1) / T::SB);
    const int per = (steps + splits - 1) / splits;
    k_per_split = per * T::SB;
    used = (steps + per - 1) / per;
}

template <class T> int launch(SplitGemm g, bool a_trans, int splits) {
    const unsigned tiles = (unsigned)(((g.M + T::BM - 1) / T::BM) * ((g.N + T::BN - 1) / T::BN));
    int used = 1;
    split_k<T>(g.K, splits, g.k_per_split, used);
    if (used == 1) g.partial = nullptr;
    const dim3 grid(tiles, (unsigned)used), block(T::THREADS);
    if (a_trans)
        hipLaunchKernelGGL((split_gemm_kernel<T, A_COLS, MatrixB<T>, OUT_MATRIX>), grid, block, 0, stream(), g,
                           SplitConv{});
    else
        hipLaunchKernelGGL((split_gemm_kernel<T, A_ROWS, MatrixB<T>, OUT_MATRIX>), grid, block, 0, stream(), g,
                           SplitConv{});
    CAMEL_RETURN_IF(check_launch("split_gemm_kernel"));
    if (used > 1) {
        const bool vec = g.N % 4 == 0 && ((uintptr_t)g.C & 15) == 0;
        const int64_t items = (int64_t)g.M * g.N / (vec ? 4 : 1);
        if (vec)
            hipLaunchKernelGGL(split_reduce_kernel<true>, dim3(grid_for(items, 256)), dim3(256), 0, stream(), g, used);
        else
            hipLaunchKernelGGL(split_reduce_kernel<false>, dim3(grid_for(items, 256)), dim3(256), 0, stream(), g, used);
        CAMEL_RETURN_IF(check_launch("split_reduce_kernel"));
    }
    return CAMEL_HIP_OK;
}

template <class T> int64_t conv_tiles(const SplitGemm &g) {
    return ((int64_t)(g.M + T::BM - 1) / T::BM) * ((g.N + T::BN - 1) / T::BN);
}

// K splits of a convolution: few tiles with many stages (small batches) leave
// the chip idle.  Estimates from measured calls, in us: a stage takes 1.9 alone
// on its CU and 3.2 beside a second work-group, a work-group 6 besides, the
// partials 3 and their traffic.  (1 x 128 x 14 x 14 -> 256 3x3, 4 tiles of 36
// stages: unsplit 80.)
int conv_splits(const SplitGemm &g, int64_t tiles, int cus) {
    const int stages = (g.K + BK - 1) / BK;
    // (Up to 9 stages stay unsplit: the fused pair of first layers, which sums 9
    // stages in one go, has to match.)
    if (stages <= 9) return 1;
    int best = 1;
    double best_t = 1e30;
    for (int want = 1; want <= 16; ++want) {
        const int per = (stages + want - 1) / want, used = (stages + per - 1) / per;
        const size_t bytes = used > 1 ? (size_t)used * g.M * g.N * sizeof(float) : 0;
        if (used != want || (want > 1 && per < 3) || bytes > CAMEL_HIP_NOALLOC_SCRATCH_BYTES) continue;
        const int64_t wgs = tiles * used;
        const double t = (wgs <= cus ? 6 + 1.9 * per : (double)((wgs + 2 * cus - 1) / (2 * cus)) * (6 + 3.2 * per)) +
                         (used > 1 ? 3 + 2.0 * bytes / 6e6 : 0);
        if (t < best_t) {
            best_t = t;
            best = used;
        }
    }
    return best;
}

template <class T, bool QUADS> int launch_patch(const SplitGemm &g, const SplitConv &c, bool pool) {
    const int64_t per = pool ? 4 * c.PP : c.P;
    const int64_t tiles_n =
        c.per_image ? g.N / per * ((per + T::BN - 1) / T::BN) : ((int64_t)g.N + T::BN - 1) / T::BN;
    const dim3 grid((unsigned)((g.M + T::BM - 1) / T::BM * tiles_n)), block(T::THREADS);
    if (pool)
        hipLaunchKernelGGL((conv_patch_kernel<T, QUADS, true>), grid, block, 0, stream(), g, c);
    else
        hipLaunchKernelGGL((conv_patch_kernel<T, QUADS, false>), grid, block, 0, stream(), g, c);
    return check_launch("conv_patch_kernel");
}

// K in runs of 32 channels, which the patch kernel needs: stride 1, several taps,
// channels that fill blocks of 32 (at most 1/8 padding) and 128-pixel tiles for
// 3/4 of the CUs without K splits.  Decided on the geometry alone, so
// that all layouts and the pooled form sum in the same order.
bool conv_blocked(const SplitConv &c, int64_t pixels, int64_t Co, int cus) {
    const int64_t blocks = (c.C + BK - 1) / BK, tile_m = Co <= 64 ? 64 : 128;
    return c.stride == 1 && c.KH * c.KW >= 4 && blocks * BK * 8 <= (int64_t)c.C * 9 &&
           (pixels + 127) / 128 * ((Co + tile_m - 1) / tile_m) * 4 >= 3 * cus;
}

// Positions a patch needs for any tile of 128 columns, 0 if over PATCH:
// `wraps` row ends (pool order: ends of two-row strips of windows) each add
// the padding between rows, the taps reach further down, and a tile across
// images adds the rows between them -- or tiles stay within images, where that
// wastes at most 1/8 of their columns.
int patch_positions(const SplitConv &c, int64_t images, bool pool, int &per_image) {
    constexpr int64_t BN = 128;
    const int64_t Wp = c.W + 2 * c.pad, OW = c.OW, PW = c.PW, per = pool ? 4 * c.PP : c.P;
    if ((images * (int64_t)(c.H + 2 * c.pad) + 1) * Wp + PATCH >= INT32_MAX) return 0;
    const int64_t reach = (c.KH - 1) * Wp + c.KW;
    const int64_t inside =
        reach + (pool ? (2 * ((BN / 4 + PW - 2) / PW) + 1) * Wp + OW : BN + (BN + OW - 2) / OW * (Wp - OW));
    const int64_t across = inside + (BN + per - 2) / per * c.KH * Wp;
    per_image = across > PATCH;
    if (!per_image) return (int)across;
    return inside <= PATCH && (per + BN - 1) / BN * BN * 8 <= per * 9 ? (int)inside : 0;
}

template <class T, bool QUADS>
int launch_conv(SplitGemm g, const SplitConv &c, bool pool, int splits, float *partial) {
    int used = 1;
    split_k<T>(g.K, splits, g.k_per_split, used);
    g.partial = used > 1 ? partial : nullptr;
    const dim3 grid((unsigned)conv_tiles<T>(g), (unsigned)used), block(T::THREADS);
    if (pool)
        hipLaunchKernelGGL((split_gemm_kernel<T, A_SPLIT, ConvB<T, QUADS, true>, OUT_POOL>), grid, block, 0,
                           stream(), g, c);
    else
        hipLaunchKernelGGL((split_gemm_kernel<T, A_SPLIT, ConvB<T, QUADS, false>, OUT_CONV>), grid, block, 0,
                           stream(), g, c);
    CAMEL_RETURN_IF(check_launch("split_gemm_kernel (conv)"));
    if (used > 1) {
        const dim3 rgrid(grid_for((int64_t)g.M * ((g.N + 3) / 4), 256));
        if (pool)
            hipLaunchKernelGGL(split_conv_reduce_kernel<true>, rgrid, dim3(256), 0, stream(), g, c, used);
        else
            hipLaunchKernelGGL(split_conv_reduce_kernel<false>, rgrid, dim3(256), 0, stream(), g, c, used);
        CAMEL_RETURN_IF(check_launch("split_conv_reduce_kernel"));
    }
    return CAMEL_HIP_OK;
}

} // namespace

// Microseconds of a product on the fp32 MFMA kernels, as their plan chooses the
// tile (256 and 128 where these fill the CUs, else 64, or 32 where 64 covers
// less than half of them) and the K splits.  Constants: least squares over 260
// measured shapes of 64..7900 rows and columns, k 64..7400 (7% rms).
static double fp32_us(int64_t M, int64_t N, int64_t K, bool at, bool ua, bool ub, int cus) {
    auto up = [](int64_t v, int64_t m) { return (v + m - 1) / m; };
    auto tiles = [&](int64_t edge) { return up(M, edge) * up(N, edge); };
    const double out = 4.0 * M * N / 5e6; // C's bytes
    const bool plain = !at && !ua && !ub;
    if (tiles(256) >= cus)
        return up(tiles(256), cus) * up(K, 64) * (plain ? 14.7 : 16.0) + out;
    if (tiles(128) >= cus)
        return 4 + up(tiles(128), cus) * up(K, 64) * (plain ? 3.7 : 4.2) + 2 * out;
    auto splits_of = [&](int64_t t) {
        return std::max<int64_t>(1, std::min<int64_t>(up(cus, t), std::min<int64_t>(K / 256, 64)));
    };
    int64_t edge = 64, splits = tiles(64) >= cus ? 1 : splits_of(tiles(64));
    if (tiles(64) * splits * 2 < cus) {
        edge = 32;
        splits = splits_of(tiles(32));
    }
    const int64_t wgs = tiles(edge) * splits, steps = up(up(K, 64), splits), rounds = up(wgs, cus);
    const double part = splits > 1 ? 8.0 * splits * M * N / 6e6 : 0.0; // partials, written and read
    if (edge == 32)
        return 2.6 + steps * std::max(1.0, (double)wgs / cus) * (0.65 + 0.2 * at + 0.2 * ub) +
               (plain ? 0 : 1.3) + (splits > 1 ? 2.5 : 0.0) + 3 * part + 2.5 * out;
    return 4 + steps * rounds * ((plain ? 1.08 : rounds == 1 ? 1.5 : 1.12) + 0.2 * at + 0.2 * ua + 0.2 * ub) +
           (splits > 1 ? 0.9 : 0.0) + 2.3 * part + 1.4 * out;
}

// The rule: the (tile, K splits) of the shortest estimate, if it is below 0.9 of
// the fp32 kernels' (the margin covers the fits' error).  A work-group takes a
// fixed time (prologue, tail, launch) plus one per step; partials are written
// and read at about 6 TB/s after a reduce launch.  128- and 256-edge tiles have
// a CU to themselves and run in whole rounds; two 64-edge ones share one.
// Constants: least squares over 1500 measured (shape, tile, splits) (6% rms).
// Over those shapes the choice is 1.21x the fp32 kernels and 2% behind the best
// one.  Sizes enter as whole 64 x 64 tiles, so that a row gives the same bits
// whether or not its tile is full.  Split / fp32, us: 4096^3 540 / 952, 1000 x 3001 x
// 2047 80 / 162, 1024 x 1024 x 8192 transposed 97 / 193, 2048^3 89 / 131, 1500^3 67 /
// 79, 768^3 15.5 / 23.3, 300 x 3000 x 800 17.5 / 26.3, 68 x 192 x 8021 transposed 13.9 /
// 16.8; and 1024^3 20.5 / 20.5, 512^3 11.5 / 11.6, 256^3 8.1 / 5.0, which stay on the
// fp32 kernels: one round of tiles whose loads are DMA, where a 64 x 64 split tile
// converts each value 16 times over, and a classifier head joins the fp32 tile's
// epilogue.
SplitPlan split_gemm_plan(int64_t M, int64_t N, int64_t K, bool a_trans, bool a_unaligned, bool b_unaligned,
                          int64_t lda, int64_t ldb, int cus) {
    SplitPlan best;
    if (K < 64 || lda >= (1 << 21) || ldb >= (1 << 28) || M > INT32_MAX / 512 || N > INT32_MAX / 512)
        return best;
    auto up = [](int64_t v, int64_t m) { return (v + m - 1) / m; };
    const size_t c_bytes = (size_t)M * N * sizeof(float);
    M = up(M, 64) * 64;
    N = up(N, 64) * 64;
    double limit = 0.9 * fp32_us(M, N, K, a_trans, a_unaligned, b_unaligned, cus);
    const double out = 4.0 * M * N / 5e6;
    // (`least`: the estimate of one step; small products, whose calls are bound by
    // the host, end here)
    auto consider = [&](SplitTile tile, int edge, int sb, double least, auto &&estimate) {
        if (limit <= least) return;
        const int64_t tiles = up(M, edge) * up(N, edge);
        if (tiles > INT32_MAX / 64) return;
        for (int want : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
            const int64_t steps = up(K, sb), per = up(steps, want), used = up(steps, per);
            const size_t bytes = used > 1 ? (size_t)used * M * N * sizeof(float) : 0;
            if (used != want || bytes > CAMEL_HIP_NOALLOC_SCRATCH_BYTES || (want > 1 && per < 4)) continue;
            const double t = estimate(tiles * used, (double)per, used > 1, 2.0 * bytes / 6e6);
            if (t < limit) {
                limit = t;
                best = {tile, (int)used, used > 1 ? (size_t)used * c_bytes : 0};
            }
        }
    };
    consider(SplitTile::T256, 256, T256::SB, 8.5 + 4.1, [&](int64_t wgs, double per, bool parts, double bytes) {
        return up(wgs, cus) * (8.5 + 4.1 * per) + (parts ? 3.6 : 0.0) + 0.9 * bytes;
    });
    consider(SplitTile::T128, 128, T128::SB, 8.9 + 2.06, [&](int64_t wgs, double per, bool parts, double bytes) {
        return up(wgs, cus) * (8.9 + 2.06 * per) + (parts ? 3.6 : 0.0) + 0.9 * bytes + 1.1 * out;
    });
    consider(SplitTile::T64, 64, T64::SB, 4.4 + 0.88, [&](int64_t wgs, double per, bool parts, double bytes) {
        const double share = wgs <= cus ? 1.0 : std::max(1.6, 0.15 + (double)wgs / cus);
        return 4.4 + per * share * (0.88 + 0.18 * a_trans) + (parts ? 2.7 : 0.0) + 1.55 * bytes + 2.5 * out;
    });
    return best;
}

int split_gemm(SplitGemm g, bool a_trans, const SplitPlan &plan, float *partial) {
    g.partial = partial;
    if (plan.tile == SplitTile::T256) return launch<T256>(g, a_trans, plan.splits);
    if (plan.tile == SplitTile::T128) return launch<T128>(g, a_trans, plan.splits);
    return launch<T64>(g, a_trans, plan.splits);
}

// Whether the fp32 kernels run a convolution of few stages faster: up to 9 stages
// there are no K splits here, and the split weights are a launch of their own.
// Microseconds up to two rounds of tiles (a tile: 128 pixels by 64 channels, or
// 128 beyond 64 channels), from 430 measured calls; the weights' reorder, which a
// caller with packed weights saves, counts half.  fp32 / split, packed weights:
// 64 -> 64 1x1 at 8 x 28 x 28 7.2 / 11.1, 32 -> 64 3x3 at 8 x 28 x 28 16.9 / 20.4; and
// unpacked 10 -> 40 3x3 at 8 x 60 x 60 14.9 / 16.4, 16 -> 32 3x3 17.3 / 16.0.  Up to
// 16 channels the two differ by less than 10% either way, and beyond 64 the
// fp32 tiles of few pixels take longer (128 -> 128 1x1 at 196 pixels 22.9 /
// 17.5) but for 2 stages: those stay split, and so do geometries of the patch
// kernel's order and of the fused pair.
static bool fp32_conv_faster(const SplitConv &c, int64_t pixels, int64_t Co, int cus) {
    const int taps = c.KH * c.KW, K = c.C * taps, stages = ((c.C + 7) / 8 * 8 * taps + BK - 1) / BK;
    const bool small = Co <= 64, nhwc = c.C % 16 == 0;
    if (stages > (small ? 9 : 2) || Co <= 16 || Co > 128 || (!nhwc && !small) || conv_blocked(c, pixels, Co, cus))
        return false;
    if (c.C == PAIR_C1 && c.KH == 3 && c.KW == 3 && c.stride == 1 && c.pad == 0 && c.W == PAIR_OW1) return false;
    const int64_t tiles = (pixels + 127) / 128, rounds = (tiles + cus - 1) / cus;
    if (rounds > 2) return false;
    const double round = !nhwc ? 6.4 + 0.065 * K : small ? 2.8 + (c.C % 32 ? 0.07 : 0.0427) * K : 3.8 + 0.081 * K;
    const double fp32 = 1.6 + round * (rounds > 1 ? (nhwc ? 1.8 : 1.45) : 1.0) + (nhwc ? 1.1 : 0.0);
    const double split = (small ? 8.7 + 1.28 * stages : 11 + 1.65 * stages) + (c.C % 8 ? 1.2 : 0.0) +
                         (rounds > 1 ? (2.5 + 0.27 * stages) * (small ? 1.0 : 1.5) : 0.0);
    return fp32 < 0.97 * split;
}

bool split_conv_serves(const SplitConv &c, int64_t N, int64_t pixels, int64_t Co, int cus) {
    const int64_t C8 = (c.C + 7) / 8 * 8, taps = (int64_t)c.KH * c.KW, K = C8 * taps;
    // 32 taps in a lane's mask; the divisions by C8 and KW and the buffer's
    // offsets (x, the reach of the first window, padded channels) stay exact;
    // channels padded by at most 1.6
    return c.C >= 5 && taps <= 32 && K >= 64 && K < 65536 && Co >= 16 &&
           4.0 * ((double)N * c.H * c.W + 2.0 * c.pad * (c.W + 1.0)) * C8 < (double)(1 << 30) &&
           !fp32_conv_faster(c, pixels, Co, cus);
}

SplitConvPlan split_conv_plan(const SplitGemm &g, const SplitConv &c, bool pool, int cus) {
    SplitConvPlan p;
    if (conv_blocked(c, g.N, g.M, cus)) {
        p.blocked = 1;
        p.patch = patch_positions(c, g.N / c.P, pool, p.per_image);
        p.weight_bytes = (size_t)((c.C + BK - 1) / BK) * c.KH * c.KW * ((g.M + 15) / 16) * 3072;
        return p;
    }
    p.splits = conv_splits(g, g.M <= 64 ? conv_tiles<C64>(g) : conv_tiles<C128>(g), cus);
    p.weight_bytes = (size_t)((g.K + BK - 1) / BK) * ((g.M + 15) / 16) * 3072;
    p.partial_bytes = p.splits > 1 ? (size_t)p.splits * g.M * g.N * sizeof(float) : 0;
    return p;
}

int split_conv(SplitGemm g, SplitConv c, bool quads, bool pool, const SplitConvPlan &plan, void *scratch) {
    if (pool) g.N = g.N / c.P * c.PP * 4;
    c.shift = c.pad * (c.W + 1) * c.pxs;
    c.patch = plan.patch;
    c.per_image = plan.per_image;
    c.taps = c.KH * c.KW;
    c.unit = plan.blocked ? BK : (c.C + 7) / 8 * 8;
    c.mul_unit = (uint32_t)(((uint64_t)1 << 32) / c.unit + 1); // (unit >= 8, k < 65536)
    c.mul_kw = tap_mul(c.KW);
    c.mul_taps = tap_mul(c.taps);
    if (plan.blocked) g.K = (c.C + BK - 1) / BK * c.taps * BK;
    const int stages = (g.K + BK - 1) / BK;
    c.kpad = stages * BK - g.K;
    c.w_split = static_cast<const u4 *>(scratch);
    float *partial = reinterpret_cast<float *>(static_cast<char *>(scratch) + plan.weight_bytes);
    hipLaunchKernelGGL(split_weights_kernel, dim3(stages, (g.M + 15) / 16), dim3(64), 0, stream(), g, c,
                       static_cast<u4 *>(scratch));
    CAMEL_RETURN_IF(check_launch("split_weights_kernel"));
    if (plan.patch) {
        g.partial = nullptr;
        c.shift = 0;
        c.bytes = (uint32_t)((int64_t)(pool ? g.N / (4 * c.PP) : g.N / c.P) * c.CHW * 4);
        if (g.M <= 64)
            return quads ? launch_patch<PatchTile<2, 4, 2, 2>, true>(g, c, pool)
                         : launch_patch<PatchTile<2, 4, 2, 2>, false>(g, c, pool);
        return quads ? launch_patch<PatchTile<2, 8, 4, 1>, true>(g, c, pool)
                     : launch_patch<PatchTile<2, 8, 4, 1>, false>(g, c, pool);
    }
    if (g.M <= 64)
        return quads ? launch_conv<C64, true>(g, c, pool, plan.splits, partial)
                     : launch_conv<C64, false>(g, c, pool, plan.splits, partial);
    return quads ? launch_conv<C128, true>(g, c, pool, plan.splits, partial)
                 : launch_conv<C128, false>(g, c, pool, plan.splits, partial);
}

bool split_pair_serves(int64_t H, int64_t W, int64_t C1, int64_t Co2) {
    return W == PAIR_W && C1 == PAIR_C1 && Co2 > 0 && Co2 % 64 == 0 && H >= 6 && (H - 4) % (2 * PAIR_BR) == 0;
}

size_t split_pair_bytes(int64_t Co2) { return (size_t)9 * (Co2 / 16) * 3072; }

int split_pair(SplitPair p, int N, void *scratch) {
    SplitGemm g{};
    SplitConv c{};
    g.A = p.w2;
    g.M = p.Co2;
    g.K = 9 * PAIR_C1;
    c.C = c.unit = PAIR_C1;
    c.taps = 9;
    c.w_packed = p.w2_packed;
    u4 *w2 = static_cast<u4 *>(scratch);
    hipLaunchKernelGGL(split_weights_kernel, dim3(9, p.Co2 / 16), dim3(64), 0, stream(), g, c, w2);
    CAMEL_RETURN_IF(check_launch("split_weights_kernel"));
    p.bands = (p.H - 4) / 2 / PAIR_BR;
    hipLaunchKernelGGL(conv_pair_kernel, dim3((unsigned)(N * p.bands), (unsigned)(p.Co2 / 64)), dim3(256), 0,
                       stream(), p, w2);
    return check_launch("conv_pair_kernel");
}

} // namespace camel_hip
