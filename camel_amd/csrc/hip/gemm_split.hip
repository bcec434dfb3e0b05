// fp32 GEMM on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16), which run 16
// times the fp32 MFMA rate.
//
// Every fp32 operand x is taken as hi + mid + lo, three bf16 values: hi = x
// rounded to nearest, mid = x - hi cut to 8 bits, lo = the rest.  24
// significant bits make three 8-bit parts, so the sum is x exactly (|x| >=
// 2^-100 and below the bf16 maximum; see below).  A product of two such
// operands is the six part products down to 2^-18 of it -- hi hi, hi mid, mid
// hi, mid mid, hi lo, lo hi -- each exact in fp32; the three dropped ones are
// at most 2^-25 of the product, below the rounding of an fp32 product.
//
// Sums: the 6 MFMAs of a 16 x 16 block and 32 k start from zero, smallest
// products first, and their sum is added to the block's fp32 accumulator on
// the vector ALU (round to nearest).  An accumulator is rounded once per 32 k:
// error against fp64 at 4096^3, U(-1, 1): 2.1e-7 (2-norm), against 1.1e-6 for
// the fp32 MFMA chain, which rounds every 2 k.  (The 6 MFMAs on the
// accumulator itself: 1.03e-6, 4% faster.)
//
// Operands outside the exact range, tile by tile: the converting lanes keep
// the smallest nonzero |hi| (two packed 16-bit operations per pair), and a
// value that is infinite, NaN or beyond the bf16 maximum makes its outputs
// non-finite (its mid part is).  A tile that saw |x| < 2^-100 or holds a
// non-finite sum is computed again in fp32 MFMA, so special values and the
// ends of the range give what they give in fp32.
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
typedef unsigned short us2 __attribute__((ext_vector_type(2)));

constexpr int BK = 32;     // k per stage: one 16x16x32 MFMA
constexpr int GROUP_M = 4; // tile rows per group of the XCD-aware order

// 2 |hi| - 1 as 16-bit integers of a bf16 below 2^-100 (zero gives 0xffff).
// From there on lo's last bit is at least 2^-123, inside the bf16 range.
constexpr unsigned short TINY = (27 << 8) - 1;

// The upper halves of two floats, x0 in the lower half.
__device__ __forceinline__ uint32_t upper_pair(float x0, float x1) {
    return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);
}
__device__ __forceinline__ float upper(float x) {
    return __uint_as_float(__float_as_uint(x) & 0xffff0000u);
}

// f[0..7] -> three chunks of 8 bf16 (hi, mid, lo); tiny: running minimum of
// 2 |hi| - 1.  (v_dot2_f32_bf16 with a -1 forms x - hi in one operation
// instead of two, but its results may not be read for 3 wait states: 4096^3
// 557 -> 578 us.)
__device__ __forceinline__ void split8(const float *f, u4 *out, us2 &tiny) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float x0 = f[2 * c], x1 = f[2 * c + 1];
        const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){x0, x1}, bf2));
        us2 twice;
        asm("v_pk_mad_u16 %0, %1, 2, -1 op_sel_hi:[1,0,0]" : "=v"(twice) : "v"(h));
        tiny = __builtin_elementwise_min(tiny, twice);
        x0 = x0 - __uint_as_float(h << 16);
        x1 = x1 - __uint_as_float(h & 0xffff0000u);
        out[0][c] = h;
        out[1][c] = upper_pair(x0, x1);
        out[2][c] = upper_pair(x0 - upper(x0), x1 - upper(x1));
    }
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

// B as a row-major matrix: lane = column, octet o of a stage = rows 8 o .. +7,
// 256 contiguous bytes of a row per load.
template <class T> struct MatrixB {
    const float *base;
    int ld;
    uint32_t off[T::B_IT];
    __device__ __forceinline__ MatrixB(const SplitGemm &g) : base(g.B), ld(g.ldb) {}
    __device__ __forceinline__ void column(const SplitGemm &g, int i, int n) {
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
    __device__ __forceinline__ static float at(const SplitGemm &g, int k, int n) {
        return g.B[(size_t)k * g.ldb + n];
    }
};

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

template <class T, bool AT>
__global__ __launch_bounds__(T::THREADS, 2) void split_gemm_kernel(SplitGemm g) {
    using BSrc = MatrixB<T>;
    __shared__ u4 smem[T::LDS + 1];
    uint32_t *const flag = reinterpret_cast<uint32_t *>(smem + T::LDS);
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
    if (tid == 0) *flag = 0;

    // Rows and columns past the problem repeat the last one (never stored).
    const int mw = m0 + wm * T::FM * 16 + r16;
    const float *a_base = AT ? g.A : g.A + (size_t)m0 * g.lda;
    uint32_t a_off[T::FM];
#pragma unroll
    for (int i = 0; i < T::FM; ++i) {
        const int row = min(mw + 16 * i, g.M - 1);
        a_off[i] = AT ? (uint32_t)row * 4u + (uint32_t)(8 * oct) * (uint32_t)g.lda * 4u
                      : (uint32_t)(row - m0) * (uint32_t)g.lda * 4u + 32u * oct;
    }
    auto load_a = [&](int k0, float (*f)[8]) {
#pragma unroll
        for (int i = 0; i < T::FM; ++i) {
            if constexpr (!AT) {
                const char *q = reinterpret_cast<const char *>(a_base + k0) + a_off[i];
                const f4 v0 = *reinterpret_cast<const f4u *>(q);
                const f4 v1 = *reinterpret_cast<const f4u *>(q + 16);
#pragma unroll
                for (int c = 0; c < 4; ++c) f[i][c] = v0[c], f[i][4 + c] = v1[c];
            } else {
                const char *q = reinterpret_cast<const char *>(a_base + (size_t)k0 * g.lda);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    f[i][j] = *reinterpret_cast<const float *>(q + a_off[i]);
                    q += (size_t)g.lda * sizeof(float);
                }
            }
        }
    };
    BSrc bsrc(g);
    int b_slot[T::B_IT], b_oct[T::B_IT];
#pragma unroll
    for (int i = 0; i < T::B_IT; ++i) {
        const int wi = w + i * T::GW, c = (wi >> 2) * 64 + lane;
        b_oct[i] = wi & 3;
        b_slot[i] = b_oct[i] * T::BN + c;
        bsrc.column(g, i, n0 + c);
    }
    auto load_b = [&](int k0, float (*f)[8]) {
#pragma unroll
        for (int i = 0; i < T::B_IT; ++i) bsrc.load(i, k0 + 8 * b_oct[i], f[i]);
    };
    us2 tiny = {0xffff, 0xffff};
    auto store_b = [&](u4 *lds, float (*f)[8]) {
#pragma unroll
        for (int i = 0; i < T::B_IT; ++i) {
            u4 c[3];
            split8(f[i], c, tiny);
#pragma unroll
            for (int q = 0; q < 3; ++q) lds[q * 4 * T::BN + b_slot[i]] = c[q];
        }
    };
    bf8 a[T::FM][3];
    auto split_a = [&](float (*f)[8]) {
#pragma unroll
        for (int i = 0; i < T::FM; ++i) {
            u4 c[3];
            split8(f[i], c, tiny);
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
    float ra[T::FM][8], rb[T::B_IT][8];
    if (kbeg >= 0) {
        load_a(kbeg, ra);
        load_b(kbeg, rb);
    } else {
#pragma unroll
        for (int i = 0; i < T::FM; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = kbeg + 8 * oct + j;
                const size_t row = min(mw + 16 * i, g.M - 1);
                ra[i][j] = k >= 0 ? (AT ? g.A[(size_t)k * g.lda + row] : g.A[row * g.lda + k]) : 0.f;
            }
#pragma unroll
        for (int i = 0; i < T::B_IT; ++i) bsrc.load_ragged(i, kbeg + 8 * b_oct[i], rb[i]);
    }
    split_a(ra);
    store_b(bufs, rb);
    load_b(k_of(1), rb);
    load_a(k_of(1), ra);
    __syncthreads();
    const int b_rd = oct * T::BN + wn * T::FN * 16 + r16;
    bf8 b[2][3];
    f4 t[2][T::FM];
    auto fetch = [&](const u4 *Bs, int j, bf8 *d) {
#pragma unroll
        for (int q = 0; q < 3; ++q)
            d[q] = __builtin_bit_cast(bf8, Bs[q * 4 * T::BN + b_rd + 16 * j]);
    };
    fetch(bufs, 0, b[0]);
    // part products, smallest first: (lo hi), (hi lo), (mid mid), (mid hi),
    // (hi mid), (hi hi)
    constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
    constexpr int J_ST = T::FN > 8 ? 2 : 0; // column during which B's next stage is stored
    for (int s = 0; s < ns; ++s) {
        const u4 *Bc = bufs + (s & 1) * T::B_ST;
        u4 *Bn = bufs + ((s + 1) & 1) * T::B_ST;
#pragma unroll
        for (int j = 0; j < T::FN; ++j) {
            // (the last column's reads for the next stage come after the
            // barrier in the one before)
            fetch(j + 1 < T::FN ? Bc : Bn, (j + 1) % T::FN, b[(j + 1) & 1]);
#pragma unroll
            for (int i = 0; i < T::FM; ++i) t[j & 1][i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < 6; ++p)
#pragma unroll
                for (int i = 0; i < T::FM; ++i)
                    t[j & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j & 1][PB[p]], a[i][PA[p]],
                                                                          t[j & 1][i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
                if (j > 0) acc[i][j - 1] += t[(j + 1) & 1][i];
            if (j == J_ST) {
                store_b(Bn, rb);
                load_b(k_of(s + 2), rb);
            }
            if (j == T::FN - 2) __syncthreads();
            // One operand read per FM MFMAs, then the adds of the column
            // before (masks: 0x8 MFMA, 0x100 LDS read, 0x2 VALU): 4096^3 580
            // -> 570 us against the compiler's order.
            if (j != J_ST) {
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
        split_a(ra);
#pragma unroll
        for (int i = 0; i < T::FM; ++i) acc[i][T::FN - 1] += t[(T::FN - 1) & 1][i];
        load_a(k_of(s + 2), ra);
    }

    bool bad = tiny.x < TINY || tiny.y < TINY;
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
        for (int j = 0; j < T::FN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) bad |= !(__builtin_fabsf(acc[i][j][v]) < INFINITY);
    if (bad) *flag = 1;
    __syncthreads();
    if constexpr (T::WK > 1) {
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
    if (*flag) {
        // In fp32: v_mfma_f32_16x16x4_f32, the same result layout.
#pragma unroll
        for (int i = 0; i < T::FM; ++i)
#pragma unroll
            for (int j = 0; j < T::FN; ++j) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int k0 = max(ks0, 0); k0 < kend; k0 += 4) {
            const int k = k0 + oct;
            float fa[T::FM], fb[T::FN];
#pragma unroll
            for (int i = 0; i < T::FM; ++i) {
                const size_t m = min(mw + 16 * i, g.M - 1);
                fa[i] = k < kend ? (AT ? g.A[(size_t)k * g.lda + m] : g.A[m * g.lda + k]) : 0.f;
            }
#pragma unroll
            for (int j = 0; j < T::FN; ++j)
                fb[j] = k < kend ? BSrc::at(g, k, min(nw + 16 * j + r16, g.N - 1)) : 0.f;
#pragma unroll
            for (int i = 0; i < T::FM; ++i)
#pragma unroll
                for (int j = 0; j < T::FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
    }
    store_matrix<T::FM, T::FN>(g, acc, split, mw, nw + 4 * oct);
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

// 256 x 256: 8 waves of 32 x 256.  128 x 128: 8 waves, 4 of 32 x 128 on each of
// two k groups.
using T256 = STile<2, 16, 8, 1, 1>;
using T128 = STile<2, 8, 4, 1, 2>;

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
        hipLaunchKernelGGL((split_gemm_kernel<T, true>), grid, block, 0, stream(), g);
    else
        hipLaunchKernelGGL((split_gemm_kernel<T, false>), grid, block, 0, stream(), g);
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

} // namespace

// The rule: microseconds of each (tile, splits) choice against those of the fp32
// MFMA kernels, from the sizes alone.  A split work-group takes a fixed time
// (prologue, tail, launch) plus one per step; partials are written and read
// at about 6 TB/s after a reduce launch.  The constants are fits to measured
// calls (start of this kernel / fp32 kernels / estimate, us): 4096^3 538 / 964
// / 533, 1000 x 3001 x 2047 88 / 162 / 87, 1024 x 1024 x 8192 transposed 95 /
// 193 / 99, 2048^3 95 / 131 / 97, 1500^3 60 / 86 / 59, 128 x 4096 x 4096 39 /
// 44 / 37; and 1024^3 32 / 21 / 26, 600^3 23 / 15, 512^3 19 / 12, which stay on
// the fp32 kernels: their 64 x 64 tiles fill the chip without partials, and a
// 64 x 64 split tile converts each value too often (22.8 us at 1024^3).
SplitPlan split_gemm_plan(int64_t M, int64_t N, int64_t K, bool unaligned, int64_t lda, int64_t ldb,
                          int cus) {
    SplitPlan best;
    if (K < 64 || lda >= (1 << 21) || ldb >= (1 << 28) || M > INT32_MAX / 512 || N > INT32_MAX / 512)
        return best;
    auto up = [](int64_t v, int64_t m) { return (v + m - 1) / m; };
    // fp32 kernels: their rate over whole 64 x 64 tiles, lower where an
    // operand is transposed or its rows are not 16-byte aligned
    const bool big = up(M, 256) * up(N, 256) >= cus;
    const double rate = big ? 140e6 : unaligned ? 85e6 : 105e6; // FLOP/us
    double limit = 0.92 * (3.5 + 2.0 * 64 * up(M, 64) * 64 * up(N, 64) * K / rate);
    auto consider = [&](SplitTile tile, int edge, int sb, double fixed, double step) {
        const int64_t tiles = up(M, edge) * up(N, edge);
        if (tiles > INT32_MAX / 64) return;
        for (int want : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
            const int64_t steps = up(K, sb), per = up(steps, want), used = up(steps, per);
            const size_t bytes = used > 1 ? (size_t)used * M * N * sizeof(float) : 0;
            if (used != want || bytes > CAMEL_HIP_NOALLOC_SCRATCH_BYTES || (want > 1 && per < 4)) continue;
            const double t = up(tiles * used, cus) * (fixed + step * per) + (used > 1 ? 2.0 + 2.0 * bytes / 6e6 : 0.0);
            if (t < limit) {
                limit = t;
                best = {tile, (int)used, bytes};
            }
        }
    };
    consider(SplitTile::T256, 256, T256::SB, 8.5, 4.1);
    consider(SplitTile::T128, 128, T128::SB, 7.0, 2.8);
    return best;
}

int split_gemm(SplitGemm g, bool a_trans, const SplitPlan &plan, float *partial) {
    g.partial = partial;
    if (plan.tile == SplitTile::T256) return launch<T256>(g, a_trans, plan.splits);
    return launch<T128>(g, a_trans, plan.splits);
}

} // namespace camel_hip
