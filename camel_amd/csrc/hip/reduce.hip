// Row softmax and the rank-2 reductions (sum / max / argmax along an axis,
// whole-tensor sum).
//
// Softmax fuses the nine-operator composition of test/run/nn/mnist.cml:13-25
// into one pass, op for op:
//   m  = first strict-'>' row max (tensorMaxAxis, runtime.cpp:924-963)
//   mb = fl32(0.0 + m*1.0)         (reshape(m) @ ones([1,k]) broadcast)
//   e  = fl32(exp(fl32(x - mb)))   (subtract, tensorExp 1013-1026; fp32 expf
//                                   here, within 1 ulp of the fp64 libm exp)
//   s  = fl32(sum_j double(e_j))   (tensorSumAxis 887-922, fp64 accumulation)
//   y  = fl32(e / s)               (divide, bit-exact through 1/s in fp64)
// One wave owns one row, several short rows share one, and long rows take a
// work-group; rows up to 32768 columns stay in registers, so HBM sees one read
// and one write per element (8 B/elem).  The fp64 sum
// differs from the reference's sequential order only in the last bits of
// the double, below the fp32 rounding of s.
//
// Max/argmax reductions across lanes keep (value, index) pairs and prefer the
// lower index on ties, which reproduces "first element, then strict '>'",
// including the order of +0/-0; NaN never wins except as element 0.
#include "common.h"
#include "row_softmax.h"

#include <cmath>

namespace camel_hip {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4))); // 16-byte access, 4-byte aligned

constexpr int WAVE = 64;

// One wave per row, the whole row in registers: ITEMS float4 per lane (VEC,
// cols % 4 == 0 and 16-byte aligned rows) or ITEMS*4 scalars per lane.  Slots
// past the end of the row hold -inf, which never wins the max and adds an
// exact 0 to the sum, so only the loads and stores are guarded.
template <int ITEMS, bool VEC>
__device__ __forceinline__ void softmax_row(const float *__restrict__ xr, float *__restrict__ yr,
                                            int cols, int lane) {
    constexpr int NV = ITEMS * 4;
    float v[NV];
    if constexpr (VEC) {
        const int nq = cols >> 2;
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int q = lane + WAVE * it;
            f4 t = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            if (q < nq) t = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(xr) + q);
#pragma unroll
            for (int c = 0; c < 4; ++c) v[4 * it + c] = t[c];
        }
    } else {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = lane + WAVE * j;
            v[j] = c < cols ? xr[c] : -INFINITY;
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) m = max_gt(m, v[j]);
    m = wave_max_gt(m);
    const float x0 = __shfl(v[0], 0); // column 0 sits in lane 0, slot 0, in both layouts
    if (x0 != x0) m = x0;
    const float mb = m + 0.0f; // fl32(0.0 + m * 1.0): the ones-matmul broadcast
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        v[j] = softmax_exp(v[j], mb);
        s += (double)v[j];
    }
    s = wave_sum(s);
    // s >= 1 (the max element contributes exp(0) = 1) or NaN, so the
    // reference's "Division by zero" cannot occur here.
    const double rcp = 1.0 / (double)(float)s;
    if constexpr (VEC) {
        const int nq = cols >> 2;
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int q = lane + WAVE * it;
            if (q < nq) {
                f4 t;
#pragma unroll
                for (int c = 0; c < 4; ++c) t[c] = softmax_div(v[4 * it + c], rcp);
                __builtin_nontemporal_store(t, reinterpret_cast<f4 *>(yr) + q);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = lane + WAVE * j;
            if (c < cols) yr[c] = softmax_div(v[j], rcp);
        }
    }
}

// Row indices of the one-wave-per-row kernels: a grid of at most
// ROW_GRID_CAP blocks of 4 waves strides over the rows, so any row count
// fits the launch's 32-bit grid (one row per wave up to 4 * ROW_GRID_CAP rows).
constexpr int64_t ROW_GRID_CAP = 1 << 20;

inline unsigned row_grid(int64_t rows) {
    return (unsigned)std::min<int64_t>((rows + 3) / 4, ROW_GRID_CAP);
}

__device__ __forceinline__ int64_t first_row() {
    return (int64_t)blockIdx.x * (blockDim.x / WAVE) + (threadIdx.x >> 6);
}

__device__ __forceinline__ int64_t row_step() { return (int64_t)gridDim.x * (blockDim.x / WAVE); }

template <int ITEMS, bool VEC>
__global__ __launch_bounds__(256) void softmax_rows_kernel(const float *__restrict__ x,
                                                           float *__restrict__ y, int64_t rows,
                                                           int cols) {
    const int lane = threadIdx.x & 63;
    for (int64_t row = first_row(); row < rows; row += row_step())
        softmax_row<ITEMS, VEC>(x + row * cols, y + row * cols, cols, lane);
}

// Short rows: a wave takes 64 >> LG rows at once, 1 << LG lanes per row, one
// float4 (VEC) or one value per lane, SHORT_ROWS such groups in flight.  The
// sums of a row are added in the order of the one-row kernel, whose further
// lanes add exact zeros.
constexpr int SHORT_ROWS = 4;

template <int LG, bool VEC>
__global__ __launch_bounds__(256) void softmax_short_rows_kernel(const float *__restrict__ x,
                                                                 float *__restrict__ y, int64_t rows,
                                                                 int cols) {
    constexpr int NV = VEC ? 4 : 1, WIDTH = 1 << LG, PER_WAVE = WAVE >> LG;
    const int lane = threadIdx.x & 63;
    const int c = (lane & (WIDTH - 1)) * NV;
    const int64_t chunk = (int64_t)PER_WAVE * SHORT_ROWS;
    for (int64_t r0 = first_row() * chunk; r0 < rows; r0 += row_step() * chunk) {
        float v[SHORT_ROWS][NV];
        int64_t at[SHORT_ROWS];
        bool in[SHORT_ROWS];
#pragma unroll
        for (int u = 0; u < SHORT_ROWS; ++u) {
            const int64_t row = r0 + u * PER_WAVE + (lane >> LG);
            at[u] = row * cols + c;
            in[u] = row < rows && c < cols;
#pragma unroll
            for (int i = 0; i < NV; ++i) v[u][i] = -INFINITY;
            if constexpr (VEC) {
                if (in[u]) {
                    const f4 t = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(x + at[u]));
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[u][i] = t[i];
                }
            } else if (in[u]) {
                v[u][0] = x[at[u]];
            }
        }
#pragma unroll
        for (int u = 0; u < SHORT_ROWS; ++u) {
            float m = -INFINITY;
#pragma unroll
            for (int i = 0; i < NV; ++i) m = max_gt(m, v[u][i]);
#pragma unroll
            for (int off = WIDTH >> 1; off > 0; off >>= 1) m = max_gt(m, __shfl_xor(m, off));
            const float x0 = __shfl(v[u][0], 0, WIDTH);
            if (x0 != x0) m = x0;
            const float mb = m + 0.0f;
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                v[u][i] = softmax_exp(v[u][i], mb);
                s += (double)v[u][i];
            }
#pragma unroll
            for (int off = WIDTH >> 1; off > 0; off >>= 1) s += __shfl_xor(s, off);
            const double rcp = 1.0 / (double)(float)s;
            if (in[u]) {
                if constexpr (VEC) {
                    f4 t;
#pragma unroll
                    for (int i = 0; i < 4; ++i) t[i] = softmax_div(v[u][i], rcp);
                    __builtin_nontemporal_store(t, reinterpret_cast<f4 *>(y + at[u]));
                } else {
                    y[at[u]] = softmax_div(v[u][0], rcp);
                }
            }
        }
    }
}

// Block-wide max and sum of a wave's values; every thread gets the result.
template <int WAVES> __device__ __forceinline__ float block_max_gt(float m, float *lds) {
    m = wave_max_gt(m);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = m;
    __syncthreads();
    m = lds[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m = max_gt(m, lds[w]);
    return m;
}
template <int WAVES> __device__ __forceinline__ double block_sum(double s, double *lds) {
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    s = lds[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) s += lds[w];
    return s;
}

// One work-group per row, the row in registers (ITEMS groups of 4 columns per
// thread, loaded and stored as 16 bytes also where rows are only 4-byte
// aligned): rows too long for a wave's registers, and rows too few to fill the
// chip with one wave each.
template <int THREADS, int ITEMS, class Quad>
__global__ __launch_bounds__(THREADS) void softmax_block_kernel(const float *__restrict__ x,
                                                                float *__restrict__ y, int64_t rows,
                                                                int cols) {
    constexpr int WAVES = THREADS / WAVE, NV = ITEMS * 4;
    __shared__ float lds_max[WAVES];
    __shared__ double lds_sum[WAVES];
    const int quads = cols >> 2, tail = cols & 3; // the last `tail` columns belong to quad number `quads`
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
        const float *xr = x + row * cols;
        float *yr = y + row * cols;
        float v[NV];
        const float x0 = xr[0];
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int q = threadIdx.x + THREADS * it;
            f4 t = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            if (q < quads) {
                t = __builtin_nontemporal_load(reinterpret_cast<const Quad *>(xr + 4 * q));
            } else if (q == quads) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c < tail) t[c] = xr[4 * q + c];
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) v[4 * it + c] = t[c];
        }
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < NV; ++j) m = max_gt(m, v[j]);
        m = block_max_gt<WAVES>(m, lds_max);
        if (x0 != x0) m = x0;
        const float mb = m + 0.0f;
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            v[j] = softmax_exp(v[j], mb);
            s += (double)v[j];
        }
        // The next row's max is stored only behind this barrier, and its sum
        // behind the barrier of that max: no thread still reads the old ones.
        s = block_sum<WAVES>(s, lds_sum);
        const double rcp = 1.0 / (double)(float)s;
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int q = threadIdx.x + THREADS * it;
            f4 t;
#pragma unroll
            for (int c = 0; c < 4; ++c) t[c] = softmax_div(v[4 * it + c], rcp);
            if (q < quads) {
                __builtin_nontemporal_store((Quad)t, reinterpret_cast<Quad *>(yr + 4 * q));
            } else if (q == quads) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c < tail) yr[4 * q + c] = t[c];
            }
        }
    }
}

// Rows beyond a work-group's registers: max pass, sum pass, write pass.
constexpr int LONG_THREADS = 1024;

__global__ __launch_bounds__(LONG_THREADS) void softmax_long_kernel(const float *__restrict__ x,
                                                                    float *__restrict__ y, int64_t rows,
                                                                    int64_t cols) {
    constexpr int WAVES = LONG_THREADS / WAVE;
    __shared__ float lds_max[WAVES];
    __shared__ double lds_sum[WAVES];
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
        const float *xr = x + row * cols;
        float *yr = y + row * cols;
        const float x0 = xr[0];
        float m = -INFINITY;
        for (int64_t c = threadIdx.x; c < cols; c += LONG_THREADS) m = max_gt(m, xr[c]);
        m = block_max_gt<WAVES>(m, lds_max);
        if (x0 != x0) m = x0;
        const float mb = m + 0.0f;
        double s = 0.0;
        for (int64_t c = threadIdx.x; c < cols; c += LONG_THREADS) s += (double)softmax_exp(xr[c], mb);
        s = block_sum<WAVES>(s, lds_sum);
        const double rcp = 1.0 / (double)(float)s;
        for (int64_t c = threadIdx.x; c < cols; c += LONG_THREADS)
            yr[c] = softmax_div(softmax_exp(xr[c], mb), rcp);
    }
}

// axis = 1: one wave per row.  kind 0 = sum, 1 = max, 2 = argmax.
__global__ __launch_bounds__(256) void reduce_rows_kernel(int kind, int dt, const void *x,
                                                          int64_t rows, int64_t cols, void *out) {
    const int lane = threadIdx.x & 63;
    for (int64_t row = first_row(); row < rows; row += row_step()) {
    const int64_t base = row * cols;
    if (kind == 0) {
        double s = 0.0;
        for (int64_t c = lane; c < cols; c += WAVE) s += load_as_double(dt, x, base + c);
        s = wave_sum(s);
        if (lane == 0) static_cast<float *>(out)[row] = (float)s;
        continue;
    }
    // Values compare as doubles (exact for fp32 and bool; int64 as the
    // reference converts it).  Track them as double to keep int64 order.
    double bv = 0.0;
    int64_t bi = INT64_MAX;
    for (int64_t c = lane; c < cols; c += WAVE) {
        const double v = load_as_double(dt, x, base + c);
        if (v != v) continue;
        if (bi == INT64_MAX || v > bv) {
            bv = v;
            bi = c;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double ov = __shfl_xor(bv, off);
        const int64_t oi = __shfl_xor(bi, off);
        if (oi != INT64_MAX && (bi == INT64_MAX || ov > bv || (ov == bv && oi < bi))) {
            bv = ov;
            bi = oi;
        }
    }
    if (lane == 0) {
        const double x0 = load_as_double(dt, x, base);
        if (x0 != x0 || bi == INT64_MAX) {
            bv = x0;
            bi = 0;
        }
        if (kind == 1)
            static_cast<float *>(out)[row] = (float)bv;
        else
            static_cast<int64_t *>(out)[row] = bi;
    }
    }
}

// axis = 0: one thread per column, rows in the reference's order (exact).
__global__ void reduce_cols_kernel(int kind, int dt, const void *x, int64_t rows, int64_t cols,
                                   void *out) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < cols; j += stride) {
        if (kind == 0) {
            double acc = 0.0;
            for (int64_t i = 0; i < rows; ++i) acc += load_as_double(dt, x, i * cols + j);
            static_cast<float *>(out)[j] = (float)acc;
        } else {
            double best = load_as_double(dt, x, j);
            int64_t best_i = 0;
            for (int64_t i = 1; i < rows; ++i) {
                const double v = load_as_double(dt, x, i * cols + j);
                if (v > best) {
                    best = v;
                    best_i = i;
                }
            }
            if (kind == 1)
                static_cast<float *>(out)[j] = (float)best;
            else
                static_cast<int64_t *>(out)[j] = best_i;
        }
    }
}

// Whole-tensor sum: per-block fp64 partials, then one block folds them.
__global__ __launch_bounds__(256) void sum_partial_kernel(int dt, const void *x, int64_t n,
                                                          double *partial) {
    __shared__ double lds[256 / WAVE];
    double s = 0.0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        s += load_as_double(dt, x, i);
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x / WAVE); ++w) t += lds[w];
        partial[blockIdx.x] = t;
    }
}

__global__ __launch_bounds__(256) void sum_final_kernel(const double *partial, int count,
                                                        double *result) {
    __shared__ double lds[256 / WAVE];
    double s = 0.0;
    for (int i = threadIdx.x; i < count; i += blockDim.x) s += partial[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x / WAVE); ++w) t += lds[w];
        *result = t;
    }
}

template <int ITEMS> int launch_softmax(const float *x, float *y, int64_t rows, int cols, bool vec) {
    dim3 grid(row_grid(rows)), block(256);
    if (vec)
        hipLaunchKernelGGL((softmax_rows_kernel<ITEMS, true>), grid, block, 0, stream(), x, y, rows,
                           cols);
    else
        hipLaunchKernelGGL((softmax_rows_kernel<ITEMS, false>), grid, block, 0, stream(), x, y,
                           rows, cols);
    return check_launch("softmax_rows_kernel");
}

template <int THREADS, int ITEMS>
int launch_softmax_block(const float *x, float *y, int64_t rows, int cols, bool vec) {
    dim3 grid((unsigned)std::min<int64_t>(rows, ROW_GRID_CAP)), block(THREADS);
    if (vec)
        hipLaunchKernelGGL((softmax_block_kernel<THREADS, ITEMS, f4>), grid, block, 0, stream(), x, y,
                           rows, cols);
    else
        hipLaunchKernelGGL((softmax_block_kernel<THREADS, ITEMS, f4u>), grid, block, 0, stream(), x, y,
                           rows, cols);
    return check_launch("softmax_block_kernel");
}

template <int LG> int launch_softmax_short(const float *x, float *y, int64_t rows, int cols, bool vec) {
    if constexpr (LG < 6)
        if ((1 << LG) * (vec ? 4 : 1) < cols) return launch_softmax_short<LG + 1>(x, y, rows, cols, vec);
    constexpr int CHUNK = (WAVE >> LG) * SHORT_ROWS;
    dim3 grid(row_grid((rows + CHUNK - 1) / CHUNK)), block(256);
    if (vec)
        hipLaunchKernelGGL((softmax_short_rows_kernel<LG, true>), grid, block, 0, stream(), x, y, rows, cols);
    else
        hipLaunchKernelGGL((softmax_short_rows_kernel<LG, false>), grid, block, 0, stream(), x, y, rows, cols);
    return check_launch("softmax_short_rows_kernel");
}

int check_axis(int64_t rows, int64_t cols, int64_t &axis, const char *what) {
    if (rows < 0 || cols < 0) return fail(CAMEL_HIP_ERR_SHAPE, std::string(what) + ": negative shape");
    if (!product_fits({rows, cols, 8}, INT64_MAX))
        return fail(CAMEL_HIP_ERR_SHAPE, std::string(what) + ": tensor too large");
    if (axis < 0) axis += 2;
    if (axis != 0 && axis != 1)
        return fail(CAMEL_HIP_ERR_SHAPE,
                    std::string(what) + "(axis): axis must be 0 or 1 for rank-2 tensors");
    return CAMEL_HIP_OK;
}

int reduce_axis(int kind, int dt, const void *x, int64_t rows, int64_t cols, int64_t axis,
                void *out, const char *what) {
    if (!valid_dtype(dt)) return fail(CAMEL_HIP_ERR_DTYPE, std::string(what) + ": unsupported dtype");
    CAMEL_RETURN_IF(check_axis(rows, cols, axis, what));
    const int64_t out_n = axis == 0 ? cols : rows;
    const int64_t red_n = axis == 0 ? rows : cols;
    if (out_n == 0) return ok();
    if (red_n == 0 && kind != 0)
        return fail(CAMEL_HIP_ERR_SHAPE, std::string(what) + ": reduction over an empty axis");
    if (!out || (red_n > 0 && !x)) return fail(CAMEL_HIP_ERR_ARG, std::string(what) + ": null pointer");
    CAMEL_LOCK();
    CAMEL_INIT_OR_RETURN();
    if (axis == 1) {
        hipLaunchKernelGGL(reduce_rows_kernel, dim3(row_grid(rows)), dim3(256), 0,
                           stream(), kind, dt, x, rows, cols, out);
        CAMEL_RETURN_IF(check_launch("reduce_rows_kernel"));
    } else {
        hipLaunchKernelGGL(reduce_cols_kernel, dim3(grid_for(cols, 256, 16)), dim3(256), 0,
                           stream(), kind, dt, x, rows, cols, out);
        CAMEL_RETURN_IF(check_launch("reduce_cols_kernel"));
    }
    return ok();
}

} // namespace
} // namespace camel_hip

using namespace camel_hip;

extern "C" {

int camel_hip_softmax_rows(const float *x, float *y, int64_t rows, int64_t cols) {
    if (rows < 0 || cols < 0) return fail(CAMEL_HIP_ERR_SHAPE, "softmax: negative shape");
    if (!product_fits({rows, cols, 4}, INT64_MAX))
        return fail(CAMEL_HIP_ERR_SHAPE, "softmax: tensor too large");
    if (rows == 0 || cols == 0) return ok();
    if (!x || !y) return fail(CAMEL_HIP_ERR_ARG, "softmax: null pointer");
    if (cols > INT32_MAX / 2) return fail(CAMEL_HIP_ERR_SHAPE, "softmax: row too long");
    CAMEL_LOCK();
    CAMEL_INIT_OR_RETURN();
    const bool vec = (cols % 4 == 0) && (((uintptr_t)x | (uintptr_t)y) & 15) == 0;
    const int c = (int)cols;
    // Up to 4096 columns a wave holds a row.  Short rows share a wave once one
    // row per wave would queue (262144 x 10: 66 -> 12.6 us, x 64: 82 -> 24; 4096
    // rows: 3.1 against 4.6, so not below 8192), wider rows later, as fewer of them
    // share a wave (one per wave / shared: 10240 x 64 4.8 / 4.5, 10240 x 128 5.3 /
    // 5.7, 12288 x 128 5.6 / 5.8, 16385 x 128 7.3 / 5.8, 12288 x 256 6.8 / 7.3, 16385 x
    // 256 8.3 / 7.9).  A row is spread over a
    // work-group where rows are too few for the chip (256 x 1024 3.5 -> 2.8 us;
    // 1024 rows: 3.9 both; 1024 x 2048 5.5 -> 4.9, 4096 rows: 11.8 against 13.1)
    // or too long for a wave: from 2048 columns on (16384 x 4096 95 -> 85 us, 3001
    // unaligned columns 113 -> 74, 1024 x 8192 108 -> 10, 4096 x 16384 422 -> 93:
    // 5.8 TB/s, 4096 x 32768 904 -> 249, 16 x 32768 234 -> 8).  Group sizes: 8
    // quads per thread beat 4 from 4096 columns on (1024 x 16384: 24.4 us against
    // 32.2 for 1024 x 4 quads and 25.5 for 256 x 16), whose work-groups of 1024
    // threads have a CU to themselves.
    if (cols <= (vec ? 256 : 64) && rows > 8192 + 32 * cols)
        CAMEL_RETURN_IF(launch_softmax_short<0>(x, y, rows, c, vec));
    else if (cols <= 256)
        CAMEL_RETURN_IF(launch_softmax<1>(x, y, rows, c, vec));
    else if (cols <= 512)
        CAMEL_RETURN_IF(launch_softmax<2>(x, y, rows, c, vec));
    else if (cols <= 1024 && rows > 512)
        CAMEL_RETURN_IF(launch_softmax<4>(x, y, rows, c, vec));
    else if (cols <= 1024)
        CAMEL_RETURN_IF((launch_softmax_block<256, 1>(x, y, rows, c, vec)));
    else if (cols <= 2048 && rows > 2048)
        CAMEL_RETURN_IF(launch_softmax<8>(x, y, rows, c, vec));
    else if (cols <= 2048)
        CAMEL_RETURN_IF((launch_softmax_block<256, 2>(x, y, rows, c, vec)));
    else if (cols <= 4096)
        CAMEL_RETURN_IF((launch_softmax_block<256, 4>(x, y, rows, c, vec)));
    else if (cols <= 8192)
        CAMEL_RETURN_IF((launch_softmax_block<256, 8>(x, y, rows, c, vec)));
    else if (cols <= 16384)
        CAMEL_RETURN_IF((launch_softmax_block<512, 8>(x, y, rows, c, vec)));
    else if (cols <= 32768)
        CAMEL_RETURN_IF((launch_softmax_block<1024, 8>(x, y, rows, c, vec)));
    else {
        hipLaunchKernelGGL(softmax_long_kernel, dim3((unsigned)std::min<int64_t>(rows, ROW_GRID_CAP)),
                           dim3(LONG_THREADS), 0, stream(), x, y, rows, cols);
        CAMEL_RETURN_IF(check_launch("softmax_long_kernel"));
    }
    return ok();
}

int camel_hip_sum_axis(int dt, const void *x, int64_t rows, int64_t cols, int64_t axis,
                       float *out) {
    return reduce_axis(0, dt, x, rows, cols, axis, out, "sum");
}

int camel_hip_max_axis(int dt, const void *x, int64_t rows, int64_t cols, int64_t axis,
                       float *out) {
    return reduce_axis(1, dt, x, rows, cols, axis, out, "max");
}

int camel_hip_argmax_axis(int dt, const void *x, int64_t rows, int64_t cols, int64_t axis,
                          int64_t *out) {
    return reduce_axis(2, dt, x, rows, cols, axis, out, "argmax");
}

int camel_hip_sum(int dt, const void *x, int64_t n, double *result) {
    if (!valid_dtype(dt)) return fail(CAMEL_HIP_ERR_DTYPE, "sum: unsupported dtype");
    if (!result || n < 0) return fail(CAMEL_HIP_ERR_ARG, "sum: bad argument");
    if (n == 0) {
        *result = 0.0;
        return ok();
    }
    if (!x) return fail(CAMEL_HIP_ERR_ARG, "sum: null input");
    CAMEL_LOCK();
    CAMEL_INIT_OR_RETURN();
    const unsigned blocks = grid_for(n, 256, 4);
    void *ws = nullptr;
    CAMEL_RETURN_IF(camel_hip_malloc(&ws, (blocks + 1) * sizeof(double)));
    double *partial = static_cast<double *>(ws);
    hipLaunchKernelGGL(sum_partial_kernel, dim3(blocks), dim3(256), 0, stream(), dt, x, n, partial);
    int rc = check_launch("sum_partial_kernel");
    if (rc == CAMEL_HIP_OK) {
        hipLaunchKernelGGL(sum_final_kernel, dim3(1), dim3(256), 0, stream(), partial, (int)blocks,
                           partial + blocks);
        rc = check_launch("sum_final_kernel");
    }
    if (rc == CAMEL_HIP_OK)
        rc = camel_hip_d2h(result, partial + blocks, sizeof(double));
    camel_hip_free(ws);
    CAMEL_RETURN_IF(rc);
    return ok();
}

} // extern "C"
