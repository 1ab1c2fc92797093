// Elementwise stretches of the GraphSAGE layers between their matrix products: relu(layer_norm(x)), and its gradient together
// with that of the dropout before it (reference: examples/graphsage/sage.py:176-211, conv -> dropout -> norm -> relu).
//
// Bound by memory: each direction reads its row operands once and writes once.  A group of G lanes owns a row of up to
// 4 * G * NV floats and holds it in registers between the reductions over the row; two rows per group are in flight.
// 150 k rows of 256 floats: forward 215 us as torch's layer_norm and relu -> 52; backward 440 us as threshold, two layer_norm
// gradients and the mask's product -> 85 (5.9 TB/s).
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace sgnn {

constexpr int kNormBlock = 256;
constexpr int kNormRows = 2;              // rows of a group in flight
constexpr int kNormBackwardBlocks = 1024; // four per CU: each leaves one partial sum of the two parameter gradients

template <int G>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
    for (int d = G / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    return v;
}

template <int G, int NV>
__global__ __launch_bounds__(kNormBlock) void norm_relu_kernel(const float *__restrict__ x, const float *__restrict__ weight,
                                                               const float *__restrict__ bias, float eps, float *__restrict__ y,
                                                               float2 *__restrict__ stats, uint8_t *__restrict__ signs, int64_t n,
                                                               int C) {
    const int lig = threadIdx.x % G;
    const int64_t row0 = ((int64_t)blockIdx.x * (kNormBlock / G) + threadIdx.x / G) * kNormRows;
    float v[kNormRows][NV][4];
#pragma unroll
    for (int r = 0; r < kNormRows; ++r) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int c = 4 * (lig + G * k);
            if (row0 + r < n && c < C) {
                vec_load_nt<4>(v[r][k], x + (row0 + r) * C + c);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[r][k][e] = 0.0f;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kNormRows; ++r) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < NV; ++k) s += (v[r][k][0] + v[r][k][1]) + (v[r][k][2] + v[r][k][3]);
        const float mean = group_sum<G>(s) / (float)C;
        float q = 0.0f;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = 4 * (lig + G * k) < C ? v[r][k][e] - mean : 0.0f;
                q = fmaf(d, d, q);
            }
        }
        const float rstd = 1.0f / sqrtf(group_sum<G>(q) / (float)C + eps);
        if (row0 + r >= n) return;
        if (lig == 0) stats[row0 + r] = make_float2(mean, rstd);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int c = 4 * (lig + G * k);
            uint32_t passed = 0;   // bit e: the rectifier passes element e (NaN passes)
            if (c < C) {
                float w[4], b[4], o[4];
                vec_load<4>(w, weight + c);
                vec_load<4>(b, bias + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float p = fmaf((v[r][k][e] - mean) * rstd, w[e], b[e]);
                    o[e] = p < 0.0f ? 0.0f : p;   // (NaN stays)
                    passed |= (p <= 0.0f ? 0u : 1u) << e;
                }
                vec_store<4>(y + (row0 + r) * C + c, o);
            }
            const uint32_t right = __shfl_xor(passed, 1, 64);   // two lanes share a byte
            if (signs && c < C && (lig & 1) == 0) signs[(row0 + r) * ((C + 7) / 8) + c / 8] = (uint8_t)(passed | right << 4);
        }
    }
}

// Gradient w.r.t. the rows x before a dropout that kept the elements of `mask` times `scale` (mask null: no dropout), and each
// workgroup's sums of the gradients w.r.t. weight and bias: partial[block][2][C].  The elements that the rectifier passed are those
// of `signs`; null: where the norm of mask * scale * x, computed anew, is above 0.
template <int G, int NV>
__global__ __launch_bounds__(kNormBlock) void norm_relu_backward_kernel(
    const float *__restrict__ g, const float *__restrict__ x, const uint8_t *__restrict__ mask, float scale,
    const float2 *__restrict__ stats, const uint8_t *__restrict__ signs, const float *__restrict__ weight, const float *__restrict__ bias,
    float *__restrict__ gx, float *__restrict__ partial, int64_t n, int C) {
    constexpr int kGroups = kNormBlock / G;
    __shared__ float sums[kGroups][2][G * NV * 4];
    const int lig = threadIdx.x % G, group = threadIdx.x / G;
    float w[NV][4], b[NV][4], gw[NV][4], gb[NV][4];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int c = 4 * (lig + G * k);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            w[k][e] = c < C ? weight[c + e] : 0.0f;
            b[k][e] = c < C ? bias[c + e] : 0.0f;
            gw[k][e] = gb[k][e] = 0.0f;
        }
    }
    const float inv = 1.0f / (float)C;
    const int64_t step = (int64_t)gridDim.x * kGroups * kNormRows;
    for (int64_t row0 = ((int64_t)blockIdx.x * kGroups + group) * kNormRows; row0 < n; row0 += step) {
        float gv[kNormRows][NV][4], xv[kNormRows][NV][4];
        uint32_t keep[kNormRows][NV], passed[kNormRows][NV];
        float2 st[kNormRows];
#pragma unroll
        for (int r = 0; r < kNormRows; ++r) {
            st[r] = row0 + r < n ? stats[row0 + r] : make_float2(0.0f, 0.0f);
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int c = 4 * (lig + G * k);
                const int64_t i = (row0 + r) * C + c;
                keep[r][k] = 0x01010101u;
                passed[r][k] = 0;
                if (row0 + r < n && c < C) {
                    if (signs) passed[r][k] = (uint32_t)signs[(row0 + r) * ((C + 7) / 8) + c / 8] >> (c & 4);
                    vec_load_nt<4>(gv[r][k], g + i);
                    vec_load_nt<4>(xv[r][k], x + i);
                    if (mask) keep[r][k] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t *>(mask + i));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) gv[r][k][e] = xv[r][k][e] = 0.0f;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < kNormRows; ++r) {
            const float mean = st[r].x, rstd = st[r].y;
            float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const bool in = row0 + r < n && 4 * (lig + G * k) < C;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float xd = keep[r][k] >> (8 * e) & 0xffu ? xv[r][k][e] * scale : 0.0f;
                    const float h = in ? (xd - mean) * rstd : 0.0f;
                    const bool pass = signs ? passed[r][k] >> e & 1u : !(fmaf(h, w[k][e], b[k][e]) <= 0.0f);
                    const float gr = pass ? gv[r][k][e] : 0.0f;
                    gw[k][e] = fmaf(gr, h, gw[k][e]);
                    gb[k][e] += gr;
                    const float gh = gr * w[k][e];
                    s1 += gh;
                    s2 = fmaf(gh, h, s2);
                    gv[r][k][e] = gh;
                    xv[r][k][e] = h;
                }
            }
            s1 = group_sum<G>(s1) * inv;
            s2 = group_sum<G>(s2) * inv;
            if (row0 + r < n) {
#pragma unroll
                for (int k = 0; k < NV; ++k) {
                    const int c = 4 * (lig + G * k);
                    if (c >= C) continue;
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = (gv[r][k][e] - s1 - xv[r][k][e] * s2) * rstd;
                        o[e] = v * (keep[r][k] >> (8 * e) & 0xffu ? scale : 0.0f);   // (NaN and infinities times 0, as the mask's product)
                    }
                    vec_store<4>(gx + (row0 + r) * C + c, o);
                }
            }
        }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sums[group][0][4 * (lig + G * k) + e] = gw[k][e];
            sums[group][1][4 * (lig + G * k) + e] = gb[k][e];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * C; i += kNormBlock) {
        const int which = i >= C, c = i - which * C;
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < kGroups; ++q) s += (double)sums[q][which][c];
        partial[(int64_t)blockIdx.x * 2 * C + i] = (float)s;
    }
}

// Sums over the rows of each column, per workgroup: partial[block][C].  Bound by memory (150 k x 256: 65 us as torch's sum,
// whose 64 workgroups leave most of the chip idle -> 30 us with the sum of the partials).
template <int G, int NV>
__global__ __launch_bounds__(kNormBlock) void column_sum_kernel(const float *__restrict__ x, float *__restrict__ partial, int64_t n, int C) {
    constexpr int kGroups = kNormBlock / G, kRows = 4;
    __shared__ float sums[kGroups][G * NV * 4];
    const int lig = threadIdx.x % G, group = threadIdx.x / G;
    float acc[NV][4] = {};
    const int64_t step = (int64_t)gridDim.x * kGroups * kRows;
    for (int64_t row0 = ((int64_t)blockIdx.x * kGroups + group) * kRows; row0 < n; row0 += step) {
        float v[kRows][NV][4];
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int c = 4 * (lig + G * k);
                if (row0 + r < n && c < C) {
                    vec_load<4>(v[r][k], x + (row0 + r) * C + c);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[r][k][e] = 0.0f;
                }
            }
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r)
#pragma unroll
            for (int k = 0; k < NV; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[k][e] += v[r][k][e];
    }
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) sums[group][4 * (lig + G * k) + e] = acc[k][e];
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += kNormBlock) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < kGroups; ++q) s += (double)sums[q][c];
        partial[(int64_t)blockIdx.x * C + c] = (float)s;
    }
}

// (a, b)[i] = sum over blocks of partial[block][i], the first n_a columns in a: 16 columns and 16 parts of the blocks per
// workgroup, in fixed order and 64 bits (the sums of 1024 workgroups lose more than their rows do otherwise).
__global__ __launch_bounds__(256) void partial_sum_kernel(const float *__restrict__ partial, float *__restrict__ a, float *__restrict__ b,
                                                          int blocks, int n_a, int n) {
    __shared__ double part[16][17];
    const int c = threadIdx.x & 15, q = threadIdx.x >> 4, i = blockIdx.x * 16 + c;
    double s = 0.0;
    if (i < n) {
#pragma unroll 8
        for (int k = q; k < blocks; k += 16) s += (double)partial[(int64_t)k * n + i];
    }
    part[q][c] = s;
    __syncthreads();
    if (q == 0 && i < n) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += part[k][c];
        if (i < n_a) a[i] = (float)t;
        else b[i - n_a] = (float)t;
    }
}

// w[i, j] += sum over rows r of g[r, i] * a[r, j], for the few rows a batched product over equal slabs leaves over: the library gives
// the whole product to one workgroup (18 ... 21 us for 48 rows of 47 ... 256 columns, here 9 ... 11; six times a training step of three layers).
// 64 x 64 outputs per workgroup, 4 x 4 per thread, 64 rows of both operands in LDS at a time: the latency of one round of loads.
constexpr int kRestRows = 64;
__global__ __launch_bounds__(256) void rest_product_kernel(const float *__restrict__ g, const float *__restrict__ a, float *__restrict__ w,
                                                           int rows, int n_out, int n_in) {
    __shared__ float gs[kRestRows][64], as[kRestRows][64];
    const int i0 = blockIdx.x * 64, j0 = blockIdx.y * 64, ti = threadIdx.x / 16, tj = threadIdx.x % 16;
    float acc[4][4] = {};
    for (int r0 = 0; r0 < rows; r0 += kRestRows) {
        float gv[kRestRows * 64 / 256], av[kRestRows * 64 / 256];
#pragma unroll
        for (int k = 0; k < kRestRows * 64 / 256; ++k) {
            const int r = r0 + (threadIdx.x + 256 * k) / 64, c = threadIdx.x % 64;
            gv[k] = r < rows && i0 + c < n_out ? g[(int64_t)r * n_out + i0 + c] : 0.0f;
            av[k] = r < rows && j0 + c < n_in ? a[(int64_t)r * n_in + j0 + c] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kRestRows * 64 / 256; ++k) {
            gs[(threadIdx.x + 256 * k) / 64][threadIdx.x % 64] = gv[k];
            as[(threadIdx.x + 256 * k) / 64][threadIdx.x % 64] = av[k];
        }
        __syncthreads();
        for (int r = 0; r < kRestRows && r0 + r < rows; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(gs[r][ti + 16 * i], as[r][tj + 16 * j], acc[i][j]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (i0 + ti + 16 * i < n_out && j0 + tj + 16 * j < n_in) w[(int64_t)(i0 + ti + 16 * i) * n_in + j0 + tj + 16 * j] += acc[i][j];
}

// f(G, NV) with the lane group of rows of C floats: the narrowest of 8 ... 64 lanes, one to four vectors each.
template <typename F>
static void with_norm_shape(int64_t C, F f) {
#define SGNN_NORM(g, nv) f(std::integral_constant<int, g>(), std::integral_constant<int, nv>())
    if (C <= 32) SGNN_NORM(8, 1);
    else if (C <= 64) SGNN_NORM(16, 1);
    else if (C <= 128) SGNN_NORM(32, 1);
    else if (C <= 256) SGNN_NORM(64, 1);
    else if (C <= 512) SGNN_NORM(64, 2);
    else SGNN_NORM(64, 4);
#undef SGNN_NORM
}

static int norm_blocks(int64_t n, int64_t C) {
    const int64_t groups = C <= 32 ? 32 : C <= 64 ? 16 : C <= 128 ? 8 : 4;
    return (int)std::min<int64_t>(kNormBackwardBlocks, (n + groups * kNormRows - 1) / (groups * kNormRows));
}

}  // namespace sgnn

using namespace sgnn;

static int check_norm(const void *a, const void *b, const void *w, const void *bias, int64_t n, int64_t C) {
    SGNN_REQUIRE(n >= 0 && C > 0 && C % 4 == 0 && C <= 1024, "rows of %lld floats: a multiple of 4 up to 1024 is needed", (long long)C);
    SGNN_REQUIRE(n < ((int64_t)1 << 31), "too many rows");
    SGNN_REQUIRE(n == 0 || (a && b && w && bias), "null argument");
    SGNN_REQUIRE(aligned(a, 16) && aligned(b, 16) && aligned(w, 16) && aligned(bias, 16), "operands must be 16-byte aligned");
    return SGNN_OK;
}

extern "C" int sgnn_norm_relu_f32(const float *x, const float *weight, const float *bias, float eps, float *y, float *stats,
                                  uint8_t *signs, int64_t n, int64_t C, sgnn_stream_t stream) {
    const int rc = check_norm(x, y, weight, bias, n, C);
    if (rc != SGNN_OK || n == 0) return rc;
    SGNN_REQUIRE(stats != nullptr && aligned(stats, 8), "stats must be non-null and 8-byte aligned");
    with_norm_shape(C, [&](auto g, auto nv) {
        const int64_t per = (kNormBlock / g) * kNormRows;
        hipLaunchKernelGGL((norm_relu_kernel<g, nv>), dim3((uint32_t)((n + per - 1) / per)), dim3(kNormBlock), 0, (hipStream_t)stream, x, weight,
                           bias, eps, y, reinterpret_cast<float2 *>(stats), signs, n, (int)C);
    });
    SGNN_HIP_CHECK(hipGetLastError());
    return SGNN_OK;
}

extern "C" int64_t sgnn_norm_relu_workspace(int64_t n, int64_t C) { return n <= 0 || C <= 0 ? 0 : (int64_t)norm_blocks(n, C) * 2 * C; }

extern "C" int sgnn_norm_relu_backward_f32(const float *g, const float *x, const uint8_t *mask, float scale, const float *stats,
                                           const uint8_t *signs, const float *weight, const float *bias, float *gx, float *workspace, float *gw,
                                           float *gb, int64_t n, int64_t C, sgnn_stream_t stream) {
    int rc = check_norm(g, x, weight, bias, n, C);
    if (rc != SGNN_OK || n == 0) return rc;
    SGNN_REQUIRE(gx && workspace && gw && gb && stats && aligned(gx, 16) && aligned(stats, 8) && aligned(mask, 4), "null or misaligned argument");
    const int blocks = norm_blocks(n, C);
    with_norm_shape(C, [&](auto gl, auto nv) {
        hipLaunchKernelGGL((norm_relu_backward_kernel<gl, nv>), dim3((uint32_t)blocks), dim3(kNormBlock), 0, (hipStream_t)stream, g, x, mask, scale,
                           reinterpret_cast<const float2 *>(stats), signs, weight, bias, gx, workspace, n, (int)C);
    });
    hipLaunchKernelGGL(partial_sum_kernel, dim3((uint32_t)((2 * C + 15) / 16)), dim3(256), 0, (hipStream_t)stream, workspace, gw, gb, blocks,
                       (int)C, (int)(2 * C));
    SGNN_HIP_CHECK(hipGetLastError());
    return SGNN_OK;
}

extern "C" int sgnn_column_sum_f32(const float *x, float *workspace, float *out, int64_t n, int64_t C, sgnn_stream_t stream) {
    const int rc = check_norm(x, x, x, x, n, C);
    if (rc != SGNN_OK) return rc;
    SGNN_REQUIRE(n > 0 && workspace && out, "null argument or no rows");
    const int blocks = norm_blocks(n, C);
    with_norm_shape(C, [&](auto g, auto nv) {
        hipLaunchKernelGGL((column_sum_kernel<g, nv>), dim3((uint32_t)blocks), dim3(kNormBlock), 0, (hipStream_t)stream, x, workspace, n, (int)C);
    });
    hipLaunchKernelGGL(partial_sum_kernel, dim3((uint32_t)((C + 15) / 16)), dim3(256), 0, (hipStream_t)stream, workspace, out, out, blocks, (int)C,
                       (int)C);
    SGNN_HIP_CHECK(hipGetLastError());
    return SGNN_OK;
}

extern "C" int sgnn_rest_product_f32(const float *g, const float *a, float *w, int64_t rows, int64_t n_out, int64_t n_in, sgnn_stream_t stream) {
    SGNN_REQUIRE(rows >= 0 && rows < (1 << 20) && n_out > 0 && n_in > 0 && n_out < (1 << 20) && n_in < (1 << 20), "sizes out of range");
    if (rows == 0) return SGNN_OK;
    SGNN_REQUIRE(g && a && w, "null argument");
    hipLaunchKernelGGL(rest_product_kernel, dim3((uint32_t)((n_out + 63) / 64), (uint32_t)((n_in + 63) / 64)), dim3(256), 0, (hipStream_t)stream, g, a,
                       w, (int)rows, (int)n_out, (int)n_in);
    SGNN_HIP_CHECK(hipGetLastError());
    return SGNN_OK;
}
