// Device helpers that the N-D executor's matrix-core kernels share (ndconv.hip, ndblock.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "../common.h"

namespace ocr {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ inline float act_dev(float v, int act) {
    if (act == ACT_RELU) return fmaxf(v, 0.f);
    if (act == ACT_SIGMOID) return 1.f / (1.f + expf(-v));
    if (act == ACT_GELU) return 0.5f * v * (1.f + erff(v * 0.70710678118654752f));
    if (act == ACT_SILU) return v / (1.f + expf(-v));
    return v;
}

// x = hi + lo to about 2^-22.
__device__ inline void split8(const float (&v)[8], half8 &hi, half8 &lo) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const _Float16 h = (_Float16)v[j];
        hi[j] = h;
        lo[j] = (_Float16)(v[j] - (float)h);
    }
}

// Values c0 .. c0 + 7 of row `row` of x [m][k] (zeros outside). vec: k % 4 == 0 and x 16-byte
// aligned.
__device__ inline void row_chunk(const float *x, int row, int m, int k, int c0, int vec, float (&v)[8]) {
    if (row < m && vec && c0 + 8 <= k) {
        const float4 *src = reinterpret_cast<const float4 *>(x + size_t(row) * k + c0);
        const float4 q0 = src[0], q1 = src[1];
        v[0] = q0.x, v[1] = q0.y, v[2] = q0.z, v[3] = q0.w, v[4] = q1.x, v[5] = q1.y, v[6] = q1.z, v[7] = q1.w;
    } else {
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = (row < m && c0 + j < k) ? x[size_t(row) * k + c0 + j] : 0.f;
    }
}

// The same for k a multiple of 4 and x of any alignment, without a branch; rows past the last
// repeat it.
__device__ inline void row_quads(const float *x, int row, int m, int k, int c0, float (&v)[8]) {
    typedef float floatu4 __attribute__((ext_vector_type(4), aligned(4)));
    const float *src = x + size_t(min(row, m - 1)) * k;
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int c = c0 + 4 * e;
        const floatu4 q = *reinterpret_cast<const floatu4 *>(src + min(c, k - 4));
#pragma unroll
        for (int j = 0; j < 4; j++) v[4 * e + j] = c < k ? q[j] : 0.f;
    }
}

// LayerNorm of 8 values of a row: (x - mean) / sqrt(var + eps) * gamma + beta. The row's k values,
// 32 KC at most, are held by the four lanes g of a matrix operand (v[c][j] = value 32 c + 8 g + j,
// zeros past k). mine: the 8 values, gb: their gammas, with the betas `beta` values after; both
// padded with zeros (zeros past k stay zeros) and 16-byte aligned.
template <int KC>
__device__ inline void norm_chunk(const float (&v)[KC][8], float (&mine)[8], const float *gb, int beta, int k, float eps,
                                  int g) {
    const float4 *gm = reinterpret_cast<const float4 *>(gb), *bt = reinterpret_cast<const float4 *>(gb + beta);
    const float4 g0 = gm[0], g1 = gm[1], b0 = bt[0], b1 = bt[1];
    // Sums in pairs: none of them is a long chain.
    float t[8];
    auto sum = [&]() __attribute__((always_inline)) {
        return ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    };
#pragma unroll
    for (int j = 0; j < 8; j++) {
        t[j] = 0.f;
#pragma unroll
        for (int c = 0; c < KC; c++) t[j] += v[c][j];
    }
    float s = sum();
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    const float mean = s / float(k);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        t[j] = 0.f;
#pragma unroll
        for (int c = 0; c < KC; c++) {
            const float d = 32 * c + 8 * g + j < k ? v[c][j] - mean : 0.f;
            t[j] += d * d;
        }
    }
    float q = sum();
    q += __shfl_xor(q, 16);
    q += __shfl_xor(q, 32);
    const float den = sqrtf(q / float(k) + eps);
    const float gv[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
    const float bv[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
    for (int j = 0; j < 8; j++) mine[j] = (mine[j] - mean) / den * gv[j] + bv[j];
}

}  // namespace ocr
