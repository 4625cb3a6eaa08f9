// The N-D executor's transformer block pieces (the SVTR neck; src/nd.rs:222-391 runs each as a
// chain of programs) for row-major float32 tensors on gfx950. Their tensors are small (16 lines x
// 109 steps x 120 values), so a launch is a chain of latencies and every launch less is time:
//
// rows_block: y = act(norm(x) W + b) + res, or an MLP, y = act2(act1(norm(x) W1 + b1) W2 + b2) +
// res; norm is a LayerNorm or nothing. A workgroup (8 wavefronts) makes 16 rows: each of the first
// wavefronts normalises and splits one 32-value chunk into LDS (float16 hi + lo, in the order the
// products' operands are read), then every wavefront makes its 16-column tiles, whose weights it
// has asked for before the rows arrived. An MLP's hidden rows stay in LDS in the same order.
// 1744 rows, 120 -> 240 -> 120: 8.3 us against 17.5 in three launches
// (LayerNorm 3.9, 6.2, 7.4); 120 -> 360 with its LayerNorm 8.8 against 11.7. With the LayerNorm in the
// row GEMM's own wavefronts, each of which has few columns, it was done over and over (12.3 us);
// with one wavefront a SIMD the long straight code itself is the time (an MLP in 4 wavefronts: 15).
//
// attention: softmax(scale q k^T) v for heads of 4 to 16 values, a wavefront 16 queries of one
// head, in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: the heads are too short for the
// float16 instructions to win back the splitting of every operand). S^T = K Q^T takes four
// instructions a 16-key tile with the values 4 g .. 4 g + 3 of a key, one 16-byte load, in lane
// group g; a lane then holds 4 keys of one query, which is the B operand of O^T = V^T P^T as it
// stands. The softmax runs over 32 keys at a time, its sums rescaled when a group raises the
// maximum. With a projection (y = act(o W + b) + res), a workgroup takes 16 queries of every head,
// a wavefront a head (or every 8th), and the heads' outputs meet in LDS as the projection's
// operand. 16 images x 109 steps x 8 heads of 15: 13 us with the projection,
// against 15.9 + 5.2 on the vector ALU and a GEMM launch; the float16 form, splitting keys, queries,
// probabilities and values, took the same and its error was larger.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../kernels.h"
#include "../nd_kernels.h"
#include "../runtime.h"
#include "nd_device.h"

namespace ocr {

namespace {

// Weights packed by pack_conv_weights for a 1 x 1 conv, by 16-column tile.
struct PackedW {
    const half8 *hi, *lo;  // lo null when the weights are float16 values
    const float *bias;
    int bn, chunks, tiles;  // tiles: 16-column tiles that hold a column
    int n, act;
};
__device__ inline size_t tile_at(const PackedW &w, int tile, int c, int r, int g) {
    const int tb = w.bn >> 4, nb = tile / tb;
    return size_t(nb * w.chunks + c) * (w.bn * 4) + (tile - nb * tb) * 64 + r * 4 + g;
}

// What an output tile adds, for columns n .. n + 3 of a row: asked for before the products.
struct Adds {
    float b[4], r[4];
};
__device__ inline void load_adds(Adds &a, const PackedW &w, const float *res, size_t row, int n) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int c = min(n + k, w.n - 1);
        a.b[k] = w.bias ? w.bias[c] : 0.f;
        a.r[k] = res ? res[row * w.n + c] : 0.f;
    }
}
// act(acc + b) + res. acc: the sums of the hi and of the lo products (apart: half as many
// roundings in the large sum).
__device__ inline void put4(const floatx4 &hi, const floatx4 &lo, const Adds &a, const PackedW &w, bool res, float *y, size_t row,
                            int n) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = act_dev(hi[k] + lo[k] + a.b[k], w.act);
        if (res) v[k] += a.r[k];
    }
    float *dst = y + row * w.n + n;
    if ((w.n & 3) == 0 && n + 4 <= w.n) {
        *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (n + k < w.n) dst[k] = v[k];
    }
}

// ---- rows_block ------------------------------------------------------------------------------
struct BlockParams {
    const float *x, *gb, *res;
    float *y;
    float eps;
    int m, k;
    PackedW w1, w2;
};

constexpr int C1 = 4, C2 = 8;  // 32-wide chunks of the inputs and of an MLP's hidden values, at most

// MLP: w2 follows w1. LO: some weights are not float16 values.
template <bool MLP, bool LO>
__global__ __launch_bounds__(512) void rows_block_kernel(BlockParams p) {
    __shared__ __align__(16) _Float16 x_h[C1][16][32], x_l[C1][16][32];
    __shared__ __align__(16) _Float16 s_h[MLP ? C2 : 1][16][32], s_l[MLP ? C2 : 1][16][32];
    constexpr int T = MLP ? 2 : 3;  // tiles a wavefront has in flight
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int row = blockIdx.x * 16 + r;
    half8 a1[T][C1], a2[MLP ? C2 : 1];
    Adds d1[T], d2;
    const size_t arow = size_t(min(row, p.m - 1));
    auto load1 = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int c = 0; c < C1; c++)
                a1[t][c] = p.w1.hi[tile_at(p.w1, min(t0 + wave + 8 * t, p.w1.tiles - 1), min(c, p.w1.chunks - 1), r, g)];
#pragma unroll
        for (int t = 0; t < T; t++) load_adds(d1[t], p.w1, MLP ? nullptr : p.res, arow, (t0 + wave + 8 * t) * 16 + 4 * g);
    };
    auto load2 = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < C2; c++) a2[c] = p.w2.hi[tile_at(p.w2, min(tile, p.w2.tiles - 1), min(c, p.w2.chunks - 1), r, g)];
        load_adds(d2, p.w2, p.res, arow, tile * 16 + 4 * g);
    };
    load1(0);
    if constexpr (MLP) load2(wave);
    if (wave < p.w1.chunks) {
        float v[C1][8];
#pragma unroll
        for (int c = 0; c < C1; c++) row_quads(p.x, row, p.m, p.k, c * 32 + 8 * g, v[c]);
        float mine[8];
#pragma unroll
        for (int j = 0; j < 8; j++) mine[j] = wave == 0 ? v[0][j] : wave == 1 ? v[1][j] : wave == 2 ? v[2][j] : v[3][j];
        if (p.gb) norm_chunk<C1>(v, mine, p.gb + 32 * wave + 8 * g, 32 * p.w1.chunks, p.k, p.eps, g);
        half8 hi, lo;
        split8(mine, hi, lo);
        *reinterpret_cast<half8 *>(&x_h[wave][r][8 * g]) = hi;
        *reinterpret_cast<half8 *>(&x_l[wave][r][8 * g]) = lo;
    }
    __syncthreads();
    for (int t0 = 0; t0 < p.w1.tiles; t0 += 8 * T) {
        if (t0) load1(t0);
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int tile = t0 + wave + 8 * t;
            if (tile >= (MLP ? 2 * p.w2.chunks : p.w1.tiles)) break;
            floatx4 acc = {0.f, 0.f, 0.f, 0.f}, accl = acc;
#pragma unroll
            for (int c = 0; c < C1; c++) {
                if (c >= p.w1.chunks) break;
                const half8 bh = *reinterpret_cast<const half8 *>(&x_h[c][r][8 * g]);
                const half8 bl = *reinterpret_cast<const half8 *>(&x_l[c][r][8 * g]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1[t][c], bh, acc, 0, 0, 0);
                accl = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1[t][c], bl, accl, 0, 0, 0);
                if constexpr (LO) {
                    if (p.w1.lo)
                        accl = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            p.w1.lo[tile_at(p.w1, min(tile, p.w1.tiles - 1), c, r, g)], bh, accl, 0, 0, 0);
                }
            }
            if constexpr (!MLP) {
                if (row < p.m) put4(acc, accl, d1[t], p.w1, p.res != nullptr, p.y, size_t(row), tile * 16 + 4 * g);
            } else {
                // Columns 4 g .. 4 g + 3 of the tile for row r: inputs 16 (tile & 1) + 4 g .. of chunk
                // tile / 2 of the second product; columns past the last are zeros.
                _Float16 hi[4], lo[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int n = tile * 16 + 4 * g + k;
                    const float h = n < p.w1.n ? act_dev(acc[k] + accl[k] + d1[t].b[k], p.w1.act) : 0.f;
                    hi[k] = (_Float16)h;
                    lo[k] = (_Float16)(h - (float)hi[k]);
                }
                uint2 qh, ql;
                __builtin_memcpy(&qh, hi, 8);
                __builtin_memcpy(&ql, lo, 8);
                *reinterpret_cast<uint2 *>(&s_h[tile >> 1][r][(tile & 1) * 16 + 4 * g]) = qh;
                *reinterpret_cast<uint2 *>(&s_l[tile >> 1][r][(tile & 1) * 16 + 4 * g]) = ql;
            }
        }
    }
    if constexpr (MLP) {
        __syncthreads();
        for (int tile = wave; tile < p.w2.tiles; tile += 8) {
            if (tile != wave) load2(tile);
            floatx4 acc = {0.f, 0.f, 0.f, 0.f}, accl = acc;
#pragma unroll
            for (int c = 0; c < C2; c++) {
                if (c >= p.w2.chunks) break;
                const half8 hh = *reinterpret_cast<const half8 *>(&s_h[c][r][8 * g]);
                const half8 hl = *reinterpret_cast<const half8 *>(&s_l[c][r][8 * g]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a2[c], hh, acc, 0, 0, 0);
                accl = __builtin_amdgcn_mfma_f32_16x16x32_f16(a2[c], hl, accl, 0, 0, 0);
                if constexpr (LO) {
                    if (p.w2.lo)
                        accl = __builtin_amdgcn_mfma_f32_16x16x32_f16(p.w2.lo[tile_at(p.w2, tile, c, r, g)], hh, accl, 0, 0, 0);
                }
            }
            if (row < p.m) put4(acc, accl, d2, p.w2, p.res != nullptr, p.y, size_t(row), tile * 16 + 4 * g);
        }
    }
}

// ---- attention -------------------------------------------------------------------------------
struct AttnParams {
    const float *x, *res;
    float *y;
    int n, t, heads, d, qtiles;
    float scale;
    PackedW w;  // the projection
};

typedef float floatu4 __attribute__((ext_vector_type(4), aligned(4)));

// One 32-key group as it is loaded: values of this lane's keys 16 u + r, and value r of keys
// 16 u + 4 g + i.
struct KeyGroup {
    floatu4 k[2];
    float v[2][4];
};

// A wavefront's 16 queries of one head: o[i] = output value 4 g + i of query r. Queries past t
// repeat the last.
__device__ inline void attend(const AttnParams &p, int img, int h, int q0, int r, int g, float (&o)[4]) {
    const int hd = p.heads * p.d;
    const unsigned row = 3u * unsigned(hd);
    const float *base = p.x + size_t(img) * p.t * row + size_t(h) * p.d;
    // Lane group g holds values at .. at + 3 of a head: its values in order, but the quadruple that
    // would end past the head starts 4 before its end (and any after it), and the values it then
    // repeats are zeros on both sides (a zero on one does not cancel an infinity on the other).
    // Nothing outside the head is read.
    const int at = min(4 * g, p.d - 4), vr = min(r, p.d - 1);
    const int fresh = 4 * g - at;  // the first value of the quadruple that is not a repeated one
    // 32-bit offsets from the group's first key (an image holds fewer than 2^31 values,
    // nd_attention_mfma_fits); keys past the last read the group's first, and their values and probabilities are
    // made zeros.
    unsigned ko[2], vo[2][4];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        ko[u] = unsigned(16 * u + r) * row;
#pragma unroll
        for (int i = 0; i < 4; i++) vo[u][i] = unsigned(16 * u + 4 * g + i) * row;
    }
    auto load = [&](KeyGroup &kg, int k0) __attribute__((always_inline)) {
        const float *first = base + size_t(k0) * row;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            kg.k[u] = *reinterpret_cast<const floatu4 *>(first + hd + at + (k0 + 16 * u + r < p.t ? ko[u] : 0u));
#pragma unroll
            for (int i = 0; i < 4; i++) kg.v[u][i] = (first + 2 * hd + vr)[k0 + 16 * u + 4 * g + i < p.t ? vo[u][i] : 0u];
        }
    };
    constexpr int AHEAD = 2;
    KeyGroup kg[AHEAD];
    const floatu4 q4 = *reinterpret_cast<const floatu4 *>(base + size_t(min(q0 + r, p.t - 1)) * row + at);
#pragma unroll
    for (int a = 0; a < AHEAD; a++)
        if (32 * a < p.t) load(kg[a], 32 * a);
    __builtin_amdgcn_sched_barrier(0);
    float q[4];
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = i >= fresh ? q4[i] * p.scale : 0.f;
    // Four partial sums of the output and of l, so that no sum is a long chain.
    float m = -INFINITY, l[2][2];
    floatx4 acc[2][2];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            l[u][i] = 0.f;
            acc[u][i] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    for (int kb = 0; kb < p.t; kb += 32 * AHEAD) {
#pragma unroll
        for (int a = 0; a < AHEAD; a++) {
            const int k0 = kb + 32 * a;
            if (k0 >= p.t) break;
            float s[2][4], v[2][4];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                floatx4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4; i++)
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(i >= fresh ? kg[a].k[u][i] : 0.f, q[i], c, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    s[u][i] = c[i];
                    v[u][i] = kg[a].v[u][i];
                }
            }
            if (k0 + 32 > p.t) {
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (k0 + 16 * u + 4 * g + i >= p.t) s[u][i] = -INFINITY, v[u][i] = 0.f;
            }
            if (k0 + 32 * AHEAD < p.t) load(kg[a], k0 + 32 * AHEAD);
            float mt = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                             fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
            mt = fmaxf(mt, __shfl_xor(mt, 16));
            mt = fmaxf(mt, __shfl_xor(mt, 32));
            const float mn = fmaxf(m, mt);
            // While every score is -inf the exponents are taken from 0: weights of 0, not of NaN.
            const float m0 = mn == -INFINITY ? 0.f : mn;
            if (k0 && __any(mn > m)) {
                const float f = m == -INFINITY ? 0.f : expf(m - mn);
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        l[u][i] *= f;
#pragma unroll
                        for (int k = 0; k < 4; k++) acc[u][i][k] *= f;
                    }
            }
            m = mn;
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float e = expf(s[u][i] - m0);
                    l[u][i & 1] += e;
                    acc[u][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[u][i], e, acc[u][i & 1], 0, 0, 0);
                }
        }
    }
    float ls = (l[0][0] + l[0][1]) + (l[1][0] + l[1][1]);
    ls += __shfl_xor(ls, 16);
    ls += __shfl_xor(ls, 32);
#pragma unroll
    for (int i = 0; i < 4; i++)
        o[i] = ((acc[0][0][i] + acc[0][1][i]) + (acc[1][0][i] + acc[1][1][i])) / ls;
}

__global__ __launch_bounds__(256) void attention_kernel(AttnParams p) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int h = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int img = blockIdx.x / p.qtiles, q0 = (blockIdx.x - img * p.qtiles) * 16;
    if (h >= p.heads) return;
    float o[4];
    attend(p, img, h, q0, r, g, o);
    if (q0 + r >= p.t) return;
    float *dst = p.y + (size_t(img) * p.t + q0 + r) * (p.heads * p.d) + size_t(h) * p.d;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (4 * g + i < p.d) dst[4 * g + i] = o[i];
}

constexpr int PROJ_C = 8;  // 32-wide input chunks of the projection, at most

// 8 wavefronts at most, each every 8th head (or as many wavefronts as heads).
template <bool LO>
__global__ __launch_bounds__(512) void attention_proj_kernel(AttnParams p) {
    __shared__ __align__(16) _Float16 s_h[PROJ_C][16][32], s_l[PROJ_C][16][32];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = int(blockDim.x >> 6);
    const int img = blockIdx.x / p.qtiles, q0 = (blockIdx.x - img * p.qtiles) * 16;
    const int hd = p.heads * p.d;
    // The operand's columns past the last value.
    for (int i = hd + int(threadIdx.x >> 4); i < p.w.chunks * 32; i += int(blockDim.x >> 4)) {
        s_h[i >> 5][threadIdx.x & 15][i & 31] = (_Float16)0.f;
        s_l[i >> 5][threadIdx.x & 15][i & 31] = (_Float16)0.f;
    }
    // The first tile's weights are on their way during the attention.
    half8 a[PROJ_C];
    Adds add;
    const size_t row = size_t(img) * p.t + min(q0 + r, p.t - 1);
    auto load = [&](int tile) __attribute__((always_inline)) {
        load_adds(add, p.w, p.res, row, tile * 16 + 4 * g);
#pragma unroll
        for (int c = 0; c < PROJ_C; c++) a[c] = p.w.hi[tile_at(p.w, min(tile, p.w.tiles - 1), min(c, p.w.chunks - 1), r, g)];
    };
    load(wave);
    for (int h = wave; h < p.heads; h += waves) {
        float o[4];
        attend(p, img, h, q0, r, g, o);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (4 * g + i >= p.d) break;
            const int c = h * p.d + 4 * g + i;
            const _Float16 hi = (_Float16)o[i];
            s_h[c >> 5][r][c & 31] = hi;
            s_l[c >> 5][r][c & 31] = (_Float16)(o[i] - (float)hi);
        }
    }
    __syncthreads();
    for (int tile = wave; tile < p.w.tiles; tile += waves) {
        if (tile != wave) load(tile);
        floatx4 acc = {0.f, 0.f, 0.f, 0.f}, accl = acc;
#pragma unroll
        for (int c = 0; c < PROJ_C; c++) {
            if (c >= p.w.chunks) break;
            const half8 hh = *reinterpret_cast<const half8 *>(&s_h[c][r][8 * g]);
            const half8 hl = *reinterpret_cast<const half8 *>(&s_l[c][r][8 * g]);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c], hh, acc, 0, 0, 0);
            accl = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c], hl, accl, 0, 0, 0);
            if constexpr (LO) {
                accl = __builtin_amdgcn_mfma_f32_16x16x32_f16(p.w.lo[tile_at(p.w, tile, c, r, g)], hh, accl, 0, 0, 0);
            }
        }
        if (q0 + r < p.t) put4(acc, accl, add, p.w, p.res != nullptr, p.y, row, tile * 16 + 4 * g);
    }
}

PackedW packed(const NdRowsArgs &a) {
    PackedW w{};
    w.hi = reinterpret_cast<const half8 *>(a.wt_hi);
    w.lo = a.pk.exact ? nullptr : reinterpret_cast<const half8 *>(a.wt_lo);
    w.bias = a.bias;
    w.bn = a.pk.bn;
    w.chunks = a.pk.chunks;
    w.tiles = (a.n + 15) / 16;
    w.n = a.n;
    w.act = a.act;
    return w;
}

double weight_bytes(const NdRowsArgs &a) { return 2.0 * double(a.pk.halves()) * (a.pk.exact ? 1 : 2); }

}  // namespace

bool nd_rows_fit(const ConvPack &w1) { return w1.kh == 1 && w1.kw == 1 && w1.chunks <= C1 && w1.cin % 4 == 0; }
bool nd_mlp_fits(const ConvPack &w1, const ConvPack &w2) {
    return nd_rows_fit(w1) && w2.kh == 1 && w2.kw == 1 && w2.chunks <= C2 && w1.cout == w2.cin;
}

void nd_rows_block(const NdRowsArgs &a, const NdRowsArgs *b, hipStream_t s) {
    if (!nd_rows_fit(a.pk) || a.pk.cin != a.k || a.pk.cout != a.n) fail("nd_rows_block: shapes");
    if (b && (!nd_mlp_fits(a.pk, b->pk) || b->k != a.n || b->pk.cout != b->n || b->m != a.m || a.res)) fail("nd_rows_block: shapes");
    if (a.m <= 0) return;
    BlockParams p{};
    p.x = a.x;
    p.gb = a.gb;
    p.eps = a.eps;
    p.m = a.m;
    p.k = a.k;
    p.res = b ? b->res : a.res;
    p.y = b ? b->y : a.y;
    p.w1 = packed(a);
    if (b) p.w2 = packed(*b);
    ProbeScope probe("nd_gemm_rows", s, 2.0 * a.m * (double(a.k) * a.n + (b ? double(b->k) * b->n : 0.0)),
                     4.0 * a.m * (double(a.k) + (b ? b->n : a.n)) + weight_bytes(a) + (b ? weight_bytes(*b) : 0.0),
                     b ? "nd_mlp" : "nd_rows_norm");
    const dim3 grid{unsigned((a.m + 15) / 16)};
    const bool lo = p.w1.lo || p.w2.lo;
    if (b && lo) hipLaunchKernelGGL((rows_block_kernel<true, true>), grid, dim3(512), 0, s, p);
    else if (b) hipLaunchKernelGGL((rows_block_kernel<true, false>), grid, dim3(512), 0, s, p);
    else if (lo) hipLaunchKernelGGL((rows_block_kernel<false, true>), grid, dim3(512), 0, s, p);
    else hipLaunchKernelGGL((rows_block_kernel<false, false>), grid, dim3(512), 0, s, p);
    OCR_HIP(hipGetLastError());
}

bool nd_attention_proj_fits(int n, int t, int heads, int d, const ConvPack &pk) {
    return nd_attention_mfma_fits(n, t, heads, d) && pk.kh == 1 && pk.kw == 1 && pk.cin == heads * d && pk.chunks <= PROJ_C;
}

static AttnParams attn_params(const float *x, int n, int t, int heads, int d, float scale, float *y) {
    AttnParams p{};
    p.x = x;
    p.y = y;
    p.n = n;
    p.t = t;
    p.heads = heads;
    p.d = d;
    p.scale = scale;
    p.qtiles = (t + 15) / 16;
    return p;
}

void nd_attention_proj(const float *x, int n, int t, int heads, int d, float scale, const NdRowsArgs &w, hipStream_t s) {
    if (n <= 0 || t <= 0) return;
    if (!nd_attention_proj_fits(n, t, heads, d, w.pk) || w.k != heads * d || w.pk.cout != w.n) fail("nd_attention_proj: shapes");
    AttnParams p = attn_params(x, n, t, heads, d, scale, w.y);
    p.res = w.res;
    p.w = packed(w);
    const double tt = double(t), m = double(n) * t;
    ProbeScope probe("nd_attention", s, 4.0 * n * heads * tt * tt * d + 2.0 * m * w.k * w.n,
                     4.0 * m * (3.0 * w.k + w.n) + weight_bytes(w), "nd_attention_proj");
    const dim3 grid{unsigned(n * p.qtiles)}, block{unsigned(64 * std::min(heads, 8))};
    if (p.w.lo) hipLaunchKernelGGL((attention_proj_kernel<true>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((attention_proj_kernel<false>), grid, block, 0, s, p);
    OCR_HIP(hipGetLastError());
}

bool nd_attention_mfma(const float *x, int n, int t, int heads, int d, float scale, float *y, hipStream_t s) {
    if (!nd_attention_mfma_fits(n, t, heads, d)) return false;
    if (n <= 0 || t <= 0) return true;
    const AttnParams p = attn_params(x, n, t, heads, d, scale, y);
    const double tt = double(t);
    ProbeScope probe("nd_attention", s, 4.0 * n * heads * tt * tt * d, 4.0 * n * tt * (3.0 * heads * d + heads * d),
                     "nd_attention_mfma");
    hipLaunchKernelGGL(attention_kernel, dim3(unsigned(n * p.qtiles), unsigned((heads + 3) / 4)), dim3(256), 0, s, p);
    OCR_HIP(hipGetLastError());
    return true;
}

}  // namespace ocr
