// Launchers of the N-D executor's kernels (kernels/nd.hip, kernels/bgemm.hip). Row-major
// (ONNX) float32 tensors.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "common.h"
#include "kernels.h"

namespace ocr {

constexpr int ND_RANK = 6;

// An index space of up to ND_RANK dimensions with two stride sets (in elements): for the copy,
// input and output strides; for a broadcast binary op, the strides of a and b (0 on a
// broadcast dimension).
struct NdIndex {
    size_t total = 0;
    int rank = 0;
    size_t dims[ND_RANK] = {};
    size_t s0[ND_RANK] = {}, s1[ND_RANK] = {};
};

enum UnaryOp : int { UN_RELU = 1, UN_SIGMOID = 2, UN_HARDSIGMOID = 3, UN_ERF = 4, UN_SQRT = 5 };
enum BinaryOp : int { BIN_ADD = 0, BIN_SUB = 1, BIN_MUL = 2, BIN_DIV = 3, BIN_POW = 4 };

void nd_unary(const float *x, float *y, size_t n, int op, float alpha, float beta, hipStream_t s);
void nd_binary(const float *a, const float *b, float *y, const NdIndex &ix, int op, hipStream_t s);
void nd_copy(const float *x, float *y, const NdIndex &ix, size_t ibase, size_t obase, hipStream_t s);
// y = x * st[c] + st[C + c], c = (i / inner) % C (BatchNormalization folded, nd.rs:788-800).
void nd_affine(const float *x, const float *st, float *y, size_t total, int c, size_t inner, hipStream_t s);
void nd_reduce_mean(const float *x, float *y, size_t rows, int len, hipStream_t s);
// gb: gamma[len] then beta[len].
void nd_layer_norm(const float *x, const float *gb, float *y, size_t rows, int len, float eps, hipStream_t s);
void nd_softmax(const float *x, float *y, size_t rows, int len, hipStream_t s);
// Arg-max per row, the first index on ties (src/nd.rs:383).
void nd_argmax(const float *x, uint32_t *best, size_t rows, int len, hipStream_t s);
// Reduces [rows][parts] (value, index-as-bits) pairs to the row's arg-max (first index on ties).
void nd_argmax_partials(const float *part, int parts, size_t rows, uint32_t *best, hipStream_t s);
void nd_pool(const float *x, float *y, size_t nc, int h, int w, int oh, int ow, int kh, int kw, int sh, int sw,
             int pt, int pl, bool avg, hipStream_t s);
void nd_resize_nearest(const float *x, float *y, size_t nc, int h, int w, int oh, int ow, float sy, float sx,
                       hipStream_t s);

// A Conv in NCHW on the general kernel (strided, grouped, depthwise). Epilogue:
// act(affine(acc + b)) + res, with in_scale[n][cin] applied to the input first (the SE gate).
struct NdConvArgs {
    const float *x = nullptr;
    int n = 0, cin = 0, h = 0, w = 0;
    const float *wt = nullptr;  // [cout][cin / group][kh][kw]
    const float *b = nullptr;
    const float *affine = nullptr;    // scale[cout] then shift[cout], or null
    const float *res = nullptr;       // [n][cout][oh][ow], or null
    const float *in_scale = nullptr;  // [n][cin], or null
    float *y = nullptr;
    int cout = 0, oh = 0, ow = 0, kh = 0, kw = 0, sh = 1, sw = 1, pt = 0, pl = 0, group = 1, act = 0;
};
void nd_conv_generic(const NdConvArgs &a, hipStream_t s);
// Depthwise (group = cin = cout, 3 x 3 or 5 x 5, strides 1 or 2 per axis; no residual or input
// scale), the taps summed as nd_conv_generic sums them. False (nothing launched) otherwise.
bool nd_conv_dw(const NdConvArgs &a, hipStream_t s);
// Group 1, 3 x 3, one or three input channels, at most 64 output channels, any stride (the
// stems): one thread an output pixel. False (nothing launched) otherwise.
bool nd_conv_small(const NdConvArgs &a, hipStream_t s);

// A group-1, stride-1 conv up to 3 x 3 in NCHW on the matrix cores (kernels/ndconv.hip), with
// the weights packed by pack_conv_weights: act(affine(acc + b)) + res, in_scale[n][cin] applied to
// the input first. False (nothing launched) for shapes it does not take.
constexpr int ND_SOURCES = 4;
struct NdMfmaConvArgs {
    const float *x = nullptr;
    int n = 0, cin = 0, h = 0, w = 0;
    float *y = nullptr;
    int cout = 0, oh = 0, ow = 0;
    const uint16_t *wt_hi = nullptr, *wt_lo = nullptr;
    ConvPack pk;
    const float *bias = nullptr, *affine = nullptr, *res = nullptr, *in_scale = nullptr;
    int pt = 0, pl = 0, act = ACT_NONE;
    int res_up = 0;             // res is [n][cout][oh >> res_up][ow >> res_up], upscaled (nearest) as it is read
    const float *x2 = nullptr;  // channels c1 .. of the input ([n][cin - c1][h][w], x then has c1), c1 % 32 == 0
    int c1 = 0;
};
// Channels c0 .. c0 + c - 1 of a conv's input: [n][c][h][w], upscaled (nearest) by 2^up as read.
struct NdConvSource {
    const float *p;
    int c0, c, h, w, up;
};
// 3 x 3, pad 1 over images of many rows (kernels/ndconv3.hip), the input a.x or the nsrc sources
// in order (c0 is set here), each from a multiple of 8 channels. saves: the sources would be written
// out as several parts if it did not take them. False (nothing launched) for what it does not take:
// few tiles or pixels, tiles mostly outside the image, x2, res_up, in_scale.
bool nd_conv_tile(const NdMfmaConvArgs &a, const NdConvSource *src, int nsrc, bool saves, hipStream_t s);
bool nd_conv_nchw_mfma(const NdMfmaConvArgs &a, hipStream_t s);

// y [m][n] = act(x [m][k] W + b) (+ res [m][n]) with W packed as n rows of k (pack_conv_weights,
// 1 x 1), on the matrix cores. False (nothing launched) for packs it does not take.
struct NdRowsArgs {
    const float *x = nullptr;
    int m = 0, k = 0, n = 0;
    const uint16_t *wt_hi = nullptr, *wt_lo = nullptr;
    ConvPack pk;
    const float *bias = nullptr, *res = nullptr;
    float *y = nullptr;
    int act = ACT_NONE;
    // LayerNorm of x's rows first (nd_rows_block): gamma, then beta, each padded with zeros to a
    // multiple of 32; or null.
    const float *gb = nullptr;
    float eps = 0.f;
};
bool nd_gemm_rows(const NdRowsArgs &a, hipStream_t s);
// a, which may have a LayerNorm, and if b is given b applied to the rows that a gives, which are
// then never written (kernels/ndblock.hip). Packs that fit: at most 128 inputs, a multiple of 4,
// and with b at most 256 hidden values.
bool nd_rows_fit(const ConvPack &w1);
bool nd_mlp_fits(const ConvPack &w1, const ConvPack &w2);
// Whether a joined step of m rows is worth one launch, against one each. n: the columns it gives,
// from k inputs with a LayerNorm first (norm) and hidden columns between (0: no second product; an
// attention's projection has neither).
//
// Few rows fill the chip only by their columns, which a joined workgroup walks 384 (an MLP: 128) at a
// time: 17 and 109 rows, 120 -> n with its LayerNorm, take 12 us for n = 720 against 13.5 apart, 14.7
// against 13.8 for 960, 51 against 13.6 for 6000; at 1744 rows n = 1440 is 23 against 25 and 6000 58
// against 49, at 8000 rows 6000 119 against 176. An attention's projection of 109 rows: 13.2 against
// 19.1 for n = 120, 19.8 against 19.2 for 768; of 1744 rows 28 against 33 for 1200 and 76 against 60 for
// 6000.
// Many rows take 16 to a workgroup whose start is most of its time when it makes few products (work: the
// columns of both products, and the LayerNorm's): work 152 20.0 us against 19.6 at 12 000 rows, 184 22.5
// against 23.6 at 16 000 and 31.2 against 25.5 at 24 000, 240 25.8 against 26.9 at 16 000 and 35.8
// against 32.7 at 24 000, 64 (k = 32) 12 against 13 at 8000 and 20 against 16 at 16 000; 360 is faster at
// every size (100 000 rows 136 against 153).
inline bool nd_block_pays(double m, double k, double hidden, double n, bool norm) {
    const double work = n + hidden + (norm ? k : 0);
    const bool joined_rows = norm || hidden;
    return (n <= 720 || m >= n) && (!joined_rows || m <= 8000 || m <= 75 * work || work >= 320);
}
void nd_rows_block(const NdRowsArgs &a, const NdRowsArgs *b, hipStream_t s);
// The CTC head without its logits: per row of x, nd_head_parts partial (max, index bits) pairs of
// x W + b (first index on ties) at part[row * parts + j], for nd_argmax_partials. Needs 64-column
// blocks and k <= 256. False (nothing launched) otherwise.
int nd_head_parts(int m, const ConvPack &pk);
bool nd_head_argmax(const NdRowsArgs &a, float *part, int parts, hipStream_t s);

// ConvTranspose, group 1, no pads; wt is ONNX's [cin][cout][kh][kw].
void nd_conv_transpose(const float *x, int n, int cin, int h, int w, const float *wt, const float *b, float *y,
                       int cout, int kh, int kw, int stride, int act, hipStream_t s);
// The PP-OCR detection input: RGB bytes (h x w x 3) -> [1][3][oh][ow], bilinear half-pixel,
// BGR, ImageNet mean / deviation (src/nd.rs:172-204).
void nd_det_prep(const uint8_t *rgb, int w, int h, float *y, int ow, int oh, hipStream_t s);
// prob > thr as bit rows: h rows of ceil(w / 32) words, bit x % 32 of word x / 32.
void nd_threshold_bits(const float *prob, int w, int h, float thr, uint32_t *bits, hipStream_t s);

// Multi-head self-attention from a fused QKV projection: x [n][t][3 heads d] (q, k, v blocks of
// heads x d), y[i][j][h d + c] = sum_k softmax_k(scale q_j . k_k) v_k[c] (kernels/attn.hip).
void nd_attention(const float *x, int n, int t, int heads, int d, float scale, float *y, hipStream_t s);
// The same on the matrix cores, for heads of 4 to 16 values (kernels/ndblock.hip). False
// (nothing launched) otherwise.
bool nd_attention_mfma(const float *x, int n, int t, int heads, int d, float scale, float *y, hipStream_t s);
// Its grid and its 32-bit offsets within an image.
inline bool nd_attention_mfma_fits(int n, int t, int heads, int d) {
    return d >= 4 && d <= 16 && heads >= 1 && heads <= 4 * 65535 && double(n) * ((double(t) + 15) / 16) <= 0x7fffffff &&
           double(t) * 3.0 * heads * d <= 0x7fffffff;
}
// And with the projection w of its rows (w.x unused, w.m = n t), whose input is never written:
// heads of 4 to 16 values, 256 values in all.
bool nd_attention_proj_fits(int n, int t, int heads, int d, const ConvPack &pk);
void nd_attention_proj(const float *x, int n, int t, int heads, int d, float scale, const NdRowsArgs &w, hipStream_t s);

// Batched C[b] = A[b] (M x K) * B[b] (K x N) on the matrix cores, both operands float32 split
// into float16 hi + lo (three passes: hi*hi, hi*lo, lo*hi), float32 accumulation. Element
// (m, k) of batch b of A is at a[b * sab + m * sam + k * sak]; likewise B and C.
struct BgemmArgs {
    const float *a = nullptr, *b = nullptr;
    float *c = nullptr;
    int batch = 0, m = 0, n = 0, k = 0;
    size_t sab = 0, sam = 0, sak = 0, sbb = 0, sbk = 0, sbn = 0, scb = 0, scm = 0, scn = 0;
};
void nd_bgemm(const BgemmArgs &g, hipStream_t s);

}  // namespace ocr
