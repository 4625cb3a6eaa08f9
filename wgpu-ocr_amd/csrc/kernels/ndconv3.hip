// 3 x 3, pad 1, stride 1 convolution of row-major (NCHW) float32 tensors on gfx950, for images of
// many rows (the DB detector's heads; src/nd.rs:222-358). The input may be up to four tensors,
// channels after channels, each a nearest-neighbour upscaling of a smaller one: what a Concat of
// Resizes would write and this kernel would read back is read from its source instead.
//
// conv_nchw (ndconv.hip) reads every operand from memory for every tap: 72 four-byte loads a lane
// for 8 channels of 16 pixels, which bound it. Here a workgroup's tile (8 rows x 32 columns) takes
// its halo of 32 channels into LDS once, split into float16 hi + lo (x = hi + lo to about 2^-22),
// 8 channels of a pixel a 16-byte unit, and the nine taps read units. A wavefront makes 2 rows,
// 4 tiles of 16 pixels x 16 NT channels; its weights come from L2. Unit (pixel, part q) lies at
// 4 pixel + (q ^ (pixel / 4 % 4)): 16 neighbouring pixels' parts fall in different banks.
// Four pages at 240 x 184, 64 -> 16 channels: 77 -> 23-25 us, and the two Resizes, the Concat's four
// copies (149 us of a pass) go. Every load of a step is issued before the first value is looked at:
// with the masking next to each load the compiler waited load by load (40 us, also on 64 tiles).
#include <hip/hip_runtime.h>

#include "../kernels.h"
#include "../nd_kernels.h"
#include "../runtime.h"
#include "nd_device.h"

namespace ocr {

namespace {

// A Concat's parts are read in place from this many workgroups on: written out first, they cost a
// launch each. Below, CUs without a tile cost more.
constexpr double PART_BLOCKS = 64;
// Any other input, which conv_nchw reads as it is: from this many pixels on (counted once a block of
// output channels). conv_nchw splits smaller launches' K steps; its time grows with its rows of 16
// pixels, which more wavefronts hide up to about 32 000 pixels, and the tile's with its K steps and
// its stores (8-byte aligned rows leave as single floats). us, conv_nchw against tiles:
//   32 -> 32 channels: 160-pixel rows 28 160 pixels 14.1 and 14.1, 34 560 17.8 and 14.4; 46-pixel rows
//   27 600 15.2 and 18.0, 33 120 18.7 and 18.4. 128 -> 64: 27 600 44.7 and 52.3, 33 120 59.2 and 53.1. 256 ->
//   64: 27 600 78 and 78, 33 120 106 and 80. 64 -> 128 (two blocks): 28 160 24.3 and 25.8, 33 120 35.6 and 34.6.
//   64 -> 64: 160-pixel rows 28 160 25.1 and 28.2, 34 560 33.3 and 30.8; rows of 190 41 040 36.8 and 40.2,
//   53 200 43.7 and 42.2.
//   16 channels a block: 64 -> 16 13 800 13.8 and 16.0, 16 560 16.4 and 16.0, 22 080 17.5 and 16.2; 16 -> 16
//   22 800 12.1 and 12.6, 27 600 13.4 and 12.8.
double plain_pixels(int bn, int cin, int w) {
    if (bn == 16) return cin >= 64 ? 16500 : 24000;
    return bn == 64 && cin <= 64 && w % 4 ? 50000 : 32000;
}

constexpr int TH = 8, TW = 32, HW = TW + 2, HPX = (TH + 2) * HW, ITEMS = HPX * 4, NI = 3;

struct TileParams {
    NdConvSource src[ND_SOURCES];
    int nsrc;
    float *y;
    const half8 *wt, *wt_lo;  // [nblock][chunk][tap][bn][32] float16 (hi; lo when not exact)
    const float *bias, *affine, *res;
    int cin, h, w, cout, bn, chunks, act, tiles_x, tiles_y;
};

template <int NT, bool LO>
__global__ __launch_bounds__(256, NT <= 2 ? 3 : 2) void conv_tile_kernel(TileParams p) {
    __shared__ __align__(16) half8 s_hi[ITEMS], s_lo[ITEMS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int nb = blockIdx.y;
    const int per = p.tiles_x * p.tiles_y, img = blockIdx.x / per, tb = blockIdx.x - img * per;
    const int ty = tb / p.tiles_x, y0 = ty * TH, x0 = (tb - ty * p.tiles_x) * TW;
    // Row 2 wave + m / 2, columns 16 (m % 2) ..; the lo products' sums apart.
    floatx4 acc[4][NT], accl[4][NT];
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[m][t] = accl[m][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int chunk = 0; chunk < p.chunks; chunk++) {
        if (chunk) __syncthreads();
        // Item i of the halo: 8 channels (part i / HPX of the chunk) of pixel i % HPX; NI items' loads
        // go out together.
#pragma unroll 1
        for (int i0 = tid; i0 < ITEMS; i0 += 256 * NI) {
            float v[NI][8];
            int left[NI];  // channels from the item's first to its source's last (0: outside)
#pragma unroll
            for (int u = 0; u < NI; u++) {
                const int i = i0 + 256 * u, q = i / HPX, px = i - q * HPX;
                const int hy = px / HW, iy = y0 + hy - 1, ix = x0 + px - hy * HW - 1;
                const int c = chunk * 32 + 8 * q;
                const bool in = i < ITEMS && iy >= 0 && iy < p.h && ix >= 0 && ix < p.w && c < p.cin;
                NdConvSource s = p.src[0];
                if (p.nsrc > 1) {
#pragma unroll
                    for (int k = 1; k < ND_SOURCES; k++)
                        if (k < p.nsrc && c >= p.src[k].c0) s = p.src[k];
                }
                const unsigned plane = unsigned(s.h) * unsigned(s.w);
                const float *base = s.p + size_t(img) * s.c * plane;
                left[u] = in ? s.c - (c - s.c0) : 0;
                unsigned at = in ? unsigned(c - s.c0) * plane + unsigned(iy >> s.up) * unsigned(s.w) + unsigned(ix >> s.up) : 0u;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    v[u][j] = base[at];
                    at += j + 1 < left[u] ? plane : 0u;
                }
            }
            // Every load is issued before the first value is looked at.
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NI; u++) {
                const int i = i0 + 256 * u, q = i / HPX, px = i - q * HPX;
                if (i >= ITEMS) break;
                half8 hi, lo;
#pragma unroll
                for (int j = 0; j < 8; j++) v[u][j] = j < left[u] ? v[u][j] : 0.f;
                split8(v[u], hi, lo);
                const int at = 4 * px + (q ^ ((px >> 2) & 3));
                s_hi[at] = hi;
                s_lo[at] = lo;
            }
        }
        __syncthreads();
#pragma unroll
        for (int ky = 0; ky < 3; ky++) {
            half8 a[3][NT], al[3][NT];
#pragma unroll
            for (int kx = 0; kx < 3; kx++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const size_t wo = (size_t(nb * p.chunks + chunk) * 9 + ky * 3 + kx) * (p.bn * 4) + t * 64 + r * 4 + g;
                    a[kx][t] = p.wt[wo];
                    if constexpr (LO) al[kx][t] = p.wt_lo[wo];
                }
#pragma unroll
            for (int kx = 0; kx < 3; kx++)
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const int px = (2 * wave + (m >> 1) + ky) * HW + 16 * (m & 1) + r + kx;
                    const int at = 4 * px + (g ^ ((px >> 2) & 3));
                    const half8 hi = s_hi[at], lo = s_lo[at];
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, a[kx][t], acc[m][t], 0, 0, 0);
                        accl[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, a[kx][t], accl[m][t], 0, 0, 0);
                        if constexpr (LO)
                            accl[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, al[kx][t], accl[m][t], 0, 0, 0);
                    }
                }
        }
    }
    // Lane (r, g) holds pixels 4 g .. 4 g + 3 of its tiles for output channel 16 t + r.
    const size_t plane = size_t(p.h) * p.w;
    const bool vec = (p.w & 3) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0 &&
                     (!p.res || (reinterpret_cast<uintptr_t>(p.res) & 15) == 0);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int co = nb * p.bn + 16 * t + r;
        if (co >= p.cout) continue;
        const float b = p.bias ? p.bias[co] : 0.f;
        const float as = p.affine ? p.affine[co] : 1.f, at = p.affine ? p.affine[p.cout + co] : 0.f;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const int y = y0 + 2 * wave + (m >> 1), x = x0 + 16 * (m & 1) + 4 * g;
            if (y >= p.h || x >= p.w) continue;
            const size_t o = (size_t(img) * p.cout + co) * plane + size_t(y) * p.w + x;
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                float u = acc[m][t][k] + accl[m][t][k] + b;
                if (p.affine) u = u * as + at;
                v[k] = act_dev(u, p.act);
            }
            if (vec && x + 4 <= p.w) {
                if (p.res) {
                    const float4 q = *reinterpret_cast<const float4 *>(p.res + o);
                    v[0] += q.x, v[1] += q.y, v[2] += q.z, v[3] += q.w;
                }
                *reinterpret_cast<float4 *>(p.y + o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (x + k < p.w) p.y[o + k] = v[k] + (p.res ? p.res[o + k] : 0.f);
            }
        }
    }
}

}  // namespace

bool nd_conv_tile(const NdMfmaConvArgs &a, const NdConvSource *src, int nsrc, bool saves, hipStream_t s) {
    const ConvPack &pk = a.pk;
    if (pk.kh != 3 || pk.kw != 3 || a.pt != 1 || a.pl != 1 || a.oh != a.h || a.ow != a.w || a.in_scale || a.res_up || a.x2) return false;
    if (pk.cin != a.cin || pk.cout != a.cout || !a.wt_hi || (!pk.exact && !a.wt_lo)) return false;
    if (pk.bn != 16 && pk.bn != 32 && pk.bn != 64) return false;
    NdConvSource one{a.x, 0, a.cin, a.h, a.w, 0};
    if (!src) src = &one, nsrc = 1;
    if (nsrc < 1 || nsrc > ND_SOURCES) return false;
    TileParams p{};
    int c0 = 0;
    for (int k = 0; k < nsrc; k++) {
        NdConvSource q = src[k];
        // An item of 8 channels lies in one source.
        if (c0 % 8 || q.c < 1 || q.up < 0 || q.up > 8 || (q.h << q.up) != a.h || (q.w << q.up) != a.w) return false;
        if (double(q.c) * q.h * q.w >= 1073741824.0) return false;
        q.c0 = c0;
        p.src[k] = q;
        c0 += q.c;
    }
    if (c0 != a.cin) return false;
    p.nsrc = nsrc;
    p.tiles_x = (a.w + TW - 1) / TW;
    p.tiles_y = (a.h + TH - 1) / TH;
    const double blocks = double(a.n) * p.tiles_x * p.tiles_y;
    if (blocks > 0x7fffffff || pk.nblocks > 65535) return false;
    // Tiles of which over half lies outside the image (one-row tensors) are work for nothing: a one-row
    // tensor's 512 -> 32 conv 122 us against 14.
    const double px = double(a.n) * a.h * a.w;
    if (blocks * TH * TW > 2.0 * px) return false;
    if (saves ? blocks * pk.nblocks < PART_BLOCKS : px * pk.nblocks < plain_pixels(pk.bn, a.cin, a.w)) return false;
    if (blocks == 0) return true;
    p.y = a.y;
    p.wt = reinterpret_cast<const half8 *>(a.wt_hi);
    p.wt_lo = reinterpret_cast<const half8 *>(a.wt_lo);
    p.bias = a.bias;
    p.affine = a.affine;
    p.res = a.res;
    p.cin = a.cin;
    p.h = a.h;
    p.w = a.w;
    p.cout = a.cout;
    p.bn = pk.bn;
    p.chunks = pk.chunks;
    p.act = a.act;
    double in = 0;
    for (int k = 0; k < nsrc; k++) in += double(a.n) * src[k].c * src[k].h * src[k].w;
    ProbeScope probe("nd_conv_nchw", s, 2.0 * px * a.cout * a.cin * 9,
                     4.0 * (in + px * a.cout) + 2.0 * double(pk.halves()) * (pk.exact ? 1 : 2), "nd_conv_tile");
    const dim3 grid{unsigned(blocks), unsigned(pk.nblocks)};
    auto launch = [&](auto *exact, auto *lo) {
        if (pk.exact) hipLaunchKernelGGL(exact, grid, dim3(256), 0, s, p);
        else hipLaunchKernelGGL(lo, grid, dim3(256), 0, s, p);
    };
    if (pk.bn == 16) launch(conv_tile_kernel<1, false>, conv_tile_kernel<1, true>);
    else if (pk.bn == 32) launch(conv_tile_kernel<2, false>, conv_tile_kernel<2, true>);
    else launch(conv_tile_kernel<4, false>, conv_tile_kernel<4, true>);
    OCR_HIP(hipGetLastError());
    return true;
}

}  // namespace ocr
