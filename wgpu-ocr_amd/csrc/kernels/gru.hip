// The bidirectional GRU recurrence (ONNX GRU, linear_before_reset = 1, hidden 256, gate order
// z, r, h), one persistent dispatch per layer for all lines; each line walks its own length and
// the backward direction starts at the line's own end. Semantics of the reference's recurrence
// programs (src/gpu.rs:680-819):
//   z = s(G_z + R_z h + Rb_z), r = s(G_r + R_r h + Rb_r), c = tanh(G_h + r (R_h h + Rb_h)),
//   h' = (1 - z) c + z h, h0 = 0,  with G = W x + Wb precomputed for all steps by one GEMM.
//
// What bounds it is one line's chain of dependent steps: the work of a step is small, and a line
// cannot start one before the step before it ends. So a workgroup owns one direction and few
// lines (2 or 4), and its step is made as short as one CU can make it. R (768 x 256 a direction,
// float16 values) is loaded once, into the registers of 8 wavefronts, and stays for every step.
//
// R h is a product with 16 rows at least on the matrix cores, and 4 lines are only 8 rows: each
// line's float16 "hi" part and its float16 remainder "lo" (h = hi + lo to about 2^-22). The
// sparse instruction v_smfmac_f32_16x16x64_f16 takes an A operand with two of every four k
// present, and twice the k of the dense one in the same cycles. So the state is the A operand
// and every part is spread over two rows, one with the first two of each four hidden units and
// one with the other two: nothing is left out, the four rows of a line add up to R h, and a step
// takes half the matrix instructions (48 a SIMD, 768 cycles). R is the dense B operand, a column
// a hidden unit. Lane group g (16 lanes) then holds the four rows of one line in its four
// accumulators: the sum needs no exchange between lanes. With 2 lines the A rows repeat, so two
// lane groups hold a line's sums and each takes one of a wavefront's two 16-unit tiles: a lane
// does the gate arithmetic of one unit a step (two with 4 lines).
//
// Every gate's arithmetic runs between the next gate's matrix instructions (reset, candidate,
// update); only the update gate and the new state follow the last one. G is loaded four steps
// ahead, the new state goes to a double-buffered LDS copy of the A operand: one barrier a step,
// for LDS only (the loads and the Y stores stay in flight).
//
// Measured (us a layer, kernel trace): 36 lines of at most 200 steps 303 -> 127, 540 lines 424 -> 186, one
// line of 50 steps 77 -> 36, against 8 lines a workgroup on the dense instruction with the state as its
// 16-column operand. So with 2 lines a step takes 0.61 us, of it 0.32 of matrix instructions, and the
// launch 6 besides; 16 wavefronts (4 a SIMD, part of R in LDS) took 1.6 a step, 4 wavefronts (one unit of
// one line a lane, R in 384 registers) 0.89.
//
// A workgroup's R takes its CU's register file whole, so nothing else runs on that CU meanwhile.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "../kernels.h"
#include "../runtime.h"
#include "lds_dma.h"

namespace ocr {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int H = 256;

// exp through the hardware base-2 exponential; 1/x through the hardware reciprocal (1 ulp).
__device__ inline float fast_exp(float v) { return __builtin_amdgcn_exp2f(v * 1.4426950408889634f); }
__device__ inline float sigm(float v) { return __builtin_amdgcn_rcpf(1.f + fast_exp(-v)); }
__device__ inline float tanh_f(float v) { return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + fast_exp(2.f * v)); }

__device__ inline half16 join(half8 a, half8 b) {
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
}

// LG lines a workgroup (2 or 4), 8 wavefronts of 32 hidden units (two 16-unit tiles each).
template <int LG>
__global__ __launch_bounds__(512) void gru_kernel(const float *__restrict__ G, const half8 *__restrict__ R,
                                                  const float *__restrict__ Rb, float *__restrict__ Y,
                                                  const uint32_t *__restrict__ lens, const uint32_t *__restrict__ order,
                                                  int ntot) {
    constexpr int T = 2;         // 16-unit tiles of a wavefront
    constexpr int REP = 4 / LG;  // lane groups that hold the same line's sums
    constexpr int U = T / REP;   // units of its line that a lane updates
    constexpr int D = 4;         // steps that G is loaded ahead (three whole steps pass before its use)
    static_assert(LG == 2 || LG == 4, "every lane has whole units");
    // The state as the A operands read it: [k-step][lane group][row][8 halves], row = 4 line + 2
    // (lo part) + (odd pair): the 64 lanes of a read take 64 neighbouring 16-byte units.
    __shared__ __align__(16) _Float16 hbuf[2][4][4][4 * LG][8];
    // With 4 lines the update gate's last k-step of R lives in LDS: the rest fills the registers.
    constexpr int TL = LG == 4 ? T : 0;
    __shared__ half8 s_rf[TL ? 8 : 1][TL ? TL : 1][2][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r = lane & 15;
    const int dir = blockIdx.y, n0 = blockIdx.x * LG;

    // R as B operands: column r = unit wave * 32 + t * 16 + r; lane group g holds k-step kt's
    // k = 8 g .. + 7 and 32 + 8 g .. + 7.
    half16 rf[3][T][4];
#pragma unroll
    for (int q = 0; q < 3; q++)
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int kt = 0; kt < 4; kt++) {
                const half8 *src = R + ((((size_t(dir) * 8 + wave) * 3 + q) * T + t) * 4 + kt) * 128 + lane;
                const half8 v0 = src[0], v1 = src[64];
                if (q == 0 && kt == 3 && t < TL) {
                    s_rf[wave][t][0][lane] = v0;
                    s_rf[wave][t][1][lane] = v1;
                } else {
                    rf[q][t][kt] = join(v0, v1);
                }
            }
    for (int i = tid; i < int(sizeof(hbuf) / 16); i += 512) reinterpret_cast<uint4 *>(hbuf)[i] = uint4{0, 0, 0, 0};

    // This lane's line and units. Slots past the last line repeat it (the same values written
    // twice).
    const int ls = g % LG, sub = g / LG;
    const int line = int(order[min(n0 + ls, ntot - 1)]);
    const int len = int(lens[line]);
    int maxlen = 0;
    for (int j = 0; j < LG; j++) maxlen = max(maxlen, int(lens[order[min(n0 + j, ntot - 1)]]));
    const size_t row = size_t(dir == 0 ? 0 : max(len - 1, 0)) * ntot + line;
    const int u0 = (wave * T + sub * U) * 16 + r;
    const float *gp = G + row * 1536 + dir * 768 + u0;
    float *yp = Y + row * 512 + dir * 256 + u0;
    const long gstep = (dir == 0 ? 1536l : -1536l) * ntot, ystep = (dir == 0 ? 512l : -512l) * ntot;
    float h[U], rb[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        h[u] = 0.f;
        rb[u] = Rb[dir * 256 + u0 + u * 16];
    }
    // G of D steps ahead; past its end a line reads its last row again.
    float gv[D][3][U];
    auto load_g = [&](int s, float (&v)[3][U]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int u = 0; u < U; u++) v[q][u] = gp[q * 256 + u * 16];
        gp += s + 1 < len ? gstep : 0;
    };
#pragma unroll
    for (int d = 0; d < D; d++) load_g(d, gv[d]);
    // Even rows of A hold each group of four k's first two values, odd rows the other two.
    const int idx = (r & 1) ? 0xEEEE : 0x4444;
    const int arow = r % (4 * LG);
    // Where the lane's new state goes: tile = 16 k of k-step tile / 4, lane group tile % 4.
    _Float16 *const hw = &hbuf[0][0][0][4 * ls + ((r >> 1) & 1)][2 * (r >> 2) + (r & 1)] + (wave * T + sub * U) * 32 * LG;
    constexpr int HB = 4 * 4 * 4 * LG * 8;  // halves of a state buffer
    __syncthreads();

    auto step = [&](int s, int cur, float (&gc)[3][U]) __attribute__((always_inline)) {
        half8 a[4];
#pragma unroll
        for (int kt = 0; kt < 4; kt++) a[kt] = *reinterpret_cast<const half8 *>(hbuf[cur][kt][g][arow]);
        floatx4 acc[3][T];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int t = 0; t < T; t++) acc[q][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        auto mfmas = [&](int q) __attribute__((always_inline)) {
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int t = 0; t < T; t++) {
                    const half16 b = q == 0 && kt == 3 && t < TL ? join(s_rf[wave][t][0][lane], s_rf[wave][t][1][lane])
                                                                 : rf[q][t][kt];
                    acc[q][t] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(a[kt], b, acc[q][t], idx, 0, 0);
                }
        };
        // The sum of gate q for the lane's unit u: the four rows of its line.
        auto total = [&](int q, int u) __attribute__((always_inline)) {
            const floatx4 c = acc[q][u];
            float v = (c[0] + c[1]) + (c[2] + c[3]);
            if (REP == 2) {
                const floatx4 d = acc[q][T - 1];
                const float w = (d[0] + d[1]) + (d[2] + d[3]);
                v = sub ? w : v;
            }
            return v;
        };
        // Each gate's arithmetic runs between the next gate's MFMAs.
        auto overlap = []() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4 * T; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // three VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        float rr[U], c[U];
        mfmas(1);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(2);
#pragma unroll
        for (int u = 0; u < U; u++) rr[u] = sigm(total(1, u) + gc[1][u]);
        overlap();
        mfmas(0);
#pragma unroll
        for (int u = 0; u < U; u++) c[u] = tanh_f(fmaf(rr[u], total(2, u) + rb[u], gc[2][u]));
        overlap();
#pragma unroll
        for (int u = 0; u < U; u++) {
            const float hn = fmaf(sigm(total(0, u) + gc[0][u]), h[u] - c[u], c[u]);
            h[u] = s < len ? hn : h[u];
            const _Float16 hi = (_Float16)h[u], lo = (_Float16)(h[u] - (float)hi);
            _Float16 *dst = hw + (cur ^ 1) * HB + u * 32 * LG;
            dst[0] = hi;
            dst[16] = lo;
        }
        __builtin_amdgcn_sched_barrier(0);
        // Past its end a line writes its last state to its last row again.
#pragma unroll
        for (int u = 0; u < U; u++) yp[u * 16] = h[u];
        yp += s + 1 < len ? ystep : 0;
        load_g(s + D, gc);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int s = 0; s < maxlen; s += D) {
#pragma unroll
        for (int d = 0; d < D; d++) step(s + d, d & 1, gv[d]);
    }
}

// Float32 recurrent weights (the reference's recurrence with F16 off, gpu.rs:858, 1476-1486):
// for R that is not float16-valued when rounding it is not allowed. R is too large to stay on
// chip next to its remainders, so this kernel streams it from L2 every step: one workgroup per
// (direction, 8 lines), thread u owns hidden unit u of all 8 lines, and R^T [dir][k][768] makes
// the 256 threads' reads of one (k, gate) row one coalesced 1 KiB access. h lives in LDS
// (double-buffered, one barrier a step); the gates use expf and a true division.
constexpr int FL = 8;  // lines per workgroup

__global__ __launch_bounds__(256) void gru_f32_kernel(const float *__restrict__ G, const float *__restrict__ Rt,
                                                      const float *__restrict__ Rb, float *__restrict__ Y,
                                                      const uint32_t *__restrict__ lens, int ntot) {
    __shared__ float hs[2][FL][H];
    const int u = threadIdx.x, dir = blockIdx.y, n0 = blockIdx.x * FL;
    const float *rt = Rt + size_t(dir) * H * 768;
    int len[FL], maxlen = 0;
#pragma unroll
    for (int l = 0; l < FL; l++) {
        len[l] = n0 + l < ntot ? int(lens[n0 + l]) : 0;
        maxlen = max(maxlen, len[l]);
        hs[0][l][u] = 0.f;
    }
    const float rbz = Rb[dir * 768 + u], rbr = Rb[dir * 768 + 256 + u], rbh = Rb[dir * 768 + 512 + u];
    float h[FL];
#pragma unroll
    for (int l = 0; l < FL; l++) h[l] = 0.f;
    __syncthreads();
    for (int s = 0; s < maxlen; s++) {
        const int cur = s & 1;
        float az[FL], ar[FL], ah[FL];
#pragma unroll
        for (int l = 0; l < FL; l++) az[l] = ar[l] = ah[l] = 0.f;
        for (int k = 0; k < H; k++) {
            const float wz = rt[size_t(k) * 768 + u], wr = rt[size_t(k) * 768 + 256 + u], wh = rt[size_t(k) * 768 + 512 + u];
#pragma unroll
            for (int l = 0; l < FL; l++) {
                const float hk = hs[cur][l][k];
                az[l] = fmaf(wz, hk, az[l]);
                ar[l] = fmaf(wr, hk, ar[l]);
                ah[l] = fmaf(wh, hk, ah[l]);
            }
        }
#pragma unroll
        for (int l = 0; l < FL; l++) {
            if (s < len[l]) {
                const int t = dir == 0 ? s : len[l] - 1 - s;
                const float *gr = G + (size_t(t) * ntot + n0 + l) * 1536 + dir * 768;
                const float z = 1.f / (1.f + expf(-(gr[u] + az[l] + rbz)));
                const float r = 1.f / (1.f + expf(-(gr[256 + u] + ar[l] + rbr)));
                const float c = tanhf(gr[512 + u] + r * (ah[l] + rbh));
                h[l] = (1.f - z) * c + z * h[l];
                Y[(size_t(t) * ntot + n0 + l) * 512 + dir * 256 + u] = h[l];
            }
            hs[cur ^ 1][l][u] = h[l];
        }
        __syncthreads();
    }
}

}  // namespace

// 2 lines a workgroup while every workgroup has a CU of its own (256 of them, two directions; a layer's
// time over its 200 steps): 0.64 us against 0.81 with 4 lines at 36 lines, 0.82 against 0.86 at 256. Past
// that 4 lines: the longest lines start first, so a 540-line pass (270 workgroups) still ends with its
// longest line, 186 us against 265 with 2 lines. Beside other work (the page pipeline's second stream)
// 4 lines for every pass, which leave more CUs, measured the same: 12 pages 13.18-13.19 ms against
// 13.12-13.21.
int gru_lines(int ntot) { return ntot <= 256 ? 2 : 4; }

void gru_pack_r(const uint16_t *r, uint16_t *out) {
    for (int dir = 0; dir < 2; dir++)
        for (int wave = 0; wave < 8; wave++)
            for (int q = 0; q < 3; q++)
                for (int t = 0; t < 2; t++)
                    for (int kt = 0; kt < 4; kt++)
                        for (int part = 0; part < 2; part++)
                            for (int lane = 0; lane < 64; lane++, out += 8) {
                                const int row = dir * 768 + q * 256 + (wave * 2 + t) * 16 + lane % 16;
                                std::memcpy(out, r + size_t(row) * 256 + kt * 64 + part * 32 + lane / 16 * 8, 16);
                            }
}

void gru_recurrence(const float *G, const uint16_t *R, const float *Rb, float *Y, const uint32_t *lens,
                    const uint32_t *order, int lines, int ntot, long long steps, hipStream_t s) {
    if (ntot <= 0) return;
    // Per line step and direction: R h (768 x 256), G read (768 floats), Y written (256 floats).
    ProbeScope probe("gru", s, 2.0 * 2.0 * double(steps) * 768 * 256,
                     2.0 * double(steps) * (768 + 256) * 4 + 2.0 * 768 * 256 * 2);
    auto launch = [&](auto *kernel) {
        hipLaunchKernelGGL(kernel, dim3(unsigned((ntot + lines - 1) / lines), 2), dim3(512), 0, s, G,
                           reinterpret_cast<const half8 *>(R), Rb, Y, lens, order, ntot);
    };
    if (lines == 2) launch(gru_kernel<2>);
    else launch(gru_kernel<4>);
    OCR_HIP(hipGetLastError());
}

void gru_recurrence_f32(const float *G, const float *Rt, const float *Rb, float *Y, const uint32_t *lens, int ntot,
                        long long steps, hipStream_t s) {
    if (ntot <= 0) return;
    dim3 grid(unsigned((ntot + FL - 1) / FL), 2);
    ProbeScope probe("gru", s, 2.0 * 2.0 * double(steps) * 768 * 256,
                     2.0 * double(steps) * (768 + 256) * 4 + 2.0 * 768 * 256 * 4);
    hipLaunchKernelGGL(gru_f32_kernel, grid, dim3(H), 0, s, G, Rt, Rb, Y, lens, ntot);
    OCR_HIP(hipGetLastError());
}

}  // namespace ocr
