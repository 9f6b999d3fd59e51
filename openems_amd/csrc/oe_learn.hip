// oe_learn.hip -- the learned ringdown extrapolator: training and inference
// kernels for gfx950 and the C ABI behind oe_extrap_*.
//
// The network (1-D convolutions + MLP, about 2 M parameters) maps the early
// window of a port's V and I to 32 damped complex exponential modes whose sum
// continues the signal.  No counterpart in the reference; the decay test it
// shortens is src/fdtd/basic_engine.rs:128-141.
//
// Every matrix product -- forward and backward, convolutions as im2col
// products -- runs on the BF16 matrix cores (v_mfma_f32_32x32x8bf16_1k)
// with FP32 accumulation: both operands are bfloat16 (rounded to nearest
// even from float32), the results float32.  Master weights, biases, GELU, the
// mode synthesis and Adam are float32 (phases of the synthesis float64).
// Activations are kept channels-last, [batch, position, channel].

#include "oe_objects.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#pragma clang fp contract(off)

using namespace oe;

namespace {

constexpr int KW = 9, STRIDE = 2, PADW = 4;  // convolution kernel, stride, zero padding
constexpr float A_SCALE = 0.05f, F_MAX = 0.5f;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// ------------------------------------------------------------------ GEMM
// C(m, n) = sum_k A(m, k) B(k, n) in bfloat16 products and float32 sums, with
// an epilogue on the sum (EPI_*).  64 x 64 tiles, 4 waves of 32 x 32, blocks
// of BK in k staged in LDS as [row][k], so each lane reads its 4 consecutive
// k of one row as one 8-byte load; the next block travels from memory to
// registers while the matrix cores work on this one.  MFMA 32x32x8 bf16
// operands: lane l supplies A[l % 32][4 (l / 32) .. +3] and
// B[4 (l / 32) .. +3][l % 32]; accumulator register v of lane l holds
// C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32].  Every element is one chain of
// these products in ascending k, whatever the tile it falls in: the sums that
// the next layer rounds to bfloat16 do not depend on the launch shape.
//
// KA / KB: the operand's k index is its contiguous one (16-byte loads of 8
// k), else its row index is (8-byte loads of 4 rows at 4 consecutive k, the
// 4 x 4 block turned in registers on its way to LDS).  VA / VB: strides and
// base are aligned for those loads; else elements are loaded one at a time.
//
// The weight gradients sum over the batch's rows (k up to 32768) for few
// outputs (64 x 18 up to 384 x 4096): there blockIdx.z takes a range of k and
// the parts are added in order by k_add_parts.
//
// What bounds it: the batch of 256 needs 17 GFLOP and about 120 MB, but the
// products are small (24 to 512 tiles), so a launch is bound by its chain of
// k blocks, each a round trip to L2.  With element loads, blocks of 32 and no
// split the backward of a batch of 256 spent 3.7 ms in these products (one
// tile of 1024 blocks for the first layer's weights, 1.7 ms), now 0.13 ms; the
// forward 0.61 ms, now 0.09 ms (0.40 ms to 0.04 ms for the 4096-long hidden
// layer, whose 24 tiles are one chain of 64 blocks).
enum { EPI_STORE = 0, EPI_GELU = 1, EPI_GELU_BACK = 2 };

struct GemmArgs {
    const uint16_t* A;
    long lda;               // stride of the index that is not contiguous
    const uint16_t* B;
    long ldb;
    int M, N, K;
    int kz;                 // k range of one blockIdx.z (a multiple of BK)
    int epi;
    float* C;               // [M][N] float32 (EPI_STORE: sum + bias, part z at C + z M N; EPI_GELU: the
                            // pre-activation, or null; EPI_GELU_BACK: the result)
    const float* bias;      // [N] or null
    const float* pre;       // EPI_GELU_BACK: [M][N] pre-activations
    uint16_t* Cb;           // EPI_GELU: gelu(C), EPI_GELU_BACK: the result, as bfloat16
};

constexpr int TM = 64, GEMM_BK = 64, TKP = GEMM_BK + 4;

__device__ __forceinline__ float gelu_f(float x) {
    const float c = 0.7978845608028654f;
    return 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
}
__device__ __forceinline__ float gelu_d(float x) {
    const float c = 0.7978845608028654f;
    const float t = tanhf(c * (x + 0.044715f * x * x * x));
    return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * c * (1.0f + 3.0f * 0.044715f * x * x);
}

typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));

// One operand's 64 x GEMM_BK block: registers of this thread, loaded by
// load() and written to LDS [row][k] by put().
template <bool KC, bool VEC>
struct Stage {
    u2 r[8];  // 16 elements of k-contiguous chunks, or a 4 x 4 block
    // row0: first row of the tile, rows: extent of the row index, k0 .. kend
    __device__ __forceinline__ void load(const uint16_t* __restrict__ P, long ld, int row0, int rows, int k0, int kend) {
        const int tid = threadIdx.x;
        if constexpr (VEC && KC) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int idx = tid + 256 * q, row = row0 + idx / 8, k = k0 + 8 * (idx % 8);
                u4 v = {0u, 0u, 0u, 0u};
                if (row < rows && k < kend) v = *reinterpret_cast<const u4*>(P + (size_t)row * ld + k);
                r[2 * q] = u2{v.x, v.y};
                r[2 * q + 1] = u2{v.z, v.w};
            }
        } else if constexpr (VEC) {
            const int row = row0 + 4 * (tid & 15), k = k0 + 4 * (tid >> 4);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                r[q] = u2{0u, 0u};
                if (row < rows && k + q < kend) r[q] = *reinterpret_cast<const u2*>(P + (size_t)(k + q) * ld + row);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                unsigned w[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int idx = (tid + 256 * q) * 2 + e, row = row0 + idx / GEMM_BK, k = k0 + idx % GEMM_BK;
                    w[e] = 0;
                    if (row < rows && k < kend) w[e] = KC ? P[(size_t)row * ld + k] : P[(size_t)k * ld + row];
                }
                r[q] = u2{w[0] | (w[1] << 16), 0u};
            }
        }
    }
    __device__ __forceinline__ void put(uint16_t (*S)[TKP]) const {
        const int tid = threadIdx.x;
        if constexpr (VEC && KC) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int idx = tid + 256 * q;
                uint16_t* d = &S[idx / 8][8 * (idx % 8)];
                *reinterpret_cast<u2*>(d) = r[2 * q];
                *reinterpret_cast<u2*>(d + 4) = r[2 * q + 1];
            }
        } else if constexpr (VEC) {
            const int row = 4 * (tid & 15), k = 4 * (tid >> 4);
            const unsigned a0 = r[0].x, a1 = r[1].x, a2 = r[2].x, a3 = r[3].x;
            const unsigned b0 = r[0].y, b1 = r[1].y, b2 = r[2].y, b3 = r[3].y;
            *reinterpret_cast<u2*>(&S[row][k]) = u2{(a0 & 0xffffu) | (a1 << 16), (a2 & 0xffffu) | (a3 << 16)};
            *reinterpret_cast<u2*>(&S[row + 1][k]) = u2{(a0 >> 16) | (a1 & 0xffff0000u), (a2 >> 16) | (a3 & 0xffff0000u)};
            *reinterpret_cast<u2*>(&S[row + 2][k]) = u2{(b0 & 0xffffu) | (b1 << 16), (b2 & 0xffffu) | (b3 << 16)};
            *reinterpret_cast<u2*>(&S[row + 3][k]) = u2{(b0 >> 16) | (b1 & 0xffff0000u), (b2 >> 16) | (b3 & 0xffff0000u)};
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int idx = (tid + 256 * q) * 2;
                *reinterpret_cast<unsigned*>(&S[idx / GEMM_BK][idx % GEMM_BK]) = r[q].x;
            }
        }
    }
};

template <bool KA, bool VA, bool KB, bool VB>
__global__ __launch_bounds__(256) void k_gemm_bf16(GemmArgs g) {
    __shared__ __align__(16) uint16_t As[TM][TKP];
    __shared__ __align__(16) uint16_t Bs[TM][TKP];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int bm = blockIdx.y * TM, bn = blockIdx.x * TM;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int kb = blockIdx.z * g.kz, ke = min(g.K, kb + g.kz);
    floatx16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    Stage<KA, VA> a;
    Stage<KB, VB> b;
    a.load(g.A, g.lda, bm, g.M, kb, ke);
    b.load(g.B, g.ldb, bn, g.N, kb, ke);
    for (int k0 = kb; k0 < ke; k0 += GEMM_BK) {
        a.put(As);
        b.put(Bs);
        __syncthreads();
        if (k0 + GEMM_BK < ke) {
            a.load(g.A, g.lda, bm, g.M, k0 + GEMM_BK, ke);
            b.load(g.B, g.ldb, bn, g.N, k0 + GEMM_BK, ke);
        }
#pragma unroll
        for (int kk = 0; kk < GEMM_BK; kk += 8) {
            const int kr = kk + 4 * (lane >> 5);
            const bf16x4 av = *reinterpret_cast<const bf16x4*>(&As[wm + (lane & 31)][kr]);
            const bf16x4 bv = *reinterpret_cast<const bf16x4*>(&Bs[wn + (lane & 31)][kr]);
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(av, bv, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    const int col = bn + wn + (lane & 31);
    if (col >= g.N) return;
    const float bias = g.bias ? g.bias[col] : 0.f;
    float* C = g.C ? g.C + (size_t)blockIdx.z * g.M * g.N : nullptr;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = bm + wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row >= g.M) continue;
        const size_t at = (size_t)row * g.N + col;
        float val = acc[v];
        if (g.bias) val += bias;
        if (g.epi == EPI_GELU) {
            g.Cb[at] = f2bf(gelu_f(val));
        } else if (g.epi == EPI_GELU_BACK) {
            val = val * gelu_d(g.pre[at]);
            g.Cb[at] = f2bf(val);
        }
        if (C) C[at] = val;
    }
}

// Sums of parts, several outputs per launch: out[i] = sum over p < parts of
// src[p count + i], p ascending.
constexpr int MAX_PARTS = 12;
struct PartSum {
    float* out;
    const float* src;
    unsigned count, parts;
    unsigned first;  // first work-group of this output
};
struct PartSums {
    int n;
    PartSum s[MAX_PARTS];
};

__global__ __launch_bounds__(256) void k_add_parts(PartSums ps) {
    int q = 0;
#pragma unroll
    for (int t = 1; t < MAX_PARTS; ++t)
        if (t < ps.n && blockIdx.x >= ps.s[t].first) q = t;
    const PartSum p = ps.s[q];
    const unsigned i = (blockIdx.x - p.first) * 256 + threadIdx.x;
    if (i >= p.count) return;
    float s = 0.f;
#pragma unroll 16
    for (unsigned r = 0; r < p.parts; ++r) s += p.src[(size_t)r * p.count + i];
    p.out[i] = s;
}

// -------------------------------------------------------------- elementwise
// cols[(b Lo + t) ld + c K + k] = x[b, 2 t + k - 4, c] (zero outside and in
// the row's padding, columns C K .. ld).  IN: float32 input (rounded here) or
// the bfloat16 activations of the layer before.  A work-group writes IM_T rows
// of one sample: the 2 IM_T + 7 input positions they draw on go to LDS once
// (each is used by 4 or 5 rows), and a thread gathers 8 consecutive columns
// into one 16-byte store.  Bound by its stores, 19 MB for each of the two wide
// layers at a batch of 256; one element per thread with two divisions took
// 23 us a layer, this form 11.5.
constexpr int IM_T = 8, IM_POS = STRIDE * (IM_T - 1) + KW, IM_C = 256;

// grid (sample, IM_T rows, IM_C channels)
template <class IN>
__global__ __launch_bounds__(256) void k_im2col(const IN* __restrict__ x, int L, int C, int ld,
                                                uint16_t* __restrict__ cols) {
    __shared__ uint16_t xs[IM_POS][IM_C + 2];
    const int Lo = L / STRIDE;
    const int b = blockIdx.x, t0 = blockIdx.y * IM_T, c0 = blockIdx.z * IM_C;
    const int nc = min(IM_C, C - c0), s0 = STRIDE * t0 - PADW;
    for (int p = threadIdx.x >> 6; p < IM_POS; p += 4) {
        const int s = s0 + p;
        const bool in = s >= 0 && s < L;
        const IN* row = x + ((size_t)b * L + (in ? s : 0)) * C + c0;
        for (int c = threadIdx.x & 63; c < nc; c += 64) {
            uint16_t v = 0;
            if (in) {
                if constexpr (sizeof(IN) == 4) v = f2bf(row[c]);
                else v = row[c];
            }
            xs[p][c] = v;
        }
    }
    __syncthreads();
    // columns of this range of channels (a multiple of 8 from c0 KW on); the
    // last range writes the row's padding too
    const int nt = min(IM_T, Lo - t0), je = c0 + nc == C ? ld - c0 * KW : nc * KW;
    for (int t = threadIdx.x >> 6; t < nt; t += 4) {
        uint16_t* row = cols + ((size_t)b * Lo + t0 + t) * ld + (size_t)c0 * KW;
        for (int j0 = 8 * (threadIdx.x & 63); j0 < je; j0 += 8 * 64) {
            int c = j0 / KW, k = j0 - c * KW;
            unsigned w[4];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const unsigned v = c < nc ? xs[STRIDE * t + k][c] : 0u;
                if (e & 1) w[e >> 1] |= v << 16;
                else w[e >> 1] = v;
                if (++k == KW) {
                    k = 0;
                    ++c;
                }
            }
            *reinterpret_cast<u4*>(row + j0) = u4{w[0], w[1], w[2], w[3]};
        }
    }
}

// The adjoint, and the activation's derivative on it: dx[b, s, c] = sum over
// (t, k) with 2 t + k - 4 = s of dcols[(b Lo + t) C K + c K + k] (t
// ascending), dpre = dx gelu'(pre).  A work-group takes CI_S positions and
// CI_C channels of one sample: the CI_T rows of dcols they draw on go to LDS
// with contiguous loads (a channel's 9 columns lie together, so the gathers
// stride 9 words and meet no bank conflict).  Bound by reading dcols, 38 MB a
// layer at a batch of 256: 24 us with gathers from memory and the derivative
// in a launch of its own (7 us), 16 us in this form.
constexpr int CI_S = 16, CI_C = 64, CI_T = CI_S / STRIDE + 4;

// grid (sample, CI_S positions, CI_C channels); WIDE: CI_C channels in every
// work-group and 16-byte rows of dcols
template <bool WIDE>
__global__ __launch_bounds__(256) void k_col2im_gelu_back(const float* __restrict__ dcols, int L, int C,
                                                          const float* __restrict__ pre, float* __restrict__ dpre,
                                                          uint16_t* __restrict__ dpreb) {
    __shared__ __align__(16) float rows[CI_T][CI_C * KW];
    const int Lo = L / STRIDE, CK = C * KW;
    const int b = blockIdx.x, s0 = blockIdx.y * CI_S, c0 = blockIdx.z * CI_C;
    const int nc = WIDE ? CI_C : min(CI_C, C - c0);
    // row t = tb + r reaches positions 2 t - 4 .. 2 t + 4
    const int tb = s0 / STRIDE - PADW / STRIDE;
    constexpr int W4 = CI_C * KW / 4;
    for (int q = threadIdx.x; q < (WIDE ? CI_T * W4 : CI_T * 64); q += 256) {
        if constexpr (WIDE) {
            const int r = q / W4, j = 4 * (q - r * W4), t = tb + r;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (t >= 0 && t < Lo) v = *reinterpret_cast<const float4*>(dcols + ((size_t)b * Lo + t) * CK + c0 * KW + j);
            *reinterpret_cast<float4*>(&rows[r][j]) = v;
        } else {
            const int r = q >> 6, t = tb + r;
            for (int j = q & 63; j < nc * KW; j += 64)
                rows[r][j] = (t >= 0 && t < Lo) ? dcols[((size_t)b * Lo + t) * CK + c0 * KW + j] : 0.f;
        }
    }
    __syncthreads();
    const int c = threadIdx.x & 63;
    if (c >= nc) return;
    for (int ds = threadIdx.x >> 6; ds < CI_S; ds += 4) {
        const int s = s0 + ds;
        if (s >= L) break;
        float acc = 0.f;
        const int t_lo = max(0, (s + PADW - (KW - 1) + STRIDE - 1) / STRIDE);
        const int t_hi = min(Lo - 1, (s + PADW) / STRIDE);
        for (int t = t_lo; t <= t_hi; ++t) acc += rows[t - tb][c * KW + s + PADW - STRIDE * t];
        const size_t at = ((size_t)b * L + s) * C + c0 + c;
        const float v = acc * gelu_d(pre[at]);
        dpre[at] = v;
        dpreb[at] = f2bf(v);
    }
}

__global__ void k_to_bf16(const float* __restrict__ a, uint16_t* __restrict__ b, size_t n) {
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        b[q] = f2bf(a[q]);
}

// Column sums of X[M, N], first part: work-group (cb, r) sums rows
// r per .. (r + 1) per of 64 columns with 4 row lanes, combined in a fixed
// order; k_add_parts adds the parts.  The host cuts M so that about 256
// work-groups read it (64 of them took 32 us for 32768 x 64, this 5 us).
__global__ __launch_bounds__(256) void k_colsum_part(const float* __restrict__ X, int M, int N, int per,
                                                     float* __restrict__ part) {
    __shared__ float red[4][64];
    const int c = blockIdx.x * 64 + (threadIdx.x & 63), rl = threadIdx.x >> 6;
    const int r1 = min(M, (int)(blockIdx.y + 1) * per);
    float s = 0.f;
    if (c < N)
#pragma unroll 4
        for (int r = blockIdx.y * per + rl; r < r1; r += 4) s += X[(size_t)r * N + c];
    red[rl][threadIdx.x & 63] = s;
    __syncthreads();
    if (rl == 0 && c < N) part[(size_t)blockIdx.y * N + c] = ((red[0][threadIdx.x] + red[1][threadIdx.x]) +
                                                               red[2][threadIdx.x]) + red[3][threadIdx.x];
}

// Mode synthesis, loss and its gradient for one sample per work-group.
// o [B, 6 M]: per mode (softplus^-1 damping, logit frequency, V re, V im,
// I re, I im).  target [B, 2, T].  The residual goes to LDS (T <= TMAX),
// the loss partial to loss[b] (float64), dL/do to dout [B, 6 M] and, as
// bfloat16, to doutb; scale is 1 / (B 2 T) of the mean.
//
// The powers z^n of a mode, z = exp(-alpha + j 2 pi f), come from two float64
// tables in LDS, z^n = z^(n0 + ZB a) z^b with n = n0 + ZB a + b: ZB + TC / ZB
// exponentials for a chunk of TC samples instead of TC, and one complex
// product per (n, mode).  The modes are taken MC at a time.  The gradient's
// sums over n run on 256 / MC threads a mode, added in a fixed order.  Bound
// by float64 arithmetic: one exponential and one sincos per (n, mode), and the
// gradient on one thread a mode, took 228 us at 256 samples, 32 modes, T = 512
// (52 us without the gradient); this form 31 us (18 us).
constexpr int TMAX = 4096, ZB = 32, TC = 512, NA = TC / ZB;

template <int MC>
size_t modes_lds(int T) {
    return ((size_t)MC * (ZB + NA) * 2 + 256 + 2 * TC) * sizeof(double) + 2 * (size_t)T * sizeof(float);
}

template <int MC>
__global__ __launch_bounds__(256) void k_modes_loss(const float* __restrict__ o, const float* __restrict__ target,
                                                    int M, int T, double scale, double* __restrict__ loss,
                                                    float* __restrict__ dout, uint16_t* __restrict__ doutb,
                                                    float* __restrict__ tails) {
    constexpr int ZL = 256 / MC;
    extern __shared__ double lds[];
    double2* zb = reinterpret_cast<double2*>(lds);          // [MC][ZB] z^b
    double2* za = zb + MC * ZB;                             // [MC][NA] z^(n0 + ZB a)
    double* red = reinterpret_cast<double*>(za + MC * NA);  // [256]
    double* sv = red + 256;                                 // [2][TC] V and I summed over the modes so far
    float* res = reinterpret_cast<float*>(sv + 2 * TC);     // [2][T] residuals
    const int b = blockIdx.x, tid = threadIdx.x;
    const float* ob = o + (size_t)b * 6 * M;
    const float* tg = target + (size_t)b * 2 * T;
    const bool once = M <= MC && T <= TC;  // one set of tables serves both passes
    auto tables = [&](int m0, int n0) {
        const int mc = min(MC, M - m0);
        __syncthreads();
        for (int q = tid; q < mc * (ZB + NA); q += 256) {
            const int m = q / (ZB + NA), e = q - m * (ZB + NA);
            const float* p = ob + 6 * (m0 + m);
            const double alpha = (double)(log1pf(expf(-fabsf(p[0]))) + fmaxf(p[0], 0.f)) * A_SCALE;
            const double f = (double)F_MAX / (1.0 + exp(-(double)p[1]));
            const int n = e < ZB ? e : n0 + ZB * (e - ZB);
            const double mag = exp(-alpha * n);
            double sn, cs;
            sincos(2.0 * M_PI * f * n, &sn, &cs);
            (e < ZB ? zb[m * ZB + e] : za[m * NA + e - ZB]) = make_double2(mag * cs, mag * sn);
        }
        __syncthreads();
    };
    auto power = [&](int m, int d) {  // of mode m0 + m at sample n0 + d
        const double2 x = za[m * NA + d / ZB], y = zb[m * ZB + d % ZB];
        return make_double2(x.x * y.x - x.y * y.y, x.x * y.y + x.y * y.x);
    };
    double l = 0.0;
    for (int n0 = 0; n0 < T; n0 += TC) {
        const int nt = min(TC, T - n0);
        for (int m0 = 0; m0 < M; m0 += MC) {
            const int mc = min(MC, M - m0);
            tables(m0, n0);
            for (int d = tid; d < nt; d += 256) {
                double v = m0 ? sv[d] : 0.0, i = m0 ? sv[TC + d] : 0.0;
                for (int m = 0; m < mc; ++m) {
                    const float* p = ob + 6 * (m0 + m);
                    const double2 z = power(m, d);
                    v += (double)p[2] * z.x - (double)p[3] * z.y;
                    i += (double)p[4] * z.x - (double)p[5] * z.y;
                }
                sv[d] = v;
                sv[TC + d] = i;
            }
        }
        for (int d = tid; d < nt; d += 256) {  // this thread's own samples
            const int n = n0 + d;
            const double v = sv[d], i = sv[TC + d];
            const float rv = (float)(v - tg[n]), ri = (float)(i - tg[T + n]);
            res[n] = rv;
            res[T + n] = ri;
            if (tails) {
                tails[(size_t)b * 2 * T + n] = (float)v;
                tails[(size_t)b * 2 * T + T + n] = (float)i;
            }
            l += (double)rv * rv + (double)ri * ri;
        }
    }
    red[tid] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (tid < s) red[tid] += red[tid + s];
        __syncthreads();
    }
    if (tid == 0) loss[b] = red[0];
    if (!dout) return;
    const int ml = tid / ZL, lane = tid % ZL;
    for (int m0 = 0; m0 < M; m0 += MC) {
        const bool on = m0 + ml < M;
        const float* p = ob + 6 * (on ? m0 + ml : m0);
        double s[6] = {0, 0, 0, 0, 0, 0};  // d V re, V im, I re, I im; sum of n (g_v a_v + g_i a_i) z^n
        for (int n0 = 0; n0 < T; n0 += TC) {
            if (!once) tables(m0, n0);
            const int nt = on ? min(TC, T - n0) : 0;
            for (int d = lane; d < nt; d += ZL) {
                const int n = n0 + d;
                const double gv = 2.0 * scale * res[n], gi = 2.0 * scale * res[T + n];
                const double2 z = power(ml, d);
                s[0] += gv * z.x;
                s[1] -= gv * z.y;
                s[2] += gi * z.x;
                s[3] -= gi * z.y;
                const double avr = (double)p[2] * z.x - (double)p[3] * z.y, avi = (double)p[2] * z.y + (double)p[3] * z.x;
                const double air = (double)p[4] * z.x - (double)p[5] * z.y, aii = (double)p[4] * z.y + (double)p[5] * z.x;
                s[4] += n * (gv * avr + gi * air);
                s[5] += n * (gv * avi + gi * aii);
            }
        }
#pragma unroll
        for (int w = ZL / 2; w > 0; w >>= 1)
#pragma unroll
            for (int q = 0; q < 6; ++q) s[q] += __shfl_xor(s[q], w, ZL);
        if (lane == 0 && on) {
            const double sig = 1.0 / (1.0 + exp(-(double)p[1]));
            const double sigmoid0 = 1.0 / (1.0 + exp(-(double)p[0]));
            const size_t at = (size_t)b * 6 * M + 6 * (m0 + ml);
            const float d[6] = {(float)(-s[4] * A_SCALE * sigmoid0),
                                (float)(2.0 * M_PI * (-s[5]) * F_MAX * sig * (1.0 - sig)),
                                (float)s[0], (float)s[1], (float)s[2], (float)s[3]};
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                dout[at + q] = d[q];
                doutb[at + q] = f2bf(d[q]);
            }
        }
    }
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       uint16_t* __restrict__ wb, size_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) {
        const float gq = g[q];
        const float mq = b1 * m[q] + (1.0f - b1) * gq;
        const float vq = b2 * v[q] + (1.0f - b2) * gq * gq;
        m[q] = mq;
        v[q] = vq;
        const float wq = w[q] - lr * (mq / c1) / (sqrtf(vq / c2) + eps);
        w[q] = wq;
        wb[q] = f2bf(wq);
    }
}

int blocks_for(size_t n) { return (int)std::min<size_t>((n + 255) / 256, 8192); }

}  // namespace

// ------------------------------------------------------------------ host
struct oe_extrap {
    int device = 0;
    hipStream_t stream = nullptr;
    oe_extrap_dims d{};
    int C[4], L[4];
    size_t off[10], cnt[10], n_params = 0;
    DevBuf w, wb, g, m, v;         // fp32 master, bf16 copy, grads, Adam moments
    DevBuf act;                    // activations and scratch for the largest batch
    uint64_t adam_t = 0;
    // activation layout (byte offsets into act)
    size_t x0, pre[3], hb[3], cols[3], dcols, dpre, dpreb, pre4, h4b, o, dout, doutb, dpre4, dpre4b, loss, parts, tails,
        bytes;
    size_t ldc[3];                 // row strides of cols (C KW rounded up to 8)
    ~oe_extrap() {
        if (stream) {
            (void)hipSetDevice(device);
            (void)hipStreamSynchronize(stream);
            (void)hipStreamDestroy(stream);
        }
    }
};

namespace {

// Row parts of a column sum over M rows and N columns, and k parts of a
// weight gradient of M x N outputs over K: enough work-groups to fill the
// chip, at least 64 rows or 8 k blocks each (k_add_parts reads the parts of
// an output one after another).
int colsum_parts(size_t M, size_t N) {
    const size_t want = std::max<size_t>(1, 256 / ((N + 63) / 64));
    return (int)std::max<size_t>(1, std::min<size_t>({want, M / 64, 128}));
}
int k_parts(size_t M, size_t N, size_t K) {
    const size_t tiles = ((M + TM - 1) / TM) * ((N + TM - 1) / TM);
    const size_t blocks = (K + GEMM_BK - 1) / GEMM_BK;
    const size_t want = std::max<size_t>(1, std::min<size_t>(512 / tiles, blocks / 8));
    const size_t per = (blocks + want - 1) / want;
    return (int)((blocks + per - 1) / per);
}
// An output of k_parts == 1 parts is written in place.
size_t parts_len(size_t M, size_t N, size_t K) {
    const size_t p = k_parts(M, N, K);
    return p > 1 ? p * M * N : 0;
}

// Rounded to 64 floats.
size_t al64(size_t n) { return (n + 63) & ~(size_t)63; }

// Offsets in the activation block (bytes, 256-aligned) for batch B.
void layout(oe_extrap* x, size_t B) {
    size_t p = 0;
    auto take = [&](size_t bytes) {
        const size_t q = p;
        p += (bytes + 255) & ~(size_t)255;
        return q;
    };
    const int* C = x->C;
    const int* L = x->L;
    const size_t H = x->d.hidden, O = 6 * (size_t)x->d.modes, T = x->d.tail, F = (size_t)L[3] * C[3];
    x->x0 = take(B * L[0] * C[0] * 4);
    size_t maxcols = 0, maxact = 0;
    // the parts of every weight gradient and bias sum, for any batch up to B
    // (the part counts grow with the batch, except that they are capped)
    size_t parts = 0;
    for (size_t b = 1; b <= B; ++b) {
        size_t n = al64(parts_len(O, H, b)) + al64(colsum_parts(b, O) * O) + al64(parts_len(H, F, b)) +
                   al64(colsum_parts(b, H) * H);
        for (int l = 0; l < 3; ++l) {
            const size_t rows = b * L[l + 1], CK = (size_t)C[l] * KW;
            n += al64(parts_len(C[l + 1], CK, rows)) + al64(colsum_parts(rows, C[l + 1]) * C[l + 1]);
        }
        parts = std::max(parts, n);
    }
    for (int l = 0; l < 3; ++l) {
        x->ldc[l] = ((size_t)C[l] * KW + 7) / 8 * 8;
        x->pre[l] = take(B * L[l + 1] * C[l + 1] * 4);
        x->hb[l] = take(B * L[l + 1] * C[l + 1] * 2);
        x->cols[l] = take(B * L[l + 1] * x->ldc[l] * 2);
        if (l > 0) maxcols = std::max(maxcols, B * L[l + 1] * (size_t)C[l] * KW);
        maxact = std::max(maxact, B * L[l + 1] * (size_t)C[l + 1]);
    }
    x->dcols = take(maxcols * 4);
    x->dpre = take(maxact * 4);
    x->dpreb = take(maxact * 2);
    x->pre4 = take(B * H * 4);
    x->h4b = take(B * H * 2);
    x->o = take(B * O * 4);
    x->dout = take(B * O * 4);
    x->doutb = take(B * O * 2);
    x->dpre4 = take(B * H * 4);
    x->dpre4b = take(B * H * 2);
    x->loss = take(B * 8);
    x->parts = take(parts * 4);
    x->tails = take(B * 2 * T * 4);
    x->bytes = p;
}

template <class T> T* at(oe_extrap* x, size_t off) { return reinterpret_cast<T*>(x->act.as<char>() + off); }

template <bool KA, bool KB>
void launch_gemm_t(const GemmArgs& g, bool va, bool vb, dim3 grid, hipStream_t s) {
    if (va && vb) hipLaunchKernelGGL((k_gemm_bf16<KA, true, KB, true>), grid, dim3(256), 0, s, g);
    else if (va) hipLaunchKernelGGL((k_gemm_bf16<KA, true, KB, false>), grid, dim3(256), 0, s, g);
    else if (vb) hipLaunchKernelGGL((k_gemm_bf16<KA, false, KB, true>), grid, dim3(256), 0, s, g);
    else hipLaunchKernelGGL((k_gemm_bf16<KA, false, KB, false>), grid, dim3(256), 0, s, g);
}

// ka / kb: the operand's contiguous index is k (else its row).  Wide loads
// need aligned rows; a chunk never reaches past the operand's stride.
hipError_t gemm(hipStream_t s, GemmArgs g, bool ka, bool kb, int parts = 1) {
    const int blocks = (g.K + GEMM_BK - 1) / GEMM_BK;
    g.kz = (blocks + parts - 1) / parts * GEMM_BK;
    auto wide = [&](const uint16_t* p, long ld, bool k, int rows) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(p);
        if (k) return a % 16 == 0 && ld % 8 == 0 && ld >= (g.K + 7) / 8 * 8;
        return a % 8 == 0 && ld % 4 == 0 && ld >= (rows + 3) / 4 * 4;
    };
    const bool va = wide(g.A, g.lda, ka, g.M), vb = wide(g.B, g.ldb, kb, g.N);
    const dim3 grid((g.N + TM - 1) / TM, (g.M + TM - 1) / TM, parts);
    if (ka && kb) launch_gemm_t<true, true>(g, va, vb, grid, s);
    else if (ka) launch_gemm_t<true, false>(g, va, vb, grid, s);
    else launch_gemm_t<false, false>(g, va, vb, grid, s);
    return hipGetLastError();
}

// Forward for B samples whose inputs are at x0; optional loss/backward.
oe_status run(oe_extrap* x, size_t B, const float* target_dev, bool backward, bool want_tails) {
    hipStream_t s = x->stream;
    const int* C = x->C;
    const int* L = x->L;
    const int H = (int)x->d.hidden, M = (int)x->d.modes, O = 6 * M, T = (int)x->d.tail;
    const float* W = x->w.as<float>();
    const uint16_t* Wb = x->wb.as<uint16_t>();
    float* G = x->g.as<float>();
    const int F = L[3] * C[3];
    // A [rows][K] k-contiguous times W [N][K]: pre = A W^T + b, then gelu
    auto forward = [&](const uint16_t* A, long lda, int rows, int N, int K, int layer, float* pre, uint16_t* hb) {
        GemmArgs g{};
        g.A = A; g.lda = lda;
        g.B = Wb + x->off[2 * layer]; g.ldb = K;
        g.M = rows; g.N = N; g.K = K;
        g.C = pre;
        g.bias = W + x->off[2 * layer + 1];
        g.epi = hb ? EPI_GELU : EPI_STORE;
        g.Cb = hb;
        return gemm(s, g, true, true);
    };
    for (int l = 0; l < 3; ++l) {
        const dim3 grid((unsigned)B, (L[l + 1] + IM_T - 1) / IM_T, (C[l] + IM_C - 1) / IM_C);
        if (l == 0)
            hipLaunchKernelGGL(k_im2col<float>, grid, dim3(256), 0, s, at<float>(x, x->x0), L[0], C[0], (int)x->ldc[0],
                               at<uint16_t>(x, x->cols[0]));
        else
            hipLaunchKernelGGL(k_im2col<uint16_t>, grid, dim3(256), 0, s, at<uint16_t>(x, x->hb[l - 1]), L[l], C[l],
                               (int)x->ldc[l], at<uint16_t>(x, x->cols[l]));
        // the pre-activations are read by the backward pass only
        HIP_OK(forward(at<uint16_t>(x, x->cols[l]), (long)x->ldc[l], (int)(B * L[l + 1]), C[l + 1], C[l] * KW, l,
                       backward ? at<float>(x, x->pre[l]) : nullptr, at<uint16_t>(x, x->hb[l])));
    }
    HIP_OK(forward(at<uint16_t>(x, x->hb[2]), F, (int)B, H, F, 3, backward ? at<float>(x, x->pre4) : nullptr,
                   at<uint16_t>(x, x->h4b)));
    HIP_OK(forward(at<uint16_t>(x, x->h4b), H, (int)B, O, H, 4, at<float>(x, x->o), nullptr));
    if (!target_dev && !want_tails) return OE_OK;
    const double scale = 1.0 / ((double)B * 2.0 * T);
    // 32 modes a pass where their tables and the residuals share 64 KB of LDS
    const bool wide_modes = M > 16 && modes_lds<32>(T) <= 65536;
    hipLaunchKernelGGL(wide_modes ? k_modes_loss<32> : k_modes_loss<16>, dim3((unsigned)B), dim3(256),
                       wide_modes ? modes_lds<32>(T) : modes_lds<16>(T), s, at<float>(x, x->o),
                       target_dev ? target_dev : at<float>(x, x->tails), M, T, scale, at<double>(x, x->loss),
                       backward ? at<float>(x, x->dout) : nullptr, at<uint16_t>(x, x->doutb),
                       want_tails ? at<float>(x, x->tails) : nullptr);
    HIP_OK(hipGetLastError());
    if (!backward) return OE_OK;

    PartSums ps{};
    unsigned wg = 0;
    size_t used = 0;
    auto parts_of = [&](float* out, size_t count, int parts) {  // where the parts of an output go
        float* src = at<float>(x, x->parts) + used;
        used += al64(count * parts);
        ps.s[ps.n++] = PartSum{out, src, (unsigned)count, (unsigned)parts, wg};
        wg += (unsigned)((count + 255) / 256);
        return src;
    };
    // G[N][K] = D^T X over the rows, D [rows][N], X [rows][K]
    auto weights = [&](const uint16_t* D, int N, const uint16_t* X, long ldx, int K, int rows, float* out) {
        const int parts = k_parts(N, K, rows);
        GemmArgs g{};
        g.A = D; g.lda = N;
        g.B = X; g.ldb = ldx;
        g.M = N; g.N = K; g.K = rows;
        g.C = parts > 1 ? parts_of(out, (size_t)N * K, parts) : out;
        return gemm(s, g, false, false, parts);
    };
    auto bias = [&](const float* D, int rows, int N, float* out) {
        const int parts = colsum_parts(rows, N);
        float* dst = parts_of(out, N, parts);
        hipLaunchKernelGGL(k_colsum_part, dim3((N + 63) / 64, parts), dim3(256), 0, s, D, rows, N,
                           (rows + parts - 1) / parts, dst);
        return hipGetLastError();
    };
    // D [rows][N] times W [N][K], then (pre) the activation's derivative
    auto data = [&](const uint16_t* D, int rows, int N, int layer, int K, const float* pre, float* out, uint16_t* outb) {
        GemmArgs g{};
        g.A = D; g.lda = N;
        g.B = Wb + x->off[2 * layer]; g.ldb = K;
        g.M = rows; g.N = K; g.K = N;
        g.epi = pre ? EPI_GELU_BACK : EPI_STORE;
        g.C = out;
        g.pre = pre;
        g.Cb = outb;
        return gemm(s, g, true, false);
    };
    // fc2
    HIP_OK(weights(at<uint16_t>(x, x->doutb), O, at<uint16_t>(x, x->h4b), H, H, (int)B, G + x->off[8]));
    HIP_OK(bias(at<float>(x, x->dout), (int)B, O, G + x->off[9]));
    HIP_OK(data(at<uint16_t>(x, x->doutb), (int)B, O, 4, H, at<float>(x, x->pre4), at<float>(x, x->dpre4),
                at<uint16_t>(x, x->dpre4b)));
    // fc1
    HIP_OK(weights(at<uint16_t>(x, x->dpre4b), H, at<uint16_t>(x, x->hb[2]), F, F, (int)B, G + x->off[6]));
    HIP_OK(bias(at<float>(x, x->dpre4), (int)B, H, G + x->off[7]));
    HIP_OK(data(at<uint16_t>(x, x->dpre4b), (int)B, H, 3, F, at<float>(x, x->pre[2]), at<float>(x, x->dpre),
                at<uint16_t>(x, x->dpreb)));
    // convolutions, last to first: dpre holds dL/dpre of layer l
    for (int l = 2; l >= 0; --l) {
        const int rows = (int)(B * L[l + 1]), CK = C[l] * KW, Co = C[l + 1];
        HIP_OK(weights(at<uint16_t>(x, x->dpreb), Co, at<uint16_t>(x, x->cols[l]), (long)x->ldc[l], CK, rows,
                       G + x->off[2 * l]));
        HIP_OK(bias(at<float>(x, x->dpre), rows, Co, G + x->off[2 * l + 1]));
        if (l > 0) {
            HIP_OK(data(at<uint16_t>(x, x->dpreb), rows, Co, l, CK, nullptr, at<float>(x, x->dcols), nullptr));
            const dim3 grid((unsigned)B, (L[l] + CI_S - 1) / CI_S, (C[l] + CI_C - 1) / CI_C);
            hipLaunchKernelGGL(C[l] % CI_C == 0 ? k_col2im_gelu_back<true> : k_col2im_gelu_back<false>, grid, dim3(256), 0, s, at<float>(x, x->dcols), L[l], C[l],
                               at<float>(x, x->pre[l - 1]), at<float>(x, x->dpre), at<uint16_t>(x, x->dpreb));
        }
    }
    hipLaunchKernelGGL(k_add_parts, dim3(wg), dim3(256), 0, s, ps);
    HIP_OK(hipGetLastError());
    return OE_OK;
}

oe_status upload_inputs(oe_extrap* x, const float* in, size_t B, const float* target, float** target_dev) {
    if (B == 0 || B > x->d.batch) return fail(OE_ERR_CONFIG, "batch %zu outside 1..%u", B, x->d.batch);
    HIP_OK(hipMemcpyAsync(at<float>(x, x->x0), in, B * x->L[0] * 2 * sizeof(float), hipMemcpyHostToDevice, x->stream));
    if (target) {
        HIP_OK(hipMemcpyAsync(at<float>(x, x->tails), target, B * 2 * x->d.tail * sizeof(float), hipMemcpyHostToDevice,
                              x->stream));
        *target_dev = at<float>(x, x->tails);
    }
    return OE_OK;
}

double sum_loss(oe_extrap* x, size_t B) {
    std::vector<double> l(B);
    (void)hipMemcpyAsync(l.data(), at<double>(x, x->loss), B * 8, hipMemcpyDeviceToHost, x->stream);
    (void)hipStreamSynchronize(x->stream);
    double s = 0.0;
    for (double v : l) s += v;
    return s / ((double)B * 2.0 * x->d.tail);
}

}  // namespace

extern "C" {

size_t oe_extrap_param_count(const oe_extrap* x) { return x ? x->n_params : 0; }

oe_status oe_extrap_create(int device, const oe_extrap_dims* dims, const float* params, uint64_t seed,
                           oe_extrap** out) {
    if (!dims || !out) return fail(OE_ERR_CONFIG, "null argument");
    const oe_extrap_dims& d = *dims;
    if (d.L0 < 8 || d.L0 % 8 || !d.c1 || !d.c2 || !d.c3 || !d.hidden || !d.modes || d.modes > 256 || !d.batch ||
        !d.tail || d.tail > (uint32_t)TMAX)
        return fail(OE_ERR_CONFIG, "bad extrapolator dimensions (L0 multiple of 8, modes <= 256, tail <= %d)", TMAX);
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(OE_ERR_DEVICE, "no HIP device available");
    if (device < 0 || device >= n) return fail(OE_ERR_CONFIG, "device %d out of range", device);
    std::unique_ptr<oe_extrap> x(new oe_extrap());
    x->device = device;
    x->d = d;
    HIP_OK(hipSetDevice(device));
    HIP_OK(hipStreamCreateWithFlags(&x->stream, hipStreamNonBlocking));
    x->C[0] = 2; x->C[1] = (int)d.c1; x->C[2] = (int)d.c2; x->C[3] = (int)d.c3;
    x->L[0] = (int)d.L0;
    for (int l = 1; l < 4; ++l) x->L[l] = x->L[l - 1] / STRIDE;
    const size_t F = (size_t)x->L[3] * x->C[3];
    const size_t shapes[10] = {(size_t)x->C[1] * x->C[0] * KW, (size_t)x->C[1], (size_t)x->C[2] * x->C[1] * KW,
                               (size_t)x->C[2], (size_t)x->C[3] * x->C[2] * KW, (size_t)x->C[3], d.hidden * F,
                               d.hidden, 6 * (size_t)d.modes * d.hidden, 6 * (size_t)d.modes};
    size_t p = 0;
    for (int q = 0; q < 10; ++q) {
        x->off[q] = p;
        x->cnt[q] = shapes[q];
        p += shapes[q];
    }
    x->n_params = p;
    std::vector<float> w(p, 0.f);
    if (params) {
        std::memcpy(w.data(), params, p * sizeof(float));
    } else {  // He initialisation of the weights, zero biases
        std::mt19937_64 rng(seed);
        std::normal_distribution<double> nd(0.0, 1.0);
        const size_t fan[5] = {(size_t)x->C[0] * KW, (size_t)x->C[1] * KW, (size_t)x->C[2] * KW, F, d.hidden};
        for (int l = 0; l < 5; ++l)
            for (size_t q = 0; q < x->cnt[2 * l]; ++q)
                w[x->off[2 * l] + q] = (float)(nd(rng) * std::sqrt(2.0 / (double)fan[l]));
    }
    HIP_OK(x->w.alloc(p * 4));
    HIP_OK(x->wb.alloc(p * 2));
    HIP_OK(x->g.alloc(p * 4));
    HIP_OK(x->m.alloc(p * 4));
    HIP_OK(x->v.alloc(p * 4));
    HIP_OK(hipMemcpy(x->w.p, w.data(), p * 4, hipMemcpyHostToDevice));
    HIP_OK(hipMemset(x->m.p, 0, p * 4));
    HIP_OK(hipMemset(x->v.p, 0, p * 4));
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks_for(p)), dim3(256), 0, x->stream, x->w.as<float>(), x->wb.as<uint16_t>(), p);
    HIP_OK(hipGetLastError());
    layout(x.get(), d.batch);
    HIP_OK(x->act.alloc(x->bytes));
    HIP_OK(hipMemsetAsync(x->act.p, 0, x->bytes, x->stream));
    HIP_OK(hipStreamSynchronize(x->stream));
    *out = x.release();
    return OE_OK;
}

void oe_extrap_destroy(oe_extrap* x) { delete x; }

oe_status oe_extrap_params(oe_extrap* x, float* out, size_t n) {
    if (!x || !out) return fail(OE_ERR_CONFIG, "null argument");
    if (n < x->n_params) return fail(OE_ERR_CONFIG, "buffer holds %zu of %zu parameters", n, x->n_params);
    HIP_OK(hipSetDevice(x->device));
    HIP_OK(hipStreamSynchronize(x->stream));
    HIP_OK(hipMemcpy(out, x->w.p, x->n_params * 4, hipMemcpyDeviceToHost));
    return OE_OK;
}

oe_status oe_extrap_set_params(oe_extrap* x, const float* in, size_t n) {
    if (!x || !in) return fail(OE_ERR_CONFIG, "null argument");
    if (n != x->n_params) return fail(OE_ERR_CONFIG, "expected %zu parameters, got %zu", x->n_params, n);
    HIP_OK(hipSetDevice(x->device));
    HIP_OK(hipMemcpyAsync(x->w.p, in, n * 4, hipMemcpyHostToDevice, x->stream));
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks_for(n)), dim3(256), 0, x->stream, x->w.as<float>(), x->wb.as<uint16_t>(), n);
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(x->stream));
    return OE_OK;
}

oe_status oe_extrap_forward(oe_extrap* x, const float* inputs, size_t B, float* modes, float* tails) {
    if (!x || !inputs) return fail(OE_ERR_CONFIG, "null argument");
    HIP_OK(hipSetDevice(x->device));
    OE_TRY(upload_inputs(x, inputs, B, nullptr, nullptr));
    OE_TRY(run(x, B, nullptr, false, tails != nullptr));
    const size_t O = 6 * (size_t)x->d.modes;
    if (modes) HIP_OK(hipMemcpyAsync(modes, at<float>(x, x->o), B * O * 4, hipMemcpyDeviceToHost, x->stream));
    if (tails)
        HIP_OK(hipMemcpyAsync(tails, at<float>(x, x->tails), B * 2 * x->d.tail * 4, hipMemcpyDeviceToHost, x->stream));
    HIP_OK(hipStreamSynchronize(x->stream));
    return OE_OK;
}

oe_status oe_extrap_gradients(oe_extrap* x, const float* inputs, const float* target, size_t B, double* loss,
                              float* grads) {
    if (!x || !inputs || !target) return fail(OE_ERR_CONFIG, "null argument");
    HIP_OK(hipSetDevice(x->device));
    float* tdev = nullptr;
    OE_TRY(upload_inputs(x, inputs, B, target, &tdev));
    OE_TRY(run(x, B, tdev, true, false));
    if (loss) *loss = sum_loss(x, B);
    if (grads) HIP_OK(hipMemcpyAsync(grads, x->g.p, x->n_params * 4, hipMemcpyDeviceToHost, x->stream));
    HIP_OK(hipStreamSynchronize(x->stream));
    return OE_OK;
}

oe_status oe_extrap_train_step(oe_extrap* x, const float* inputs, const float* target, size_t B, float lr,
                               double* loss) {
    if (!x || !inputs || !target) return fail(OE_ERR_CONFIG, "null argument");
    if (!(lr > 0.f)) return fail(OE_ERR_CONFIG, "learning rate must be positive");
    HIP_OK(hipSetDevice(x->device));
    float* tdev = nullptr;
    OE_TRY(upload_inputs(x, inputs, B, target, &tdev));
    OE_TRY(run(x, B, tdev, true, false));
    x->adam_t += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)x->adam_t), c2 = 1.0f - std::pow(b2, (float)x->adam_t);
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(x->n_params)), dim3(256), 0, x->stream, x->w.as<float>(),
                       x->g.as<float>(), x->m.as<float>(), x->v.as<float>(), x->wb.as<uint16_t>(), x->n_params, lr, b1,
                       b2, 1e-8f, c1, c2);
    HIP_OK(hipGetLastError());
    if (loss) *loss = sum_loss(x, B);
    HIP_OK(hipStreamSynchronize(x->stream));
    return OE_OK;
}

}  // extern "C"
