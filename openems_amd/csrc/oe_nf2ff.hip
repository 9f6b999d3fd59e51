// oe_nf2ff.hip -- near-field to far-field transform on gfx950.
//
// The radiation integrals of matlab/AnalyzeNF2FF.m:186-197 for one face with
// in-plane axes p, q (node coordinates x_p, x_q, trapezoid weights w_p, w_q)
// and the four tangential equivalent currents B_c(ip, iq) factor per angle a
// with direction cosines kappa = (sin t cos f, sin t sin f, cos t) as
//   G[a, iq, c] = sum_ip exp(+j k kappa_p(a) x_p[ip]) w_p[ip] B_c(ip, iq)
//   S[a, c]     = exp(+j k kappa_0(a) x_0) sum_iq w_q[iq] exp(+j k kappa_q(a) x_q[iq]) G[a, iq, c].
// G depends on the angle only through kappa_p, and only through |kappa_p| up
// to a sign: with C = cos(k |kappa_p| x_p), S = sin(k |kappa_p| x_p) and
// s = sign(kappa_p), G = (C Br - s S Bi) + j (C Bi + s S Br).  So the first
// contraction runs once per DISTINCT |kappa_p| (U values) as one real GEMM
//   [C_u; S_u]_{u} (2U x n_p)  x  [Br | Bi] (n_p x 8 n_q)
// on the FP32 matrix cores (v_mfma_f32_32x32x2f32), and p is the in-plane
// axis with the fewer distinct values (|cos t| on a (t, f) grid has at most
// n_t of them).  The second contraction, the per-angle phase and the
// projection are float64.
//
// Every step is one launch over all faces (up to 6 at a time), which read
// their sizes and buffers from a table in device memory: pack, operands
// (phase rows and split B), the contractions, the reduction, the projection.
// The faces of a small box are a few microseconds of work each, so a launch
// per face and step (about 35 of them, on two streams) was what a transform
// of two pattern cuts cost: 232 us for 181 x 2 angles and 62 x 55 x 41 nodes,
// where six launches take 77.

#include "oe_internal.h"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <memory>
#include <numeric>
#include <vector>

#pragma clang fp contract(off)

namespace oe {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int GBM = 128, GBN = 128, GBK = 16;  // M, N padding and K step of the FP32 GEMM
constexpr int KPAD = 32;                        // K padding (a multiple of both GEMMs' K steps)
constexpr int LDS_PAD = 32;  // row stride = tile + 32 words: the two half-waves read different bank halves

// C[M x N] = A[M x K] * B[K x N], row-major float32; M, N multiples of TILE,
// K a multiple of 16 (the caller pads with zeros).  256 threads: 4 waves in
// a 2 x 2 grid, each owning a (TILE/2) x (TILE/2) sub-tile as MB x MB MFMA
// 32x32 blocks (MB = TILE/64).  The next K step's tiles are loaded into
// registers while the matrix cores work on the current one.
// MFMA 32x32x2 operands: lane l supplies A[l % 32][l / 32] and
// B[l / 32][l % 32]; accumulator register v of lane l holds
// C[8 (v / 4) + 4 (l / 32) + (v % 4)][l % 32].
//
// A launch covers the faces of kind KIND_FP32 (TILE = 64) or KIND_FP32_LARGE
// (128), each N / TILE x M / TILE work-groups from its first one on.  Rows of
// B at and past np (the K padding) count as zeros whatever they hold.
enum { KIND_FP32 = 0, KIND_FP32_LARGE = 1, KIND_SPLIT16 = 2 };

// One face as the kernels see it.
struct FaceDev {
    const void* src;
    double scale;
    int kind, n1, n2, swap, sign;  // source layout (0 float64 pairs, 1 float32 quads), nodes, p is axis 2
    int np, nq, K, N, nb;          // contraction sizes; work-groups of the pack
    const double *xp, *wp, *xq, *wq;
    float *B, *A, *G;              // operands and result of the first contraction
    _Float16 *Bhi, *Blo;
    float* bsc;                    // scale of the split B and its inverse
    double* part;                  // radiated-power partials
    float* pmax;                   // block maxima of |B|
    int split;                     // some chunk runs on the FP16 matrix cores
    const double* uval;
    int uni_p, uni_q;
    double dxp, dxq, x0;
    const double *kapq, *kap0;     // per angle
    const float* usgn;             // per angle: sign of kappa_p
    const int* uidx;               // per angle: row
    const int* order;              // angles sorted by row
    const int2* groups;            // (first index into order, count <= REDUCE_M)
    const int4* mgroups;           // mirror groups (row, first index into members, count, 0)
    const double* gkq;             // per mirror group: |kappa_q| of its first member
    const int* members;
    double* S;                     // [n_ang][4] complex: this face's sums
    int a1, a2;
};

// The part of a face in one chunk of rows.
struct ChunkDev {
    int kind;            // KIND_*
    int u0, u1, M;       // rows u0 .. u1 (two each), padded
    int first;           // its first work-group in the launch of its kind
    int mirror;          // reduced by mirror groups [g0, g1), else by groups
    int g0, g1;
};
constexpr int MAX_FACES = 6;

// Whether a launch over the kinds of a bit mask takes this chunk.
__device__ __forceinline__ bool takes(const ChunkDev& c, int kinds) { return c.kind >= 0 && (kinds >> c.kind & 1); }

// The face whose work-groups hold blockIdx.x in a launch over kind.
__device__ __forceinline__ int face_of_block(const ChunkDev* ch, int nf, int kind) {
    int f = -1;
    for (int q = 0; q < nf; ++q)
        if (ch[q].kind == kind && (int)blockIdx.x >= ch[q].first) f = q;
    return f;
}

template <int TILE>
__global__ __launch_bounds__(256) void k_sgemm_mfma(const FaceDev* __restrict__ fc, const ChunkDev* __restrict__ ch,
                                                    int nf) {
    const int fi = face_of_block(ch, nf, TILE == 64 ? KIND_FP32 : KIND_FP32_LARGE);
    const FaceDev& fd = fc[fi];
    const float* __restrict__ A = fd.A;
    const float* __restrict__ B = fd.B;
    float* __restrict__ C = fd.G;
    const int N = fd.N, K = fd.K, np = fd.np, tile = blockIdx.x - ch[fi].first, tn = N / TILE;
    constexpr int MB = TILE / 64;        // MFMA blocks per wave and dimension
    constexpr int LV = TILE / 64;        // float4 loads per thread and matrix per K step
    __shared__ float As[GBK][TILE + LDS_PAD];
    __shared__ __align__(16) float Bs[GBK][TILE + LDS_PAD];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int bm = tile / tn * TILE, bn = tile % tn * TILE;
    const int wm = (wave >> 1) * (TILE / 2), wn = (wave & 1) * (TILE / 2);
    // A: thread loads row ar, columns ac .. ac + 4 LV - 1 of the 16-wide K slice
    const int ar = tid & (TILE - 1), ac = (tid / TILE) * 4 * LV;
    // B: thread loads row br, columns bc .. bc + 4 LV - 1
    const int br = tid / (TILE / (4 * LV)), bc = (tid % (TILE / (4 * LV))) * 4 * LV;
    floatx16 acc[MB][MB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

    floatx4 ra[LV], rb[LV];
    const floatx4* sa = reinterpret_cast<const floatx4*>(A + (size_t)(bm + ar) * K + ac);
    const floatx4* sb = reinterpret_cast<const floatx4*>(B + (size_t)br * N + bn + bc);
#pragma unroll
    for (int q = 0; q < LV; ++q) {
        ra[q] = sa[q];
        rb[q] = sb[q];
    }
    for (int k0 = 0; k0 < K; k0 += GBK) {
        const bool row = k0 + br < np;
#pragma unroll
        for (int q = 0; q < LV; ++q) {
            As[ac + 4 * q + 0][ar] = ra[q][0];
            As[ac + 4 * q + 1][ar] = ra[q][1];
            As[ac + 4 * q + 2][ar] = ra[q][2];
            As[ac + 4 * q + 3][ar] = ra[q][3];
            const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<floatx4*>(&Bs[br][bc + 4 * q]) = row ? rb[q] : zero;
        }
        __syncthreads();
        // prefetch the next K slice; the last step re-reads its own slice
        // (in bounds) so that the loads stay unconditional and ra/rb stay in
        // registers
        if (k0 + GBK < K) {
            sa += GBK / 4;
            sb += (size_t)GBK * N / 4;
        }
#pragma unroll
        for (int q = 0; q < LV; ++q) {
            ra[q] = sa[q];
            rb[q] = sb[q];
        }
#pragma unroll
        for (int kk = 0; kk < GBK; kk += 2) {
            const int kr = kk + (lane >> 5);
            float av[MB], bv[MB];
#pragma unroll
            for (int q = 0; q < MB; ++q) {
                av[q] = As[kr][wm + 32 * q + (lane & 31)];
                bv[q] = Bs[kr][wn + 32 * q + (lane & 31)];
            }
#pragma unroll
            for (int mi = 0; mi < MB; ++mi)
#pragma unroll
                for (int ni = 0; ni < MB; ++ni)
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[mi], bv[ni], acc[mi][ni], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int mi = 0; mi < MB; ++mi)
#pragma unroll
        for (int ni = 0; ni < MB; ++ni)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = bm + wm + mi * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                const int col = bn + wn + ni * 32 + (lane & 31);
                C[(size_t)row * N + col] = acc[mi][ni][v];
            }
}

// C = A B on the FP16 matrix cores with FP32-like accuracy: each operand
// arrives split into two fp16 halves, x = hi + lo (hi = fp16(x), lo =
// fp16(x - hi): 22 significant bits together), and C accumulates
// hi_a hi_b + hi_a lo_b + lo_a hi_b in FP32; the dropped lo_a lo_b term is
// below 2^-22 of |a||b|.  A is [M][K] (k fastest, halves Ah then Al), B is
// given transposed, [N][K] (Bh then Bl), scaled by a power of two whose
// inverse bsc[1] multiplies C at the end (exact).  Tiles of 128 x 128, K
// steps of 32 (K a multiple of 32), 4 waves of 2 x 2 blocks of
// v_mfma_f32_32x32x16_f16 (gfx950): lane l takes A[l % 32][8 (l / 32) + j]
// and B[8 (l / 32) + j][l % 32], j = 0..7, and holds the 32x32 accumulator
// as the FP32 MFMA does.  In LDS the tiles keep k fastest (rows of 40
// halves), so each lane reads its 8 halves with one 16-byte load, and every
// global load is a 16-byte copy.
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
constexpr int HK = 32;    // K step of the split FP16 GEMM
constexpr int HROW = 40;  // LDS row stride in halves: 32 of K plus 8 of padding

__global__ __launch_bounds__(256) void k_hgemm3(const FaceDev* __restrict__ fc, const ChunkDev* __restrict__ ch,
                                               int nf) {
    constexpr int TILE = 128, MB = 2;
    const int fi = face_of_block(ch, nf, KIND_SPLIT16);
    const FaceDev& fd = fc[fi];
    const int N = fd.N, K = fd.K, tile = blockIdx.x - ch[fi].first, tn = N / TILE;
    const _Float16* __restrict__ Ahi = reinterpret_cast<const _Float16*>(fd.A);
    const _Float16* __restrict__ Alo = Ahi + (size_t)ch[fi].M * K;
    const _Float16* __restrict__ Bhi = fd.Bhi;
    const _Float16* __restrict__ Blo = fd.Blo;
    float* __restrict__ C = fd.G;
    const float* __restrict__ bsc = fd.bsc;
    __shared__ __align__(16) _Float16 Ah[TILE][HROW];
    __shared__ __align__(16) _Float16 Al[TILE][HROW];
    __shared__ __align__(16) _Float16 Bh[TILE][HROW];
    __shared__ __align__(16) _Float16 Bl[TILE][HROW];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int bm = tile / tn * TILE, bn = tile % tn * TILE;
    const int wm = (wave >> 1) * (TILE / 2), wn = (wave & 1) * (TILE / 2);
    // every thread copies 16 halves (2 x 16 B) of one row of each of the four tiles
    const int r = tid >> 1, kq = (tid & 1) * 16;
    floatx16 acc[MB][MB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;
    half8 ga[4], gb[4];  // [hi 0..7, hi 8..15, lo 0..7, lo 8..15] of this thread's row segment
    auto load = [&](int k0) {
        const _Float16* pa = Ahi + (size_t)(bm + r) * K + k0 + kq;
        const _Float16* pl = Alo + (size_t)(bm + r) * K + k0 + kq;
        const _Float16* pb = Bhi + (size_t)(bn + r) * K + k0 + kq;
        const _Float16* ql = Blo + (size_t)(bn + r) * K + k0 + kq;
        ga[0] = *reinterpret_cast<const half8*>(pa);
        ga[1] = *reinterpret_cast<const half8*>(pa + 8);
        ga[2] = *reinterpret_cast<const half8*>(pl);
        ga[3] = *reinterpret_cast<const half8*>(pl + 8);
        gb[0] = *reinterpret_cast<const half8*>(pb);
        gb[1] = *reinterpret_cast<const half8*>(pb + 8);
        gb[2] = *reinterpret_cast<const half8*>(ql);
        gb[3] = *reinterpret_cast<const half8*>(ql + 8);
    };
    load(0);
    for (int k0 = 0; k0 < K; k0 += HK) {
        *reinterpret_cast<half8*>(&Ah[r][kq]) = ga[0];
        *reinterpret_cast<half8*>(&Ah[r][kq + 8]) = ga[1];
        *reinterpret_cast<half8*>(&Al[r][kq]) = ga[2];
        *reinterpret_cast<half8*>(&Al[r][kq + 8]) = ga[3];
        *reinterpret_cast<half8*>(&Bh[r][kq]) = gb[0];
        *reinterpret_cast<half8*>(&Bh[r][kq + 8]) = gb[1];
        *reinterpret_cast<half8*>(&Bl[r][kq]) = gb[2];
        *reinterpret_cast<half8*>(&Bl[r][kq + 8]) = gb[3];
        __syncthreads();
        if (k0 + HK < K) load(k0 + HK);
#pragma unroll
        for (int kk = 0; kk < HK; kk += 16) {
            const int kc = kk + 8 * (lane >> 5);
            half8 ah[MB], al[MB], bh[MB], bl[MB];
#pragma unroll
            for (int q = 0; q < MB; ++q) {
                ah[q] = *reinterpret_cast<const half8*>(&Ah[wm + 32 * q + (lane & 31)][kc]);
                al[q] = *reinterpret_cast<const half8*>(&Al[wm + 32 * q + (lane & 31)][kc]);
                bh[q] = *reinterpret_cast<const half8*>(&Bh[wn + 32 * q + (lane & 31)][kc]);
                bl[q] = *reinterpret_cast<const half8*>(&Bl[wn + 32 * q + (lane & 31)][kc]);
            }
#pragma unroll
            for (int mi = 0; mi < MB; ++mi)
#pragma unroll
                for (int ni = 0; ni < MB; ++ni) {
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[mi], bh[ni], acc[mi][ni], 0, 0, 0);
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mi], bl[ni], acc[mi][ni], 0, 0, 0);
                    acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[mi], bh[ni], acc[mi][ni], 0, 0, 0);
                }
        }
        __syncthreads();
    }
    const float cs = bsc[1];
#pragma unroll
    for (int mi = 0; mi < MB; ++mi)
#pragma unroll
        for (int ni = 0; ni < MB; ++ni)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = bm + wm + mi * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                const int col = bn + wn + ni * 32 + (lane & 31);
                C[(size_t)row * N + col] = acc[mi][ni][v] * cs;
            }
}

// B [K][N] float -> Bhi, Blo [N][K] halves of B s, s = 2^(14 - e) for the
// largest entry m = f 2^e (0.5 <= f < 1) of the pack's block maxima
// pmax[0..nb) (s = 1 when m is 0 or not finite), so every scaled entry is
// below 2^14.  Entries outside the packed p < np, n < 8 nq (padding, which may
// hold an earlier face's values) are written as zeros.  64 x 64 tiles through
// LDS: reads along n, writes along k.  The first work-group stores (s, 1 / s).
__device__ __forceinline__ void bsplit(const FaceDev& f) {
    __shared__ float red[256];
    __shared__ float t[64][65];
    const int tid = threadIdx.x, K = f.K, N = f.N, nv = 8 * f.nq;
    float m = 0.f;
    for (int q = tid; q < f.nb; q += 256) m = fmaxf(m, f.pmax[q]);
    red[tid] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) red[tid] = fmaxf(red[tid], red[tid + o]);
        __syncthreads();
    }
    float sc = 1.f, inv = 1.f;
    if (red[0] > 0.f && red[0] < 3.0e38f) {
        int e = 0;
        (void)frexpf(red[0], &e);
        sc = ldexpf(1.f, 14 - e);
        inv = ldexpf(1.f, e - 14);
    }
    if (blockIdx.x == 0 && tid == 0) {
        f.bsc[0] = sc;
        f.bsc[1] = inv;
    }
    const int tn = N / 64, tiles = tn * ((K + 63) / 64);
    const int tx = tid & 63, ty = tid >> 6;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int k0 = tile / tn * 64, n0 = tile % tn * 64;
        for (int y = ty; y < 64; y += 4) {
            const int k = k0 + y, n = n0 + tx;
            t[y][tx] = (k < f.np && n < nv) ? f.B[(size_t)k * N + n] * sc : 0.f;
        }
        __syncthreads();
        for (int y = ty; y < 64; y += 4) {
            const int n = n0 + y, k = k0 + tx;
            if (k < K) {
                const float x = t[tx][y];
                const _Float16 h = (_Float16)x;
                f.Bhi[(size_t)n * K + k] = h;
                f.Blo[(size_t)n * K + k] = (_Float16)(x - (float)h);
            }
        }
        __syncthreads();
    }
}

// Rows of A in float32: row r of the chunk holds cos (even r) or sin (odd r)
// of k uval[u] xp[i], u = u0 + r / 2, for u < u1 and i < np, zeros elsewhere.
__device__ __forceinline__ void phase_rows(const FaceDev& f, const ChunkDev& c, double k) {
    const size_t total = (size_t)c.M * f.K;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < total; t += (size_t)gridDim.x * 256) {
        const int r = (int)(t / f.K), i = (int)(t - (size_t)r * f.K);
        const int u = c.u0 + (r >> 1);
        float v = 0.f;
        if (u < c.u1 && i < f.np) {
            double sn, cs;
            sincos(k * f.uval[u] * f.xp[i], &sn, &cs);
            v = (float)((r & 1) ? sn : cs);
        }
        f.A[t] = v;
    }
}

// The same rows as fp16 halves (hi, then lo, of the float64 value).  One
// thread per 8 consecutive columns of a row (K is a multiple of 8); on a
// uniform grid (xp[i] = xp[0] + i dxp) the thread takes one sincos and steps
// the other 7 columns by angle addition in float64.
__device__ __forceinline__ void phase_rows16(const FaceDev& f, const ChunkDev& c, double k) {
    const size_t total = (size_t)c.M * f.K, groups = total / 8;
    _Float16* Ahi = reinterpret_cast<_Float16*>(f.A);
    _Float16* Alo = Ahi + total;
    for (size_t g = (size_t)blockIdx.x * 256 + threadIdx.x; g < groups; g += (size_t)gridDim.x * 256) {
        const size_t t0 = 8 * g;
        const int r = (int)(t0 / f.K), i0 = (int)(t0 - (size_t)r * f.K);
        const int u = c.u0 + (r >> 1);
        const bool odd = (r & 1) != 0;
        half8 h, l;
        if (u < c.u1 && i0 < f.np) {
            const double ku = k * f.uval[u];
            double sn, cs, sd = 0.0, cd = 1.0;
            sincos(ku * f.xp[i0], &sn, &cs);
            if (f.uni_p) sincos(ku * f.dxp, &sd, &cd);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                double v = 0.0;
                if (i0 + q < f.np) {
                    if (!f.uni_p && q > 0) sincos(ku * f.xp[i0 + q], &sn, &cs);
                    v = odd ? sn : cs;
                }
                h[q] = (_Float16)v;
                l[q] = (_Float16)(v - (double)h[q]);
                if (f.uni_p) {
                    const double c2 = cs * cd - sn * sd;
                    sn = sn * cd + cs * sd;
                    cs = c2;
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q) h[q] = l[q] = (_Float16)0.f;
        }
        *reinterpret_cast<half8*>(Ahi + t0) = h;
        *reinterpret_cast<half8*>(Alo + t0) = l;
    }
}

__device__ __forceinline__ void chunk_rows(const FaceDev& f, const ChunkDev& c, double k) {
    if (c.M == 0) return;
    if (c.kind == KIND_SPLIT16) phase_rows16(f, c, k);
    else phase_rows(f, c, k);
}

// The contraction's operands of the first chunk, every face in one launch:
// grid (work-groups, face, 2), z = 0 the phase rows, z = 1 the split of B for
// the faces that need it.  The rows of the chunks that follow are formed in
// the launch of the reduction before them (next): A is free by then, and the
// arithmetic of the rows (31 us a chunk) runs beside the reduction's loads.
__global__ __launch_bounds__(256) void k_nf2ff_operands(const FaceDev* __restrict__ fc, const ChunkDev* __restrict__ ch,
                                                        double k) {
    const FaceDev& f = fc[blockIdx.y];
    if (blockIdx.z == 0) chunk_rows(f, ch[blockIdx.y], k);
    else if (f.split) bsplit(f);
}

// The large contractions on the FP16 matrix cores when split16 (operands
// split into fp16 halves), the others in FP32.
int gemm_kind(int M, int N, bool split16) {
    const bool large = (M / 128) * (N / 128) >= 512;
    return !large ? KIND_FP32 : split16 ? KIND_SPLIT16 : KIND_FP32_LARGE;
}

// B = [Br | Bi] for one face: row ip, columns 4 iq + c and 4 nq + 4 iq + c
// hold w_p[ip] times the equivalent current c = (J_a1, J_a2, M_a1, M_a2) at
// node (i1, i2) (ip = i1, iq = i2, or swapped when swap = 1), with J = n x H
// and M = -n x E (matlab/AnalyzeNF2FF.m:186-191): J_a1 = -s H_a2,
// J_a2 = s H_a1, M_a1 = s E_a2, M_a2 = -s E_a1 for the outward normal
// n = s e_axis.  The block partial of the radiated power,
// 1/2 sum w_p w_q Re((E x H*) . n) (matlab/AnalyzeNF2FF.m:201-209), goes to
// part[blockIdx.x].
__global__ __launch_bounds__(256) void k_nf2ff_pack(const FaceDev* __restrict__ fc) {
    const FaceDev& f = fc[blockIdx.y];
    if ((int)blockIdx.x >= f.nb) return;
    __shared__ double red[256];
    __shared__ float redm[256];
    const int tid = threadIdx.x, n1 = f.n1, n2 = f.n2;
    const int q = blockIdx.x * 256 + tid;
    double p = 0.0;
    float mx = 0.f;
    if (q < n1 * n2) {
        const int i1 = q / n2, i2 = q - i1 * n2;
        const int ip = f.swap ? i2 : i1, iq = f.swap ? i1 : i2, nq = f.nq;
        double vr[4], vi[4];
        if (f.kind == 0) {
            const double2* v = reinterpret_cast<const double2*>(f.src) + 4 * (size_t)q;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                vr[c] = f.scale * v[c].x;
                vi[c] = f.scale * v[c].y;
            }
        } else {
            const float4* v = reinterpret_cast<const float4*>(f.src) + 4 * (size_t)q;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                vr[c] = f.scale * (double)v[c].x;
                vi[c] = f.scale * (double)v[c].y;
            }
        }
        const double sg = f.sign, w = f.wp[ip];
        const double cr[4] = {-sg * vr[3], sg * vr[2], sg * vr[1], -sg * vr[0]};
        const double ci[4] = {-sg * vi[3], sg * vi[2], sg * vi[1], -sg * vi[0]};
        float* row = f.B + (size_t)ip * f.N;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float br = (float)(w * cr[c]), bi = (float)(w * ci[c]);
            row[4 * iq + c] = br;
            row[4 * nq + 4 * iq + c] = bi;
            mx = fmaxf(mx, fmaxf(fabsf(br), fabsf(bi)));
        }
        p = 0.5 * w * f.wq[iq] * sg * (vr[0] * vr[3] + vi[0] * vi[3] - vr[1] * vr[2] - vi[1] * vi[2]);
    }
    red[tid] = p;
    redm[tid] = mx;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            red[tid] += red[tid + o];
            redm[tid] = fmaxf(redm[tid], redm[tid + o]);
        }
        __syncthreads();
    }
    if (tid == 0) {
        f.part[blockIdx.x] = red[0];
        f.pmax[blockIdx.x] = redm[0];
    }
}

#ifndef REDUCE_M
#define REDUCE_M 2  // 2: 0.894 ms device per frequency; 3: 0.978; 4: 0.914 (fewer waves)
#endif
// e^{j pi x}, x in half turns reduced to one turn first.
__device__ __forceinline__ void cis_pi(double x, double* c, double* s) {
    sincospi(x - 2.0 * rint(0.5 * x), s, c);
}

// Second contraction, one group of angles at a time: the angles of a group
// share one G row (the same |kappa_p|), so each G load serves all of them.
// QL lanes split the q sum (lane l takes q = l, l + QL, ...; consecutive
// lanes read consecutive G entries); the QL partial sums of every angle are
// added by a fixed xor butterfly (deterministic) and the group's first lane
// stores the results, rotated by the face-position phase, as the face's sums.  G = GC -/+
// j GS is formed in float32 (one rounding of the matrix-core output, 6e-8
// relative); the phase products are accumulated in float64 with fused
// multiply-adds.
constexpr int QL = 16;
constexpr int REDUCE_THREADS = 256;
constexpr int REDUCE_GROUPS = REDUCE_THREADS / QL;

__global__ __launch_bounds__(REDUCE_THREADS) void k_nf2ff_reduce(const FaceDev* __restrict__ fc,
                                                                 const ChunkDev* __restrict__ ch,
                                                                 const ChunkDev* __restrict__ next, int kinds,
                                                                 double k) {
    constexpr int M = REDUCE_M;
    const FaceDev& r = fc[blockIdx.y];
    if (blockIdx.z == 1) {
        chunk_rows(r, next[blockIdx.y], k);
        return;
    }
    const ChunkDev& ck = ch[blockIdx.y];
    if (ck.mirror || !takes(ck, kinds)) return;
    const int ql = threadIdx.x & (QL - 1);
    const int gi = ck.g0 + blockIdx.x * REDUCE_GROUPS + (int)(threadIdx.x / QL);
    if (gi >= ck.g1) return;  // whole groups of QL lanes
    const int2 grp = r.groups[gi];
    const int n = grp.y, nq = r.nq;
    const double kp = k * M_1_PI;
    int am[M];
    float sgf[M];
    double pr[M], pi[M], str[M], sti[M];
    double sr[M][4], si[M][4];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        am[m] = r.order[grp.x + min(m, grp.y - 1)];
        sgf[m] = r.usgn[am[m]];
        const double kk = kp * r.kapq[am[m]];
        pr[m] = 1.0; pi[m] = 0.0; str[m] = 1.0; sti[m] = 0.0;
        if (r.uni_q && ql < nq) {
            cis_pi(kk * r.xq[ql], &pr[m], &pi[m]);
            cis_pi(kk * (QL * r.dxq), &str[m], &sti[m]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) sr[m][c] = si[m][c] = 0.0;
    }
    const float* gc = r.G + (size_t)(2 * (r.uidx[am[0]] - ck.u0)) * r.N;
    const float* gs = gc + r.N;
    auto body = [&](int iq, bool uniform) {
        const float4 cr4 = *reinterpret_cast<const float4*>(gc + 4 * iq);
        const float4 ci4 = *reinterpret_cast<const float4*>(gc + 4 * nq + 4 * iq);
        const float4 sr4 = *reinterpret_cast<const float4*>(gs + 4 * iq);
        const float4 si4 = *reinterpret_cast<const float4*>(gs + 4 * nq + 4 * iq);
        const double w = r.wq[iq];
        const float gcr[4] = {cr4.x, cr4.y, cr4.z, cr4.w}, gci[4] = {ci4.x, ci4.y, ci4.z, ci4.w};
        const float gsr[4] = {sr4.x, sr4.y, sr4.z, sr4.w}, gsi[4] = {si4.x, si4.y, si4.z, si4.w};
#pragma unroll
        for (int m = 0; m < M; ++m) {
            double cs = pr[m], sn = pi[m];
            if (uniform) {
                const double t = pr[m] * str[m] - pi[m] * sti[m];
                pi[m] = pr[m] * sti[m] + pi[m] * str[m];
                pr[m] = t;
            } else {
                cis_pi(kp * r.kapq[am[m]] * r.xq[iq], &cs, &sn);
            }
            const double wr = w * cs, wi = w * sn;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const double gr = (double)(gcr[c] - sgf[m] * gsi[c]);
                const double gi = (double)(gci[c] + sgf[m] * gsr[c]);
                sr[m][c] = fma(wr, gr, fma(-wi, gi, sr[m][c]));
                si[m][c] = fma(wr, gi, fma(wi, gr, si[m][c]));
            }
        }
    };
    if (r.uni_q) {
        for (int iq = ql; iq < nq; iq += QL) body(iq, true);
    } else {
        for (int iq = ql; iq < nq; iq += QL) body(iq, false);
    }
#pragma unroll
    for (int o = QL / 2; o > 0; o >>= 1)
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                sr[m][c] += __shfl_xor(sr[m][c], o, QL);
                si[m][c] += __shfl_xor(si[m][c], o, QL);
            }
    if (ql != 0) return;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        if (m >= n) break;
        const int a = am[m];
        double sn, cs;
        cis_pi(kp * r.kap0[a] * r.x0, &cs, &sn);
        double2* o = reinterpret_cast<double2*>(r.S) + (size_t)a * 4;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            o[c] = make_double2(cs * sr[m][c] - sn * si[m][c], cs * si[m][c] + sn * sr[m][c]);
    }
}

// Second contraction over mirror groups: the angles of one G row (one |kappa_p|)
// whose |kappa_q| also agree, e.g. (theta, pi - theta) x (phi, -phi, pi - phi,
// pi + phi) on a regular grid.  With sigma = sign kappa_p and s = sign kappa_q,
// a member's sum
//   sum_q w_q e^{j s k |kappa_q| x_q} (GC_q + j sigma GS_q)
//     = P1 + j sigma P2 + j s P3 - s sigma P4,
//   P1 = sum w cos GC, P2 = sum w cos GS, P3 = sum w sin GC, P4 = sum w sin GS,
// needs only the group's four partial sums (phase k |kappa_q| x_q of the
// group's first member; members agree to 1e-12 in |kappa_q|).  Each G row is
// read once per group, and the float64 work per q is that of one angle for
// the whole group.
//
// 4 MQ lanes per group: lane = 4 ql + c takes component c at q = ql, ql + MQ,
// ... (the four lanes of one ql read 16 consecutive bytes), with eight float64
// accumulators, and issues the loads of four q steps before using them.  The
// MQ lanes of each component are added by row rotations (MQ = 4: a group is
// one 16-lane row), and lane (ql, c) then finishes component c of members ql,
// ql + MQ, ...  What bounds it is instructions: for each group the start and
// end phases (three sincos) and the sums over lanes cost as much as the steps
// in q when a whole wave works on one group, so a wave takes four groups.
// 65160 angles, 349x349x221 nodes: the six faces take 106 us, against 6 x 32
// with a wave a group.
constexpr int MIRROR_MAX = 16;  // most members of a group
constexpr int MQ = 4;
constexpr int MIRROR_THREADS = 256;
constexpr int MIRROR_GROUPS = MIRROR_THREADS / (4 * MQ);

// v of the lane n further on in its row of 16.
template <int N>
__device__ __forceinline__ double row_ror(double v) {
    union {
        double d;
        int i[2];
    } x{v};
    x.i[0] = __builtin_amdgcn_update_dpp(0, x.i[0], 0x120 + N, 0xf, 0xf, true);
    x.i[1] = __builtin_amdgcn_update_dpp(0, x.i[1], 0x120 + N, 0xf, 0xf, true);
    return x.d;
}
__device__ __forceinline__ void add_lanes(double& v) {
    v += row_ror<4>(v);
    v += row_ror<8>(v);
#pragma unroll
    for (int o = 16; o < 4 * MQ; o <<= 1) v += __shfl_xor(v, o);
}

// UNI: uniform q grid (phases by recurrence)
template <bool UNI>
__device__ __forceinline__ void mirror_reduce(const FaceDev& r, const ChunkDev& ck, double k) {
    const int gi = ck.g0 + blockIdx.x * MIRROR_GROUPS + (int)(threadIdx.x / (4 * MQ));
    const bool on = gi < ck.g1;  // every lane takes part in the rotations
    const int c = threadIdx.x & 3;
    const int ql = (threadIdx.x >> 2) & (MQ - 1);
    const int4 grp = r.mgroups[on ? gi : ck.g0];
    const int nq = on ? r.nq : 0;
    const double kp = k * M_1_PI, kk = kp * r.gkq[on ? gi : ck.g0];
    double pr = 1.0, pi = 0.0, str = 1.0, sti = 0.0;
    if (UNI && ql < nq) {
        cis_pi(kk * r.xq[ql], &pr, &pi);
        cis_pi(kk * (MQ * r.dxq), &str, &sti);
    }
    // P1..P4 of component c, real and imaginary
    double p1r = 0.0, p1i = 0.0, p2r = 0.0, p2i = 0.0, p3r = 0.0, p3i = 0.0, p4r = 0.0, p4i = 0.0;
    const float* gc = r.G + (size_t)(2 * (grp.x - ck.u0)) * r.N + c;
    const float* gs = gc + r.N;
    const double* __restrict__ wq = r.wq;
    const int n4 = 4 * r.nq;
    auto step = [&](int q, float a, float b, float e, float f, double w) {
        double cs = pr, sn = pi;
        if (UNI) {
            const double t = pr * str - pi * sti;
            pi = pr * sti + pi * str;
            pr = t;
        } else {
            cis_pi(kk * r.xq[q], &cs, &sn);
        }
        const double wc = w * cs, ws = w * sn;
        p1r = fma(wc, (double)a, p1r);
        p1i = fma(wc, (double)b, p1i);
        p2r = fma(wc, (double)e, p2r);
        p2i = fma(wc, (double)f, p2i);
        p3r = fma(ws, (double)a, p3r);
        p3i = fma(ws, (double)b, p3i);
        p4r = fma(ws, (double)e, p4r);
        p4i = fma(ws, (double)f, p4i);
    };
    int iq = ql;
    for (; iq + 3 * MQ < nq; iq += 4 * MQ) {
        float va[4], vb[4], ve[4], vf[4];
        double vw[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int q = iq + u * MQ;
            va[u] = gc[4 * q];
            vb[u] = gc[n4 + 4 * q];
            ve[u] = gs[4 * q];
            vf[u] = gs[n4 + 4 * q];
            vw[u] = wq[q];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) step(iq + u * MQ, va[u], vb[u], ve[u], vf[u], vw[u]);
    }
    for (; iq < nq; iq += MQ) step(iq, gc[4 * iq], gc[n4 + 4 * iq], gs[4 * iq], gs[n4 + 4 * iq], wq[iq]);
    add_lanes(p1r);
    add_lanes(p1i);
    add_lanes(p2r);
    add_lanes(p2i);
    add_lanes(p3r);
    add_lanes(p3i);
    add_lanes(p4r);
    add_lanes(p4i);
    if (!on) return;
    for (int m = ql; m < grp.z; m += MQ) {
        const int a = r.members[grp.y + m];
        const double sg = (double)r.usgn[a];
        const double s = r.kapq[a] < 0.0 ? -1.0 : 1.0;
        const double ss = s * sg;
        double sn, cs;
        cis_pi(kp * r.kap0[a] * r.x0, &cs, &sn);
        // P1 + j sigma P2 + j s P3 - s sigma P4
        const double tr = p1r - sg * p2i - s * p3i - ss * p4r;
        const double ti = p1i + sg * p2r + s * p3r - ss * p4i;
        reinterpret_cast<double2*>(r.S)[(size_t)a * 4 + c] = make_double2(cs * tr - sn * ti, cs * ti + sn * tr);
    }
}

__global__ __launch_bounds__(MIRROR_THREADS) void k_nf2ff_reduce_mirror(const FaceDev* __restrict__ fc,
                                                                        const ChunkDev* __restrict__ ch,
                                                                        const ChunkDev* __restrict__ next, int kinds,
                                                                        double k) {
    const FaceDev& r = fc[blockIdx.y];
    if (blockIdx.z == 1) {
        chunk_rows(r, next[blockIdx.y], k);
        return;
    }
    const ChunkDev& ck = ch[blockIdx.y];
    if (!ck.mirror || !takes(ck, kinds) || ck.g0 + (int)blockIdx.x * MIRROR_GROUPS >= ck.g1) return;
    if (r.uni_q) mirror_reduce<true>(r, ck, k);
    else mirror_reduce<false>(r, ck, k);
}

// N, L of angle a: nl (or zero) plus the faces' sums, in face order.
__device__ __forceinline__ void gather_nl(const FaceDev* __restrict__ fc, int nf, const double* __restrict__ nl,
                                          size_t a, double* v) {
#pragma unroll
    for (int c = 0; c < 12; ++c) v[c] = nl ? nl[12 * a + c] : 0.0;
    for (int f = 0; f < nf; ++f) {
        const double2* S = reinterpret_cast<const double2*>(fc[f].S) + 4 * a;
        const int a1 = fc[f].a1;  // a2 = a1 + 1 cyclically
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const double2 s = S[c];
            const int slot = (c >= 2 ? 3 : 0) + ((c & 1) ? (a1 == 2 ? 0 : a1 + 1) : a1);
#pragma unroll
            for (int q = 0; q < 6; ++q)
                if (q == slot) {
                    v[2 * q] += s.x;
                    v[2 * q + 1] += s.y;
                }
        }
    }
}

// Surfaces of more than one set of faces: the sums of one set.
__global__ __launch_bounds__(256) void k_nf2ff_gather(const FaceDev* __restrict__ fc, int nf, double* nl, int first,
                                                      size_t n_ang) {
    const size_t a = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (a >= n_ang) return;
    double v[12];
    gather_nl(fc, nf, first ? nullptr : nl, a, v);
#pragma unroll
    for (int c = 0; c < 12; ++c) nl[12 * a + c] = v[c];
}

// E_theta = -fac (L_phi + Z0 N_theta), E_phi = fac (L_theta - Z0 N_phi) with
// fac = jk e^{-jkr}/(4 pi r) (matlab/AnalyzeNF2FF.m:98-105) and
// U = r^2/(2 Z0)(|E_theta|^2 + |E_phi|^2) (:112): out = [4][n_ang]
// (E_theta re, im, E_phi re, im); the block maximum of U goes to umax[block].
__global__ __launch_bounds__(256) void k_nf2ff_project(const FaceDev* __restrict__ fc, int nf,
                                                       const double* __restrict__ nl,
                                                       const double* __restrict__ theta,
                                                       const double* __restrict__ phi, int n_phi, size_t n_ang,
                                                       double fr, double fi, double r, double* __restrict__ out,
                                                       double* __restrict__ umax) {
    __shared__ double red[256];
    const size_t a = (size_t)blockIdx.x * 256 + threadIdx.x;
    double u = 0.0;
    if (a < n_ang) {
        const int it = (int)(a / n_phi), ip = (int)(a - (size_t)it * n_phi);
        double st, ct, sp, cp;
        sincos(theta[it], &st, &ct);
        sincos(phi[ip], &sp, &cp);
        double v[12];
        gather_nl(fc, nf, nl, a, v);
        const double ntr = v[0] * (ct * cp) + v[2] * (ct * sp) - v[4] * st;
        const double nti = v[1] * (ct * cp) + v[3] * (ct * sp) - v[5] * st;
        const double npr = -v[0] * sp + v[2] * cp, npi = -v[1] * sp + v[3] * cp;
        const double ltr = v[6] * (ct * cp) + v[8] * (ct * sp) - v[10] * st;
        const double lti = v[7] * (ct * cp) + v[9] * (ct * sp) - v[11] * st;
        const double lpr = -v[6] * sp + v[8] * cp, lpi = -v[7] * sp + v[9] * cp;
        const double ar = lpr + Z0 * ntr, ai = lpi + Z0 * nti;  // E_theta = -fac * A
        const double br = ltr - Z0 * npr, bi = lti - Z0 * npi;  // E_phi = fac * B
        const double etr = -(fr * ar - fi * ai), eti = -(fr * ai + fi * ar);
        const double epr = fr * br - fi * bi, epi = fr * bi + fi * br;
        // interleaved complex: [E_theta][a][re, im], then [E_phi][a][re, im]
        out[2 * a] = etr;
        out[2 * a + 1] = eti;
        out[2 * n_ang + 2 * a] = epr;
        out[2 * n_ang + 2 * a + 1] = epi;
        u = r * r / (2.0 * Z0) * (etr * etr + eti * eti + epr * epr + epi * epi);
    }
    red[threadIdx.x] = u;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) umax[blockIdx.x] = red[0];
}

inline size_t round_up(size_t v, size_t m) { return (v + m - 1) / m * m; }

std::vector<double> trapz_weights(const std::vector<double>& c) {
    std::vector<double> w(c.size(), 0.0);
    for (size_t i = 0; i + 1 < c.size(); ++i) {
        const double h = 0.5 * (c[i + 1] - c[i]);
        w[i] += h;
        w[i + 1] += h;
    }
    return w;
}

// x[i] == x[0] + i * d within 1e-9 d
bool uniform_spacing(const std::vector<double>& x, double* d) {
    *d = x.size() > 1 ? (x.back() - x.front()) / (double)(x.size() - 1) : 0.0;
    for (size_t i = 0; i < x.size(); ++i)
        if (std::fabs(x[i] - (x.front() + (double)i * *d)) > 1e-9 * std::fabs(*d)) return false;
    return true;
}

struct EventPair {
    hipEvent_t a = nullptr, b = nullptr;
    EventPair() = default;
    EventPair(const EventPair&) = delete;
    EventPair& operator=(const EventPair&) = delete;
    ~EventPair() {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
    }
};

#define NF_OK(expr)                              \
    do {                                         \
        hipError_t _e = (expr);                  \
        if (_e != hipSuccess) return _e;         \
    } while (0)

}  // namespace

// Angle plan and work buffers, kept between calls with the same angles.
struct PinnedBuf {
    void* p = nullptr;
    size_t bytes = 0;
    PinnedBuf() = default;
    PinnedBuf(const PinnedBuf&) = delete;
    PinnedBuf& operator=(const PinnedBuf&) = delete;
    ~PinnedBuf() { if (p) (void)hipHostFree(p); }
    hipError_t alloc(size_t n) {
        if (p) { (void)hipHostFree(p); p = nullptr; }
        bytes = 0;  // as DevBuf
        const hipError_t e = n ? hipHostMalloc(&p, n, hipHostMallocDefault) : hipSuccess;
        if (e == hipSuccess) bytes = n;
        else p = nullptr;
        return e;
    }
};

struct Nf2ffCache {
    std::vector<double> theta, phi;
    size_t n_ang = 0;
    DevBuf kap;  // [3][n_ang] double, then theta[nt], phi[np]
    PinnedBuf host;  // far-field staging
    struct Axis {
        int U = 0;
        std::vector<int> start;  // U + 1 offsets into order
        std::vector<int> gstart; // U + 1 offsets into groups
        DevBuf groups;           // int2 per group: first index into order, angle count (<= REDUCE_M)
        DevBuf uval;             // U doubles (|kappa| of each distinct value)
        DevBuf uidx;             // n_ang ints
        DevBuf usgn;             // n_ang floats
        DevBuf order;            // n_ang ints, angles sorted by u
        std::vector<int> horder; // host copy of order
    } ax[3];
    // Mirror groups of the faces normal to each axis (k_nf2ff_reduce_mirror):
    // the angles of every row u of that face's first-contraction axis,
    // grouped by equal |kappa| along its second axis, at most MIRROR_MAX each.
    struct Mirror {
        std::vector<int> mstart;  // U + 1 offsets into groups
        DevBuf groups;            // int4 (u, first index into members, count, 0)
        DevBuf gkq;               // double per group
        DevBuf members;           // n_ang ints
    } mir[3];
    DevBuf work;
    // timing events, created on first use and kept: [0] brackets the whole
    // transform, the others one GEMM launch each
    std::vector<std::unique_ptr<EventPair>> events;
    // beside the large contractions: the faces of the small ones
    hipStream_t side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    ~Nf2ffCache() {
        if (side) (void)hipStreamSynchronize(side);
        if (fork) (void)hipEventDestroy(fork);
        if (join) (void)hipEventDestroy(join);
        if (side) (void)hipStreamDestroy(side);
    }
    Nf2ffCache() = default;
    Nf2ffCache(const Nf2ffCache&) = delete;
    Nf2ffCache& operator=(const Nf2ffCache&) = delete;
};

Nf2ffCache* nf2ff_cache_new() { return new Nf2ffCache(); }
void nf2ff_cache_free(Nf2ffCache* c) { delete c; }

// The faces normal to axis f contract first over the in-plane axis p with
// fewer distinct |kappa| (fewer GEMM rows), then over the other, q.
static void face_axes(const Nf2ffCache& c, int f, int* p, int* q) {
    const int a1 = (f + 1) % 3, a2 = (f + 2) % 3;
    const bool swap = c.ax[a2].U < c.ax[a1].U;
    *p = swap ? a2 : a1;
    *q = swap ? a1 : a2;
}

static hipError_t plan_angles(Nf2ffCache& c, const double* theta, int nt, const double* phi, int np, hipStream_t s) {
    if (c.n_ang && c.theta.size() == (size_t)nt && c.phi.size() == (size_t)np &&
        std::equal(c.theta.begin(), c.theta.end(), theta) && std::equal(c.phi.begin(), c.phi.end(), phi))
        return hipSuccess;
    c.n_ang = 0;
    const size_t n = (size_t)nt * np;
    std::vector<double> kap(3 * n);
    for (int it = 0; it < nt; ++it)
        for (int ip = 0; ip < np; ++ip) {
            const size_t a = (size_t)it * np + ip;
            kap[a] = std::sin(theta[it]) * std::cos(phi[ip]);
            kap[n + a] = std::sin(theta[it]) * std::sin(phi[ip]);
            kap[2 * n + a] = std::cos(theta[it]);
        }
    kap.insert(kap.end(), theta, theta + nt);
    kap.insert(kap.end(), phi, phi + np);
    NF_OK(c.kap.alloc(kap.size() * sizeof(double)));
    NF_OK(hipMemcpyAsync(c.kap.p, kap.data(), kap.size() * 8, hipMemcpyHostToDevice, s));
    std::vector<int> order(n), uidx(n);
    std::vector<float> sgn(n);
    std::vector<double> uval;
    for (int x = 0; x < 3; ++x) {
        const double* kx = kap.data() + x * n;
        std::iota(order.begin(), order.end(), 0);
        std::sort(order.begin(), order.end(), [&](int p, int q) {
            const double a = std::fabs(kx[p]), b = std::fabs(kx[q]);
            return a < b || (a == b && p < q);
        });
        uval.clear();
        auto& A = c.ax[x];
        A.start.clear();
        for (size_t i = 0; i < n; ++i) {
            const double v = std::fabs(kx[order[i]]);
            // values within 1e-12 of a group's first one share its row: the
            // phase error k * 1e-12 * |x| is far below float32 resolution
            if (uval.empty() || v - uval.back() > 1e-12) {
                uval.push_back(v);
                A.start.push_back((int)i);
            }
            uidx[order[i]] = (int)uval.size() - 1;
            sgn[order[i]] = kx[order[i]] < 0.0 ? -1.f : 1.f;
        }
        A.start.push_back((int)n);
        A.U = (int)uval.size();
        // groups of up to REDUCE_M angles of one row: the reduction applies
        // every G load of the row to all of a group's angles
        std::vector<int2> groups;
        A.gstart.assign(1, 0);
        for (int u = 0; u < A.U; ++u) {
            for (int i = A.start[u]; i < A.start[u + 1]; i += REDUCE_M)
                groups.push_back(make_int2(i, std::min(REDUCE_M, A.start[u + 1] - i)));
            A.gstart.push_back((int)groups.size());
        }
        NF_OK(A.groups.alloc(groups.size() * sizeof(int2)));
        NF_OK(hipMemcpyAsync(A.groups.p, groups.data(), groups.size() * sizeof(int2), hipMemcpyHostToDevice, s));
        NF_OK(A.uval.alloc(uval.size() * 8));
        NF_OK(A.uidx.alloc(n * 4));
        NF_OK(A.usgn.alloc(n * 4));
        NF_OK(A.order.alloc(n * 4));
        NF_OK(hipMemcpyAsync(A.uval.p, uval.data(), uval.size() * 8, hipMemcpyHostToDevice, s));
        NF_OK(hipMemcpyAsync(A.uidx.p, uidx.data(), n * 4, hipMemcpyHostToDevice, s));
        NF_OK(hipMemcpyAsync(A.usgn.p, sgn.data(), n * 4, hipMemcpyHostToDevice, s));
        NF_OK(hipMemcpyAsync(A.order.p, order.data(), n * 4, hipMemcpyHostToDevice, s));
        A.horder = order;
        NF_OK(hipStreamSynchronize(s));  // host vectors are reused for the next axis
    }
    for (int f = 0; f < 3; ++f) {
        int p, q;
        face_axes(c, f, &p, &q);
        const auto& A = c.ax[p];
        const double* kq = kap.data() + (size_t)q * n;
        std::vector<int> members(n);
        std::vector<int4> groups;
        std::vector<double> gkq;
        auto& M = c.mir[f];
        M.mstart.assign(1, 0);
        for (int u = 0; u < A.U; ++u) {
            const int b = A.start[u], e = A.start[u + 1];
            for (int i = b; i < e; ++i) members[i] = A.horder[i];
            std::sort(members.begin() + b, members.begin() + e, [&](int x, int y) {
                const double a1 = std::fabs(kq[x]), a2 = std::fabs(kq[y]);
                return a1 < a2 || (a1 == a2 && x < y);
            });
            for (int i = b; i < e;) {
                const double v0 = std::fabs(kq[members[i]]);
                int j = i + 1;
                // a bounded number of members (the poles
                // alone would otherwise make one group of every phi)
                while (j < e && j - i < MIRROR_MAX && std::fabs(kq[members[j]]) - v0 <= 1e-12) ++j;
                groups.push_back(make_int4(u, i, j - i, 0));
                gkq.push_back(v0);
                i = j;
            }
            M.mstart.push_back((int)groups.size());
        }
        NF_OK(M.groups.alloc(std::max<size_t>(groups.size(), 1) * sizeof(int4)));
        NF_OK(M.gkq.alloc(std::max<size_t>(gkq.size(), 1) * sizeof(double)));
        NF_OK(M.members.alloc(n * 4));
        NF_OK(hipMemcpyAsync(M.groups.p, groups.data(), groups.size() * sizeof(int4), hipMemcpyHostToDevice, s));
        NF_OK(hipMemcpyAsync(M.gkq.p, gkq.data(), gkq.size() * sizeof(double), hipMemcpyHostToDevice, s));
        NF_OK(hipMemcpyAsync(M.members.p, members.data(), n * 4, hipMemcpyHostToDevice, s));
        NF_OK(hipStreamSynchronize(s));
    }
    c.theta.assign(theta, theta + nt);
    c.phi.assign(phi, phi + np);
    c.n_ang = n;
    return hipSuccess;
}

// Work buffers of at most about OE_NF2FF_MB MB (1024): fewer faces share the
// launches and the buffers of more of them follow one another.
size_t work_limit() {
    const char* v = getenv("OE_NF2FF_MB");
    return (size_t)std::max(0L, v ? atol(v) : 1024L) << 20;
}

// G stays within 64 Mi floats over the faces of a launch; larger U is split
// into chunks of u, each with the angles whose u falls in it.
hipError_t nf2ff_compute(const std::vector<Nf2ffFace>& faces, double freq, const double* theta, int n_theta,
                         const double* phi, int n_phi, double r, const double center[3], hipStream_t s,
                         Nf2ffCache* cache, Nf2ffOut* out) {
    if (faces.empty() || n_theta <= 0 || n_phi <= 0 || !theta || !phi || !out || !cache || !(r > 0) || !(freq > 0))
        return hipErrorInvalidValue;
    const size_t n_ang = (size_t)n_theta * n_phi;
    if (n_ang > (size_t)INT32_MAX / 16) return hipErrorInvalidValue;
    for (const auto& f : faces) {
        const size_t n1 = f.c1.size(), n2 = f.c2.size();
        if (n1 < 1 || n2 < 1 || !f.src || f.axis < 0 || f.axis > 2 || (f.src_kind != 0 && f.src_kind != 1))
            return hipErrorInvalidValue;
        if (n1 * n2 > (size_t)INT32_MAX / 16) return hipErrorInvalidValue;
    }
    NF_OK(plan_angles(*cache, theta, n_theta, phi, n_phi, s));
    Nf2ffCache& C = *cache;
    const double k = 2.0 * M_PI * freq / C0;
    const double* d_kap = C.kap.as<double>();
    // the large contractions on the FP16 matrix cores (operands split in two
    // halves, k_hgemm3) unless OE_NF2FF_SPLIT16=0
    bool split16 = true;
    if (const char* v = getenv("OE_NF2FF_SPLIT16")) split16 = atoi(v) != 0;
    // the second contraction by mirror groups where they hold two or more
    // angles on average, unless OE_NF2FF_MIRROR=0
    bool mirror = true;
    if (const char* v = getenv("OE_NF2FF_MIRROR")) mirror = atoi(v) != 0;

    // faces of small contractions on a side stream beside the large ones unless
    // OE_NF2FF_STREAMS=1
    bool beside = true;
    if (const char* v = getenv("OE_NF2FF_STREAMS")) beside = atoi(v) != 1;

    // per face: first-contraction axis p (fewer distinct |kappa|), sizes
    struct Plan {
        int p, q, np, nq, K, N, swap, need, rows, chunk, n_chunks;  // need: rows of all of U, rows: of one chunk
        std::vector<double> xp, xq;
    };
    const int nf = (int)faces.size();
    std::vector<Plan> plans(nf);
    size_t coord_len = 0, blocks = 0;
    for (int q = 0; q < nf; ++q) {
        const Nf2ffFace& f = faces[q];
        Plan& pl = plans[q];
        const int a1 = (f.axis + 1) % 3, a2 = (f.axis + 2) % 3;
        pl.swap = C.ax[a2].U < C.ax[a1].U;
        pl.p = pl.swap ? a2 : a1;
        pl.q = pl.swap ? a1 : a2;
        const auto& cp = pl.swap ? f.c2 : f.c1;
        const auto& cq = pl.swap ? f.c1 : f.c2;
        pl.np = (int)cp.size();
        pl.nq = (int)cq.size();
        pl.K = (int)round_up(pl.np, KPAD);
        pl.N = (int)round_up(8 * (size_t)pl.nq, GBN);
        for (double v : cp) pl.xp.push_back(v - center[pl.p]);
        for (double v : cq) pl.xq.push_back(v - center[pl.q]);
        coord_len += 2 * ((size_t)pl.np + pl.nq);
        blocks += (cp.size() * cq.size() + 255) / 256;
        pl.need = (int)round_up(2 * (size_t)C.ax[pl.p].U, GBM);
    }
    // Rows of one chunk: the most, the same for every face of a launch, for
    // which G of all of them stays within 256 MB, the size of the cache that
    // the reduction then reads it from.  349x349x221 nodes, us per transform
    // with 256 MB a face / 256 MB together: 54300 irregular angles 3000 / 2884,
    // 22500 1360 / 1313 (128 MB together 2950, 384 MB 2960).
    const size_t budget = (size_t)64 << 20;
    // Sets of up to `per` faces share the launches and, from one set to the
    // next, the buffers: as many as MAX_FACES, fewer where their buffers pass
    // work_limit().
    struct Slot {
        size_t B = 0, A = 0, G = 0, S = 0, b = 0, a = 0, g = 0;
    } slot[MAX_FACES];
    const size_t pblocks = (n_ang + 255) / 256;
    const size_t out_len = 4 * n_ang + pblocks + blocks;  // E_theta, E_phi, block maxima of U, power partials
    int per = MAX_FACES, n_sets = 0;
    std::vector<int> set_chunks;
    size_t face_off = 0, chunk_off = 0, coord_off = 0, up_bytes = 0, out_off = 0, nl_off = 0, pmax_off = 0, bsc_off = 0;
    size_t off = 0;
    // device workspace: the tables (uploaded in one copy), then results,
    // partials and per face slot the operands
    auto lay_out = [&] {
        n_sets = (nf + per - 1) / per;
        for (int s0 = 0; s0 < nf; s0 += per) {
            const int s1 = std::min(nf, s0 + per);
            size_t rows = 0;
            for (int q = s0; q < s1; ++q) rows = std::max(rows, (size_t)plans[q].need);
            auto held = [&](size_t r) {
                size_t g = 0;
                for (int q = s0; q < s1; ++q) g += std::min(r, (size_t)plans[q].need) * plans[q].N;
                return g;
            };
            size_t lo = GBM;  // the most rows within the budget, by halving
            for (size_t hi = rows; lo < hi;) {
                const size_t mid = round_up((lo + hi) / 2, GBM);
                if (held(mid) <= budget) lo = mid;
                else hi = mid - GBM;
            }
            for (int q = s0; q < s1; ++q) {
                plans[q].rows = (int)std::min(lo, (size_t)plans[q].need);
                plans[q].chunk = plans[q].rows / 2;
                plans[q].n_chunks = (C.ax[plans[q].p].U + plans[q].chunk - 1) / plans[q].chunk;
            }
        }
        set_chunks.assign(n_sets, 0);
        for (int q = 0; q < nf; ++q) set_chunks[q / per] = std::max(set_chunks[q / per], plans[q].n_chunks);
        size_t n_table = 0;
        for (int m : set_chunks) n_table += (size_t)m * MAX_FACES;
        chunk_off = round_up(nf * sizeof(FaceDev), 64);
        coord_off = round_up(chunk_off + n_table * sizeof(ChunkDev), 64);
        up_bytes = coord_off + coord_len * sizeof(double);
        out_off = round_up(up_bytes, 256);
        nl_off = round_up(out_off + out_len * sizeof(double), 256);
        pmax_off = nl_off + (n_sets > 1 ? round_up(12 * n_ang * sizeof(double), 256) : 0);
        bsc_off = round_up(pmax_off + blocks * sizeof(float), 256);
        off = round_up(bsc_off + 2 * (size_t)nf * sizeof(float), 256);
        for (Slot& t : slot) t = Slot{};
        for (int q = 0; q < nf; ++q) {
            const Plan& pl = plans[q];
            Slot& t = slot[q % per];
            const size_t M = pl.rows;
            t.b = std::max(t.b, (size_t)pl.K * pl.N);
            t.a = std::max(t.a, M * pl.K);
            t.g = std::max(t.g, M * pl.N);
        }
        for (int q = 0; q < std::min(nf, per); ++q) {
            Slot& t = slot[q];
            t.B = off;  // B, then its split halves [N][K] each
            t.A = round_up(t.B + 2 * t.b * sizeof(float), 256);
            t.G = round_up(t.A + t.a * sizeof(float), 256);
            t.S = round_up(t.G + t.g * sizeof(float), 256);
            off = round_up(t.S + 8 * n_ang * sizeof(double), 256);
        }
    };
    lay_out();
    for (const size_t most = work_limit(); off > most && per > 1;) {
        per = (per + 1) / 2;
        lay_out();
    }
    if (C.work.bytes < off) {
        NF_OK(hipStreamSynchronize(s));
        NF_OK(C.work.alloc(off));
    }
    const size_t host_bytes = std::max(up_bytes, out_len * sizeof(double));
    if (C.host.bytes < host_bytes) NF_OK(C.host.alloc(host_bytes));
    char* wk = C.work.as<char>();
    double* d_out = reinterpret_cast<double*>(wk + out_off);
    double* d_umax = d_out + 4 * n_ang;
    double* d_nl = n_sets > 1 ? reinterpret_cast<double*>(wk + nl_off) : nullptr;

    FaceDev* hf = reinterpret_cast<FaceDev*>(static_cast<char*>(C.host.p) + face_off);
    ChunkDev* hc = reinterpret_cast<ChunkDev*>(static_cast<char*>(C.host.p) + chunk_off);
    double* hx = reinterpret_cast<double*>(static_cast<char*>(C.host.p) + coord_off);
    const double* dx = reinterpret_cast<const double*>(wk + coord_off);
    double flop = 0.0, flop_split = 0.0;
    struct Launch {  // one chunk of one set
        int wg[3] = {0, 0, 0};  // work-groups per KIND_*
        int operands = 0, table = 0;
        int mirror[2] = {0, 0}, plain[2] = {0, 0};  // work-groups of the reductions, [1] of KIND_SPLIT16
    };
    std::vector<std::vector<Launch>> launches(n_sets);
    std::vector<int> pack_blocks(n_sets, 0);
    size_t co = 0, bo = 0, tb = 0;
    for (int set = 0; set < n_sets; ++set) {
        launches[set].resize(set_chunks[set]);
        for (size_t c = 0; c < launches[set].size(); ++c) launches[set][c].table = (int)(tb + c * MAX_FACES);
        std::memset(hc + tb, 0, launches[set].size() * MAX_FACES * sizeof(ChunkDev));
        for (int q = set * per; q < std::min(nf, (set + 1) * per); ++q) {
            const Nf2ffFace& f = faces[q];
            const Plan& pl = plans[q];
            const auto& A = C.ax[pl.p];
            const auto& M = C.mir[f.axis];
            const Slot& t = slot[q % per];
            FaceDev d{};
            d.src = f.src;
            d.scale = f.scale;
            d.kind = f.src_kind;
            d.n1 = (int)f.c1.size();
            d.n2 = (int)f.c2.size();
            d.swap = pl.swap;
            d.sign = f.sign;
            d.np = pl.np; d.nq = pl.nq; d.K = pl.K; d.N = pl.N;
            d.nb = (d.n1 * d.n2 + 255) / 256;
            auto put = [&](const std::vector<double>& v) {
                std::copy(v.begin(), v.end(), hx + co);
                const double* at = dx + co;
                co += v.size();
                return at;
            };
            d.xp = put(pl.xp);
            d.wp = put(trapz_weights(pl.xp));
            d.xq = put(pl.xq);
            d.wq = put(trapz_weights(pl.xq));
            d.B = reinterpret_cast<float*>(wk + t.B);
            d.Bhi = reinterpret_cast<_Float16*>(d.B + t.b);
            d.Blo = d.Bhi + (size_t)pl.N * pl.K;
            d.A = reinterpret_cast<float*>(wk + t.A);
            d.G = reinterpret_cast<float*>(wk + t.G);
            d.S = reinterpret_cast<double*>(wk + t.S);
            d.bsc = reinterpret_cast<float*>(wk + bsc_off) + 2 * q;
            d.part = d_umax + pblocks + bo;
            d.pmax = reinterpret_cast<float*>(wk + pmax_off) + bo;
            bo += d.nb;
            d.uval = A.uval.as<double>();
            d.uni_p = uniform_spacing(pl.xp, &d.dxp);
            d.uni_q = uniform_spacing(pl.xq, &d.dxq);
            d.x0 = f.c0 - center[f.axis];
            d.kapq = d_kap + (size_t)pl.q * n_ang;
            d.kap0 = d_kap + (size_t)f.axis * n_ang;
            d.usgn = A.usgn.as<float>();
            d.uidx = A.uidx.as<int>();
            d.order = A.order.as<int>();
            d.groups = A.groups.as<int2>();
            d.mgroups = M.groups.as<int4>();
            d.gkq = M.gkq.as<double>();
            d.members = M.members.as<int>();
            d.a1 = (f.axis + 1) % 3;
            d.a2 = (f.axis + 2) % 3;
            pack_blocks[set] = std::max(pack_blocks[set], d.nb);
            for (int c = 0; c < pl.n_chunks; ++c) {
                Launch& L = launches[set][c];
                ChunkDev& ck = hc[L.table + q % per];
                ck.u0 = c * pl.chunk;
                ck.u1 = std::min(A.U, ck.u0 + pl.chunk);
                ck.M = (int)round_up(2 * (size_t)(ck.u1 - ck.u0), GBM);
                ck.kind = gemm_kind(ck.M, pl.N, split16);
                ck.first = L.wg[ck.kind];
                const int tile = ck.kind == KIND_FP32 ? 64 : 128;
                L.wg[ck.kind] += (pl.N / tile) * (ck.M / tile);
                if (ck.kind == KIND_SPLIT16) d.split = 1;
                const int nm = M.mstart[ck.u1] - M.mstart[ck.u0];
                // two or more angles per mirror group on average
                ck.mirror = mirror && 2 * (size_t)nm <= (size_t)(A.start[ck.u1] - A.start[ck.u0]);
                const auto& gs = ck.mirror ? M.mstart : A.gstart;
                ck.g0 = gs[ck.u0];
                ck.g1 = gs[ck.u1];
                const int ng = ck.g1 - ck.g0;
                int& wgs = (ck.mirror ? L.mirror : L.plain)[ck.kind == KIND_SPLIT16];
                wgs = std::max(wgs, ck.mirror ? (ng + MIRROR_GROUPS - 1) / MIRROR_GROUPS
                                              : (ng + REDUCE_GROUPS - 1) / REDUCE_GROUPS);
                const size_t work = (size_t)ck.M * pl.K / (ck.kind == KIND_SPLIT16 ? 8 : 1);
                L.operands = std::max(L.operands, (int)std::min<size_t>((work + 255) / 256, 2048));
                const double fl = 2.0 * (2.0 * (ck.u1 - ck.u0)) * (8.0 * pl.nq) * pl.np;  // useful (unpadded) work
                flop += fl;
                if (ck.kind == KIND_SPLIT16) flop_split += fl;
            }
            hf[q] = d;
        }
        // a face past its last chunk: no kind of launch holds it
        for (size_t c = 0; c < launches[set].size(); ++c)
            for (int q = 0; q < MAX_FACES; ++q)
                if (hc[tb + c * MAX_FACES + q].M == 0) hc[tb + c * MAX_FACES + q].kind = -1;
        tb += launches[set].size() * MAX_FACES;
    }
    NF_OK(hipMemcpyAsync(wk, C.host.p, up_bytes, hipMemcpyHostToDevice, s));

    size_t n_ev = 0;
    auto next_events = [&](EventPair** out) -> hipError_t {
        if (n_ev == C.events.size()) {
            std::unique_ptr<EventPair> p(new EventPair());
            NF_OK(hipEventCreate(&p->a));
            NF_OK(hipEventCreate(&p->b));
            C.events.push_back(std::move(p));
        }
        *out = C.events[n_ev++].get();
        return hipSuccess;
    };
    EventPair* all = nullptr;
    NF_OK(next_events(&all));
    std::vector<EventPair*> gemm_ev;
    std::vector<bool> gemm_split;  // launch ran the split FP16 kernel
    NF_OK(hipEventRecord(all->a, s));
    const FaceDev* d_faces = reinterpret_cast<const FaceDev*>(wk + face_off);
    const ChunkDev* d_chunks = reinterpret_cast<const ChunkDev*>(wk + chunk_off);
    for (int set = 0; set < n_sets; ++set) {
        const FaceDev* fd = d_faces + set * per;
        const int n = std::min(per, nf - set * per);
        hipLaunchKernelGGL(k_nf2ff_pack, dim3(pack_blocks[set], n), dim3(256), 0, s, fd);
        bool any_split = false;
        for (int q = 0; q < n; ++q) any_split = any_split || hf[set * per + q].split;
        for (size_t c = 0; c < launches[set].size(); ++c) {
            const Launch& L = launches[set][c];
            const ChunkDev* cd = d_chunks + L.table;
            if (c == 0)
                hipLaunchKernelGGL(k_nf2ff_operands, dim3(L.operands, n, any_split ? 2 : 1), dim3(256), 0, s, fd, cd, k);
            auto gemm = [&](int kind, hipStream_t on) -> hipError_t {
                if (!L.wg[kind]) return hipSuccess;
                EventPair* ev = nullptr;
                NF_OK(next_events(&ev));
                gemm_ev.push_back(ev);
                gemm_split.push_back(kind == KIND_SPLIT16);
                NF_OK(hipEventRecord(ev->a, on));
                const dim3 grid(L.wg[kind]);
                if (kind == KIND_SPLIT16) hipLaunchKernelGGL(k_hgemm3, grid, dim3(256), 0, on, fd, cd, n);
                else if (kind == KIND_FP32) hipLaunchKernelGGL(k_sgemm_mfma<64>, grid, dim3(256), 0, on, fd, cd, n);
                else hipLaunchKernelGGL(k_sgemm_mfma<128>, grid, dim3(256), 0, on, fd, cd, n);
                return hipEventRecord(ev->b, on);
            };
            // the reductions of some kinds; the next chunk's rows go with the
            // first of them when asked for
            auto reduce = [&](int kinds, int mirror, int plain, int rows, hipStream_t on) {
                const ChunkDev* nx = cd + MAX_FACES;
                if (mirror) {
                    hipLaunchKernelGGL(k_nf2ff_reduce_mirror, dim3(std::max(mirror, rows), n, rows ? 2 : 1),
                                       dim3(MIRROR_THREADS), 0, on, fd, cd, nx, kinds, k);
                    rows = 0;
                }
                if (plain)
                    hipLaunchKernelGGL(k_nf2ff_reduce, dim3(std::max(plain, rows), n, rows ? 2 : 1), dim3(REDUCE_THREADS), 0,
                                       on, fd, cd, nx, kinds, k);
            };
            const int rows = c + 1 < launches[set].size() ? launches[set][c + 1].operands : 0;
            const int split = 1 << KIND_SPLIT16, fp32 = 1 << KIND_FP32 | 1 << KIND_FP32_LARGE;
            // The faces of the small contractions go beside the large ones of
            // the others (349x349x221 nodes, us per transform with their rows in
            // launches of their own and one stream / rows with the reductions /
            // and beside: 181x360 regular angles 490 / 490 / 476, 22500
            // irregular ones 1313 / 1314 / 1291, 54300 2884 / 2858 / 2820).
            const bool both = beside && L.wg[KIND_SPLIT16] && (L.wg[KIND_FP32] || L.wg[KIND_FP32_LARGE]);
            if (both) {
                if (!C.side) {
                    NF_OK(hipStreamCreateWithFlags(&C.side, hipStreamNonBlocking));
                    NF_OK(hipEventCreateWithFlags(&C.fork, hipEventDisableTiming));
                    NF_OK(hipEventCreateWithFlags(&C.join, hipEventDisableTiming));
                }
                NF_OK(hipEventRecord(C.fork, s));
                NF_OK(hipStreamWaitEvent(C.side, C.fork, 0));
                NF_OK(gemm(KIND_SPLIT16, s));
                for (int kind : {KIND_FP32_LARGE, KIND_FP32}) NF_OK(gemm(kind, C.side));
                reduce(fp32, L.mirror[0], L.plain[0], 0, C.side);
                NF_OK(hipEventRecord(C.join, C.side));
                NF_OK(hipStreamWaitEvent(s, C.join, 0));
                reduce(split, L.mirror[1], L.plain[1], rows, s);
            } else {
                for (int kind : {KIND_SPLIT16, KIND_FP32_LARGE, KIND_FP32}) NF_OK(gemm(kind, s));
                reduce(split | fp32, std::max(L.mirror[0], L.mirror[1]), std::max(L.plain[0], L.plain[1]), rows, s);
            }
        }
        if (set + 1 < n_sets)
            hipLaunchKernelGGL(k_nf2ff_gather, dim3((unsigned)pblocks), dim3(256), 0, s, fd, n, d_nl, set == 0, n_ang);
        NF_OK(hipGetLastError());
    }
    typedef std::complex<double> cd;
    const cd fac = cd(0.0, k) * std::exp(cd(0.0, -k * r)) / (4.0 * M_PI * r);
    hipLaunchKernelGGL(k_nf2ff_project, dim3((unsigned)pblocks), dim3(256), 0, s, d_faces + (n_sets - 1) * per,
                       nf - (n_sets - 1) * per, d_nl, d_kap + 3 * n_ang, d_kap + 3 * n_ang + n_theta, n_phi, n_ang,
                       fac.real(), fac.imag(), r, d_out, d_umax);
    NF_OK(hipGetLastError());
    NF_OK(hipEventRecord(all->b, s));
    double* h = reinterpret_cast<double*>(C.host.p);
    NF_OK(hipMemcpyAsync(h, d_out, out_len * sizeof(double), hipMemcpyDeviceToHost, s));
    NF_OK(hipStreamSynchronize(s));
    float ms = 0.f;
    NF_OK(hipEventElapsedTime(&ms, all->a, all->b));
    out->total_ms = ms;
    out->gemm_ms = 0.0;
    out->gemm_split_ms = 0.0;
    for (size_t q = 0; q < gemm_ev.size(); ++q) {
        NF_OK(hipEventElapsedTime(&ms, gemm_ev[q]->a, gemm_ev[q]->b));
        out->gemm_ms += ms;
        if (gemm_split[q]) out->gemm_split_ms += ms;
    }
    out->gemm_flop = flop;
    out->gemm_split_flop = flop_split;
    double prad = 0.0;
    for (size_t i = 0; i < blocks; ++i) prad += h[4 * n_ang + pblocks + i];
    out->prad = prad;
    double umax = 0.0;
    for (size_t i = 0; i < pblocks; ++i) umax = std::max(umax, h[4 * n_ang + i]);
    if (out->et) std::memcpy(out->et, h, 2 * n_ang * sizeof(double));
    if (out->ep) std::memcpy(out->ep, h + 2 * n_ang, 2 * n_ang * sizeof(double));
    double* dst[4] = {out->et_re, out->et_im, out->ep_re, out->ep_im};
    for (int q = 0; q < 4; ++q)
        if (dst[q]) {
            const double* src = h + (q / 2) * 2 * n_ang + (q % 2);
            for (size_t a = 0; a < n_ang; ++a) dst[q][a] = src[2 * a];
        }
    out->dmax = prad > 0.0 ? 4.0 * M_PI * umax / prad : 0.0;
    return hipSuccess;
}

}  // namespace oe
