// oe_ride.h -- the small per-step work that rides in the Yee launches.
//
// Probes, port DFTs and the captures before an E update (ADE's E^n, Mur's pre
// values) read a few cells each.  As launches of their own they cost 4 to 7
// us apiece, as long as a half-step of a grid of a million cells, for a
// microsecond of work.  None of them writes a field, so they run as extra
// work-groups at the front of a Yee launch that leaves what they read alone:
//
//   H launch of step s    E^(s) is still: E probes and E signals of step
//                         s - 1 (after its sources and post-E hooks), the
//                         ADE and Mur captures for step s, the values of
//                         the sources that the E launch of step s adds
//   E launch of step s    H is still: H probes and H signals of step s
//
// After the batch's last step a launch of the H launch's part alone records
// the last E values.  The step comes from device counters, so the launches
// of a step are the same for every step and replay from a graph: step_a (the
// step under way) is advanced by the first H launch and read by E launches
// only, step_b (steps whose E launch has begun) is advanced by the first E
// launch and read by H launches only.
#pragma once

#include "oe_internal.h"

namespace oe {

#ifdef __HIPCC__
#pragma clang fp contract(off)

// exp(-j 2 pi f t).
__device__ __forceinline__ void dft_phasor(double f, double t, double& c, double& s) {
    const double x = f * t;
    double sn;
    sincospi(2.0 * (x - rint(x)), &sn, &c);
    s = -sn;
}

// One sample's update of the running sums of (frequency, signal) number a.
__device__ __forceinline__ void dft_add(const DftDev& d, size_t a, double s, double cr, double ci) {
    if (d.prec == 0) {
        d.acc64[2 * a] += s * cr;
        d.acc64[2 * a + 1] += s * ci;
    } else {
        const float svf = (float)s;
        float* acc = d.acc32 + 4 * a;
        const float yr = svf * (float)cr - acc[2];
        const float tr = acc[0] + yr;
        acc[2] = (tr - acc[0]) - yr;
        acc[0] = tr;
        const float yi = svf * (float)ci - acc[3];
        const float ti = acc[1] + yi;
        acc[3] = (ti - acc[1]) - yi;
        acc[1] = ti;
    }
}

__device__ __forceinline__ void ade_pre_cell(const float* __restrict__ F, size_t N, const AdeDev& a, int c) {
    const size_t p = a.idx[c];
#pragma unroll
    for (int d = 0; d < 3; ++d) a.Eprev[(size_t)d * a.n + c] = F[(size_t)d * N + p];
}

__device__ __forceinline__ size_t mur_cell(const Grid& g, const MurDev& m, int line, int a, int b) {
    int pos[3];
    pos[m.ny] = line;
    pos[m.nyp] = a;
    pos[m.nypp] = b;
    return ((size_t)pos[0] * g.ny + pos[1]) * g.nz + pos[2];
}

// MurAbc::pre_voltage_update (src/extensions/mur_abc.rs:213-254) of one cell.
__device__ __forceinline__ void mur_pre_cell(const float* __restrict__ F, const Grid& g, const MurDev& m, int q) {
    const int a = q / m.s1, b = q % m.s1;
    const size_t pb = mur_cell(g, m, m.line, a, b), ps = mur_cell(g, m, m.shift, a, b);
    const float* A = F + (size_t)m.nyp * g.N;
    const float* B = F + (size_t)m.nypp * g.N;
    m.v_nyp[q] = A[ps] - m.coeff * A[pb];
    m.v_nypp[q] = B[ps] - m.coeff * B[pb];
}

// Signal m of a DFT: its terms in order, four loaded at a time (one after
// the other, a term costs the 0.35 us of its two dependent loads).
__device__ __forceinline__ double dft_signal(const float* __restrict__ F, size_t N, const DftDev& d, int m) {
    double s = 0.0;
    uint64_t k = d.off[m];
    const uint64_t end = d.off[m + 1];
    for (; k + 4 <= end; k += 4) {
        double w[4];
        float f[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            w[q] = d.w[k + q];
            f[q] = F[(size_t)d.comp[k + q] * N + d.cell[k + q]];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) s += w[q] * (double)f[q];
    }
    for (; k < end; ++k) s += d.w[k] * (double)F[(size_t)d.comp[k] * N + d.cell[k]];
    return s;
}

// Work-group wg (256 lanes) of the riders of an H (h) or E launch.
//
// A DFT's two halves ride in different launches, so what each of them does is
// what its half needs: the half's signals are listed, a phasor is formed once
// for each frequency, and the (frequency, signal) pairs are those of the list.
// What bounds it is latency, and a DFT rides on any grid, so this may not take
// longer than the grid's half-step and a launch of the DFT's own.  us per step
// at 72x60x32, plain, as a launch / riding with a phasor a pair and a term at a
// time / in this form: 64 signals of 4 terms at 64 frequencies 18.9 / 30.1 /
// 13.7, 64 of 32 terms at 10 frequencies 35.2 / 42.9 / 18.6, voltage and
// current of 4 terms at 64 frequencies 14.4 / 10.4 / 8.5.
__device__ __forceinline__ void ride(const Ride& r, int wg, bool h) {
    constexpr int FC = 256;  // frequencies at a time
    __shared__ double sv[RIDE_SIGNALS];     // the half's signals
    __shared__ int sig[RIDE_SIGNALS];       // and their numbers
    __shared__ double ph[FC][2];
    __shared__ int n_half;
    const int tid = threadIdx.x;
    if (wg >= r.first_ade) {  // H launches only
        if (wg >= r.first_mur) {
            int f = 0;
            while (f + 1 < r.n_mur && wg >= r.mur[f + 1].first) ++f;
            const MurDev m = *r.mur[f].face;
            const int q = (wg - r.mur[f].first) * 256 + tid;
            if (q < m.s0 * m.s1) mur_pre_cell(r.F, r.g, m, q);
        } else {
            int x = 0;
            while (x + 1 < r.n_ade && wg >= r.ade_first[x + 1]) ++x;
            const int c = (wg - r.ade_first[x]) * 256 + tid;
            if (c < r.ade[x].n) ade_pre_cell(r.F, r.g.N, r.ade[x], c);
        }
        return;
    }
    uint64_t st;
    if (h) {
        const uint64_t b = *r.step_b;
        if (wg == 0 && r.first_dft > 0 && tid < r.n_src) {
            const PointExc& x = r.src[tid];
            SourceValue v{0.f, 0};
            const uint32_t code = 1u | (x.soft ? 2u : 0u) | (x.comp << 2);
            if (b < x.n_samples) v = SourceValue{x.samples[b], code};
            else if (x.zero_after) v.code = code;
            r.src_val[tid] = v;
        }
        if (b == 0) return;  // the batch's first step has no step before it
        st = b - 1;
    } else {
        st = *r.step_a;
    }
    if (wg < r.first_dft) {
        for (int q = tid; q < r.n_probe; q += 256) {
            const PointProbe p = r.probe[q];
            const uint64_t c = p.count0 + st;
            if (c < p.capacity) {
                double* o = p.out + 6 * c + (h ? 0 : 3);
                const float* f = r.F + (h ? 0 : 3 * r.g.N) + p.idx;
#pragma unroll
                for (int d = 0; d < 3; ++d) o[d] = (double)f[(size_t)d * r.g.N];
            }
            if (h) *p.count = c + 1;
        }
        return;
    }
    const RideDft& x = r.dft[wg - r.first_dft];
    const DftDev& d = x.d;
    const uint64_t sample = x.sample0 + st;
    if (tid < 64) {  // RIDE_SIGNALS lanes, one wave
        const bool mine = tid < d.n_sig && (d.is_h[tid] != 0) != h;
        const unsigned long long all = __ballot(mine);
        if (tid == 0) n_half = __popcll(all);
        if (mine) {
            const int at = __popcll(all & ((1ull << tid) - 1));
            const double s = dft_signal(r.F, r.g.N, d, tid);
            if (d.series && sample < d.series_cap) d.series[sample * d.n_sig + tid] = s;
            sv[at] = s;
            sig[at] = tid;
        }
    }
    const double t = (r.t0 + (double)st + (h ? 1.0 : 0.5)) * r.dt;
    for (int f0 = 0; f0 < d.n_f; f0 += FC) {
        const int nf = min(FC, d.n_f - f0);
        if (f0) __syncthreads();  // the phasors before are read
        const int p = nf <= 128 ? tid - 128 : tid;  // waves that have no signals, where they hold all
        if (p >= 0 && p < nf) dft_phasor(d.freqs[f0 + p], t, ph[p][0], ph[p][1]);
        __syncthreads();
        const int n = n_half;
        for (int q = tid; q < nf * n; q += 256) {
            const int f = q / n, g = q - f * n;
            dft_add(d, (size_t)(f0 + f) * d.n_sig + sig[g], sv[g], ph[f][0], ph[f][1]);
        }
    }
}
#endif  // __HIPCC__

}  // namespace oe
