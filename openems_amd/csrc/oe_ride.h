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

// Work-group wg (256 lanes) of the riders of an H (h) or E launch.
__device__ __forceinline__ void ride(const Ride& r, int wg, bool h) {
    __shared__ double sv[RIDE_SIGNALS];
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
    if (tid < d.n_sig && (d.is_h[tid] != 0) != h) {
        double s = 0.0;
        for (uint64_t k = d.off[tid]; k < d.off[tid + 1]; ++k)
            s += d.w[k] * (double)r.F[(size_t)d.comp[k] * r.g.N + d.cell[k]];
        if (d.series && sample < d.series_cap) d.series[sample * d.n_sig + tid] = s;
        sv[tid] = s;
    }
    __syncthreads();
    const double t = (r.t0 + (double)st + (h ? 1.0 : 0.5)) * r.dt;
    for (int q = tid; q < d.n_f * d.n_sig; q += 256) {
        const int f = q / d.n_sig, m = q - f * d.n_sig;
        if ((d.is_h[m] != 0) == h) continue;
        double c, s;
        dft_phasor(d.freqs[f], t, c, s);
        dft_add(d, (size_t)q, sv[m], c, s);
    }
}
#endif  // __HIPCC__

}  // namespace oe
