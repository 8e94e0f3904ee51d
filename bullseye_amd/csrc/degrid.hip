// degrid.hip -- the degridding adjoint of the gridding kernels.
//
// bullseye has no degridder in C++ (writing_and_wiki/notebooks/Resampling.ipynb sketches the
// gather in Python).  For the visibility modes this kernel computes the exact transpose, over
// the reals, of the map the gridding kernels apply from visibilities to the unnormalised grids,
// summed over facets.  Per (row, channel) and facet, with the forward's geometry, tap choice,
// edge drop and plane choice:
//   s_k = sum over the footprint of conj(C) * model_k      (C real for the AA kernel)
//   s_k = conj(s_k) if the w-projection sample had w < 0  (the forward conjugated it)
//   s_k *= exp(-i x) (facet phase), s_k *= weight_k (zero when flagged),
//   S = Pinv^H S Qinv in the Jones mode (the forward applies V -> Pinv V Qinv^H),
// and out[row][chan][corr_k] = sum over facets of s_k; every other correlation is zero.
//
// A gather: no atomics.  Three ways to sum a sample's taps; launch_t says which and why.
//   degrid_aa_kernel     AA, W = 3..11: a lane a sample.  The FP64 geometry and rotor (200
//                        instructions) are prepared once, both tap runs sit in registers, the
//                        model is read in rows of W complex values; neighbouring lanes are
//                        neighbouring channels, whose footprints share cache lines.  9
//                        instructions a sample's tap row and correlation, no exchange between
//                        lanes (6 facets x 4 correlations, 1.01 M samples: 1.69 -> 0.38 ms a call
//                        against sixteen lanes a sample).
//   degrid_wave_kernel   w-projection, large calls: a wavefront sums the footprints of its 64
//                        samples one after the other, since a sample's w-kernel block is W_p x
//                        W_p consecutive taps, which lanes of their own samples could only read
//                        line by line.  Eight samples' partial sums are reduced together (each
//                        exchange halves the samples a lane keeps: 10 exchanges for eight, not 6
//                        for each).
//   degrid_group_kernel  everything else: sixteen lanes a sample, every one of which prepares it.
//                        The preparation is repeated, but a call has sixteen times as many
//                        wavefronts in flight and a sample's chain of loads is short.
#include "device_common.h"

namespace bam {
namespace dg {

constexpr int BLOCK = 256;
constexpr int PACK = 8;     // samples reduced together
constexpr int GL = 16;      // lanes a sample of degrid_group_kernel

struct DArgs {
    GridArgs g;                      // inputs and geometry (g.grid and g.norm unused)
    const grid_base_type *model;     // complex [facet][cube][P][ny][nx]
    visibility_base_type *out;       // complex [row][chan][npol]
    const void *taps;                // w-projection taps per (plane, frac_v, frac_u), acc_t
    const uint64_t *plane_off;
    const uint32_t *plane_half;
    uint32_t wplanes, nf, fbase, wproj;
    float wmax_f;
    uint32_t P;                      // correlation slices per (facet, cube) group
    uint64_t rows;
    uint64_t first;                  // first sample of the launch
};

// One sample: what does not depend on the facet.
template <int MODE, int PATH> struct Sample {
    static constexpr int NC = ModeTraits<MODE>::NCORR;
    typedef typename PathTraits<PATH>::acc_t T;
    bool in_range, live;
    uint32_t row, c, s;
    uint64_t cgi;
    size_t base;
    T wt[NC];
    size_t jb1, jb2;
    double u, v, w;

    // the checks are the forward's, in its order
    __device__ __forceinline__ void load(const DArgs &d, uint64_t sample) {
        const GridArgs &a = d.g;
        in_range = sample < d.rows * a.chan;
        row = in_range ? (uint32_t)(sample / a.chan) : 0;
        c = in_range ? (uint32_t)(sample % a.chan) : 0;
        base = ((size_t)row * a.chan + c) * a.npol;
        live = in_range;
        s = 0;
        cgi = 0;
        jb1 = jb2 = 0;
        u = v = w = 0;
#pragma unroll
        for (int k = 0; k < NC; ++k) wt[k] = T(0);
        if (live) {
            s = a.spw[row];
            if (s >= a.spw_count) {
                atomicOr(a.error_flag, 4);
                live = false;
            }
        }
        if (live && !a.enabled[s * a.chan + c]) live = false;
        if (live) {
            cgi = a.cgi[s * a.chan + c];
            if (cgi >= a.cube) {
                atomicOr(a.error_flag, 4);
                live = false;
            }
        }
        if (live && (a.row_flags[row] || a.field[row] != a.imaging_field)) live = false;
        if (live) {
            bool any = false;
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                const size_t idx = base + a.pol_idx[k];
                wt[k] = a.flags[idx] ? T(0) : (T)a.weights[idx];
                any |= wt[k] != T(0);
            }
            live = any;
        }
        if constexpr (MODE == MODE_4J) {
            if (live) {
                const size_t t = a.time_ids[row];
                if (t >= a.ntime || a.ant1[row] >= a.antenna_count ||
                    a.ant2[row] >= a.antenna_count) {
                    atomicOr(a.error_flag, 4);
                    live = false;
                } else {
                    jb1 = ((size_t)t * a.antenna_count + a.ant1[row]) * a.facets;
                    jb2 = ((size_t)t * a.antenna_count + a.ant2[row]) * a.facets;
                }
            }
        }
        if (live) {
            const double rw = 1.0 / (double)a.wavelengths[s * a.chan + c];
            u = (double)a.uvw[3 * (size_t)row] * rw;
            v = (double)a.uvw[3 * (size_t)row + 1] * rw;
            w = (double)a.uvw[3 * (size_t)row + 2] * rw;
        }
    }
};

// Place of a sample on a facet's grid.
template <typename T> struct Place {
    bool on, conj;
    T cs, sn;              // the forward's rotor
    int x0, y0, fu, fv, wp;
    uint32_t tb;
};

template <int MODE, int PATH, bool WPROJ>
__device__ __forceinline__ Place<typename PathTraits<PATH>::acc_t>
place(const DArgs &d, const Sample<MODE, PATH> &sm, uint32_t f) {
    typedef typename PathTraits<PATH>::acc_t T;
    const GridArgs &a = d.g;
    const FacetGeom *gp = a.geom + f;
    Place<T> p = {sm.live, false, T(1), T(0), 0, 0, 0, 0, 0, 0};
    double u = sm.u, v = sm.v, w = sm.w;
    if (p.on && a.phase) {  // the forward's rotor, in turns, FP64 argument
        const double turns = u * gp->dl + v * gp->dm + w * gp->dn;
        const double fr = 2.0 * (turns - rint(turns));
        if constexpr (PATH == PATH_FP64) {
            double s_, c_;
            sincospi(fr, &s_, &c_);
            p.sn = s_;
            p.cs = c_;
        } else {
            float s_, c_;
            sincospi_unit((float)fr, &s_, &c_);
            p.sn = s_;
            p.cs = c_;
        }
    }
    if (a.transform) {
        u = u - w * gp->u_term;
        v = v - w * gp->v_term;
    }
    u *= a.u_scale;
    v *= a.v_scale;
    if constexpr (!WPROJ) {  // AA tap choice under the forward's floor rounding
        const double flu = floor(u), flv = floor(v);
        p.x0 = (int)flu + (int)a.off_x;
        p.y0 = (int)flv + (int)a.off_y;
        p.fu = (int)((1.0 - u + flu) * a.OS);
        p.fv = (int)((1.0 - v + flv) * a.OS);
        p.wp = (int)a.W;
        if (p.x0 < 0 || p.y0 < 0 || p.x0 >= (int)a.nx - p.wp - 2 || p.y0 >= (int)a.ny - p.wp - 2)
            p.on = false;
    } else {  // w-projection: w < 0 conjugation, nearest rounding, plane choice
        if (w < 0) {
            p.conj = true;
            u = -u;
            v = -v;
            w = -w;
        }
        const double ru = rint(u), rv = rint(v);
        const int dx = (int)rint(u + a.off_x), dy = (int)rint(v + a.off_y);
        const int fu = (int)((1.0 - u + ru) * a.OS) - (int)d.fbase;
        const int fv = (int)((1.0 - v + rv) * a.OS) - (int)d.fbase;
        const double pl = rint(w / (double)d.wmax_f * (double)(d.wplanes - 1));
        const int padded = 2 * (int)a.S + 3;
        if (dx < 0 || dy < 0 || dx >= (int)a.nx - padded || dy >= (int)a.ny - padded ||
            pl >= (double)d.wplanes || (uint32_t)fu >= d.nf || (uint32_t)fv >= d.nf)
            p.on = false;
        if (p.on) {
            const int plane = (int)pl;
            const int sp = (int)d.plane_half[plane];
            p.wp = 2 * sp + 1;
            p.x0 = dx + (int)a.S - sp;
            p.y0 = dy + (int)a.S - sp;
            p.tb = (uint32_t)(d.plane_off[plane] +
                              ((uint64_t)fv * d.nf + (uint64_t)fu) * (uint64_t)(p.wp * p.wp));
        }
    }
    return p;
}

// The sample's footprint sums to its visibilities: conjugation, rotor, weights, Jones terms.
template <int MODE, int PATH>
__device__ __forceinline__ void finish(const DArgs &d, const Sample<MODE, PATH> &sm,
                                       const Place<typename PathTraits<PATH>::acc_t> &p, uint32_t f,
                                       cpx<typename PathTraits<PATH>::acc_t> (&sk)[ModeTraits<MODE>::NCORR],
                                       cpx<typename PathTraits<PATH>::acc_t> (&acc)[ModeTraits<MODE>::NCORR]) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    typedef typename PathTraits<PATH>::acc_t T;
    const GridArgs &a = d.g;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        if (p.conj) sk[k] = conjg(sk[k]);
        sk[k] = cmul(sk[k], cpx<T>{p.cs, -p.sn});
        sk[k].re *= sm.wt[k];
        sk[k].im *= sm.wt[k];
    }
    if constexpr (MODE == MODE_4J) {  // S = Pinv^H S Qinv
        const size_t j1 = ((sm.jb1 + f) * a.spw_count + sm.s) * a.chan + sm.c;
        const size_t j2 = ((sm.jb2 + f) * a.spw_count + sm.s) * a.chan + sm.c;
        const cpx<T> *A = reinterpret_cast<const cpx<T> *>(a.jones_inv) + 4 * j1;
        const cpx<T> *B = reinterpret_cast<const cpx<T> *>(a.jones_inv) + 4 * j2;
        const cpx<T> a0 = conjg(A[0]), a1 = conjg(A[1]), a2 = conjg(A[2]), a3 = conjg(A[3]);
        const cpx<T> t0 = cadd(cmul(a0, sk[0]), cmul(a2, sk[2]));
        const cpx<T> t1 = cadd(cmul(a0, sk[1]), cmul(a2, sk[3]));
        const cpx<T> t2 = cadd(cmul(a1, sk[0]), cmul(a3, sk[2]));
        const cpx<T> t3 = cadd(cmul(a1, sk[1]), cmul(a3, sk[3]));
        sk[0] = cadd(cmul(t0, B[0]), cmul(t1, B[2]));
        sk[1] = cadd(cmul(t0, B[1]), cmul(t1, B[3]));
        sk[2] = cadd(cmul(t2, B[0]), cmul(t3, B[2]));
        sk[3] = cadd(cmul(t2, B[1]), cmul(t3, B[3]));
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = cadd(acc[k], sk[k]);
}

template <int MODE, int PATH>
__device__ __forceinline__ void store(const DArgs &d, const Sample<MODE, PATH> &sm,
                                      const cpx<typename PathTraits<PATH>::acc_t> (&acc)[ModeTraits<MODE>::NCORR]) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    typedef typename PathTraits<PATH>::acc_t T;
    if (!sm.in_range) return;
    for (uint32_t cc = 0; cc < d.g.npol; ++cc) {
        cpx<T> val = {T(0), T(0)};
#pragma unroll
        for (int k = 0; k < NC; ++k)
            if (d.g.pol_idx[k] == cc) val = cadd(val, acc[k]);
        d.out[2 * (sm.base + cc)] = (visibility_base_type)val.re;
        d.out[2 * (sm.base + cc) + 1] = (visibility_base_type)val.im;
    }
}

__device__ __forceinline__ const grid_base_type *slice_of(const DArgs &d, uint32_t f, uint64_t cgi) {
    return d.model + ((size_t)f * d.g.cube + cgi) * d.P * ((size_t)d.g.nx * d.g.ny) * 2;
}

// AA, W compile-time: a lane sums its sample's footprint.
template <int MODE, int PATH, int W>
__global__ __launch_bounds__(BLOCK) void degrid_aa_kernel(DArgs d) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    typedef typename PathTraits<PATH>::acc_t T;
    const GridArgs &a = d.g;
    extern __shared__ __align__(16) unsigned char smem[];
    T *conv = reinterpret_cast<T *>(smem);
    for (uint32_t i = threadIdx.x; i < a.csz; i += BLOCK)
        conv[i] = reinterpret_cast<const T *>(a.conv)[i];
    __syncthreads();
    Sample<MODE, PATH> sm;
    sm.load(d, d.first + (uint64_t)blockIdx.x * BLOCK + threadIdx.x);
    const size_t slice = (size_t)a.nx * a.ny;
    cpx<T> acc[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = {T(0), T(0)};
    for (uint32_t f = 0; f < a.facets; ++f) {
        const Place<T> p = place<MODE, PATH, false>(d, sm, f);
        if (!p.on) continue;
        T cu[W];
#pragma unroll
        for (int k = 0; k < W; ++k) cu[k] = conv[p.fu + k * (int)a.OS];
        const grid_base_type *g =
            slice_of(d, f, sm.cgi) + 2 * ((size_t)p.y0 * a.nx + (size_t)p.x0);
        cpx<T> sk[NC];
#pragma unroll
        for (int k = 0; k < NC; ++k) sk[k] = {T(0), T(0)};
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const T cv = conv[p.fv + j * (int)a.OS];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                grid_base_type m[2 * W];   // a row of the footprint, in wide loads
                __builtin_memcpy(m, g + 2 * ((size_t)c * slice + (size_t)j * a.nx), sizeof m);
                cpx<T> t = {T(0), T(0)};
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    t.re = fma(cu[k], (T)m[2 * k], t.re);
                    t.im = fma(cu[k], (T)m[2 * k + 1], t.im);
                }
                sk[c].re = fma(cv, t.re, sk[c].re);
                sk[c].im = fma(cv, t.im, sk[c].im);
            }
        }
        finish(d, sm, p, f, sk, acc);
    }
    store(d, sm, acc);
}

template <typename T> __device__ __forceinline__ T group_sum(T v) {
#pragma unroll
    for (int o = GL / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, GL);
    return v;
}

// Wavefronts a SIMD the group kernel is scheduled for.  FP64 with Jones terms: scheduled for four
// (124 registers) its loads wait for each other, 2.06 M samples of a W <= 15 stack take 4.8 ms
// against 3.6 with three (142 registers).
constexpr int group_waves(int mode, int path) {
    return mode == MODE_4J && path == PATH_FP64 ? 3 : 8;
}

// Any kernel: GL lanes a sample, their partial sums added by a butterfly.
template <int MODE, int PATH, bool WPROJ>
__global__ __launch_bounds__(BLOCK)
__attribute__((amdgpu_waves_per_eu(1, group_waves(MODE, PATH)))) void degrid_group_kernel(DArgs d) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    typedef typename PathTraits<PATH>::acc_t T;
    const GridArgs &a = d.g;
    const int gl = (int)(threadIdx.x % GL);
    Sample<MODE, PATH> sm;
    sm.load(d, d.first + ((uint64_t)blockIdx.x * BLOCK + threadIdx.x) / GL);
    const size_t slice = (size_t)a.nx * a.ny;
    const T *conv = reinterpret_cast<const T *>(a.conv);
    const cpx<T> *wtaps = reinterpret_cast<const cpx<T> *>(d.taps);
    cpx<T> acc[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = {T(0), T(0)};
    for (uint32_t f = 0; f < a.facets; ++f) {
        const Place<T> p = place<MODE, PATH, WPROJ>(d, sm, f);
        cpx<T> sk[NC];
#pragma unroll
        for (int k = 0; k < NC; ++k) sk[k] = {T(0), T(0)};
        if (p.on) {
            const grid_base_type *g =
                slice_of(d, f, sm.cgi) + 2 * ((size_t)p.y0 * a.nx + (size_t)p.x0);
            const int ntap = p.wp * p.wp;
            for (int t = gl; t < ntap; t += GL) {
                const int y = t / p.wp, x = t - y * p.wp;
                cpx<T> tap;
                if constexpr (WPROJ) {
                    tap = conjg(wtaps[p.tb + (uint32_t)t]);
                } else {
                    tap = {conv[p.fu + x * (int)a.OS] * conv[p.fv + y * (int)a.OS], T(0)};
                }
                const grid_base_type *cell = g + 2 * ((size_t)y * a.nx + (size_t)x);
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    const cpx<T> gv = {(T)cell[2 * (size_t)k * slice],
                                       (T)cell[2 * (size_t)k * slice + 1]};
                    sk[k] = cadd(sk[k], cmul(tap, gv));
                }
            }
        }
        // the whole group takes part, samples that are off included
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            sk[k].re = group_sum(sk[k].re);
            sk[k].im = group_sum(sk[k].im);
        }
        if (p.on) finish(d, sm, p, f, sk, acc);
    }
    if (gl == 0) store(d, sm, acc);
}

template <typename T> __device__ __forceinline__ T xor_lane(T v, int mask) {
    return __shfl_xor(v, mask, 64);
}

// W-projection: the wavefront sums the footprints of its 64 samples one after the other.
// What bounds it is the latency of taps and grid cells, so the first 64 taps of GROUP samples are
// loaded together, then the rest of the wide ones AHEAD loads at a time.  One million w-projected
// samples, one correlation: 489 us with sixteen lanes a sample and 639 with one sample's loads at
// a time on a spread observation (1.3e8 taps), 359 with this; on 4 timesteps of 8128 baselines
// 263, 151 and 162 us.
template <int MODE, int PATH>
__global__ __launch_bounds__(BLOCK) void degrid_wave_kernel(DArgs d) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    typedef typename PathTraits<PATH>::acc_t T;
    const GridArgs &a = d.g;
    __shared__ cpx<T> res[BLOCK / 64][64][NC];
    const int lane = threadIdx.x & 63;
    cpx<T>(*mine)[NC] = res[threadIdx.x >> 6];
    Sample<MODE, PATH> sm;
    sm.load(d, d.first + (uint64_t)blockIdx.x * BLOCK + threadIdx.x);
    const size_t slice = (size_t)a.nx * a.ny;
    const cpx<T> *wtaps = reinterpret_cast<const cpx<T> *>(d.taps);
    cpx<T> acc[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = {T(0), T(0)};
    constexpr int WORDS = NC * (int)sizeof(T) / 4;
    constexpr int GROUP = WORDS <= 1 ? 8 : WORDS <= 2 ? 4 : 2, AHEAD = WORDS <= 2 ? 4 : 2;
    // The footprint of the sample of lane r, in scalar registers (one tap of the table and the
    // grid's first cell where the sample does not count).
    struct Footprint {
        uint32_t wp, tb, ntap, inv, cg;
        int x0, y0;
        __device__ __forceinline__ Footprint(const Place<T> &p, uint32_t cgi,
                                             uint32_t lane_inv, int r, uint64_t on) {
            const bool live = (on >> r) & 1;
            wp = live ? (uint32_t)__builtin_amdgcn_readlane(p.wp, r) : 1u;
            tb = live ? (uint32_t)__builtin_amdgcn_readlane((int)p.tb, r) : 0u;
            x0 = live ? __builtin_amdgcn_readlane(p.x0, r) : 0;
            y0 = live ? __builtin_amdgcn_readlane(p.y0, r) : 0;
            cg = live ? (uint32_t)__builtin_amdgcn_readlane((int)cgi, r) : 0u;
            inv = live ? (uint32_t)__builtin_amdgcn_readlane((int)lane_inv, r) : 0u;
            ntap = wp * wp;
        }
    };
    // Tap t of a footprint (conjugated) and the grid values under it.
    auto load_tap = [&](const Footprint &q, uint32_t f, uint32_t t, cpx<T> &tap, cpx<T> (&gv)[NC]) {
        const uint32_t y = (t * q.inv) >> 20, x = t - y * q.wp;
        tap = conjg(wtaps[q.tb + t]);
        const grid_base_type *cell = slice_of(d, f, q.cg) +
                                     2 * ((size_t)q.y0 * a.nx + (size_t)q.x0) +
                                     2 * ((size_t)y * a.nx + x);
#pragma unroll
        for (int k = 0; k < NC; ++k)
            gv[k] = {(T)cell[2 * (size_t)k * slice], (T)cell[2 * (size_t)k * slice + 1]};
    };
    for (uint32_t f = 0; f < a.facets; ++f) {
        const Place<T> p = place<MODE, PATH, true>(d, sm, f);
        const uint64_t on = __ballot(p.on);
        const uint64_t wide = __ballot(p.on && p.wp * p.wp > 64);
        // t / wp as t * (2^20 / wp + 1) >> 20: exact while t times the reciprocal's excess (at most
        // 1) stays below 2^20 / wp, and t < wp^2 <= 63^2 with 63^3 < 2^20
        const uint32_t inv = p.on ? (1u << 20) / (uint32_t)p.wp + 1 : 0u;
        for (int r0 = 0; r0 < 64; r0 += PACK) {
            if (!((on >> r0) & ((1ull << PACK) - 1))) continue;
            cpx<T> part[PACK][NC];
            // a sample's first 64 taps: the loads of GROUP samples leave together
#pragma unroll
            for (int j0 = 0; j0 < PACK; j0 += GROUP) {
                cpx<T> tap[GROUP], gv[GROUP][NC];
                bool mine_too[GROUP];
#pragma unroll
                for (int j = 0; j < GROUP; ++j) {
                    const Footprint q(p, sm.cgi, inv, r0 + j0 + j, on);
                    mine_too[j] = (uint32_t)lane < q.ntap;
                    load_tap(q, f, min((uint32_t)lane, q.ntap - 1), tap[j], gv[j]);
                }
#pragma unroll
                for (int j = 0; j < GROUP; ++j)
#pragma unroll
                    for (int k = 0; k < NC; ++k) {
                        const cpx<T> v = cmac(cpx<T>{T(0), T(0)}, tap[j], gv[j][k]);
                        part[j0 + j][k].re = mine_too[j] ? v.re : T(0);
                        part[j0 + j][k].im = mine_too[j] ? v.im : T(0);
                    }
            }
            // the taps beyond, AHEAD loads in flight while there are that many
#pragma unroll
            for (int j = 0; j < PACK; ++j) {
                if (!((wide >> (r0 + j)) & 1)) continue;
                const Footprint q(p, sm.cgi, inv, r0 + j, on);
                uint32_t t0 = 64;
                for (; t0 + 64 < q.ntap; t0 += 64 * AHEAD) {
                    cpx<T> tap[AHEAD], gv[AHEAD][NC];
#pragma unroll
                    for (int h = 0; h < AHEAD; ++h)
                        load_tap(q, f, min(t0 + 64 * h + (uint32_t)lane, q.ntap - 1), tap[h], gv[h]);
#pragma unroll
                    for (int h = 0; h < AHEAD; ++h)
                        if (t0 + 64 * h + (uint32_t)lane < q.ntap)
#pragma unroll
                            for (int k = 0; k < NC; ++k)
                                part[j][k] = cmac(part[j][k], tap[h], gv[h][k]);
                }
                if (t0 < q.ntap && t0 + (uint32_t)lane < q.ntap) {
                    cpx<T> tap, gv[NC];
                    load_tap(q, f, t0 + (uint32_t)lane, tap, gv);
#pragma unroll
                    for (int k = 0; k < NC; ++k) part[j][k] = cmac(part[j][k], tap, gv[k]);
                }
            }
            // reduce: at each of three steps a lane keeps the half of the samples that its bit
            // names and adds its partner's sums for them; then three plain steps
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                cpx<T> v[PACK];
#pragma unroll
                for (int j = 0; j < PACK; ++j) v[j] = part[j][k];
#pragma unroll
                for (int h = PACK / 2, m = 32; h >= 1; h /= 2, m /= 2) {
                    const bool up = (lane & m) != 0;
#pragma unroll
                    for (int j = 0; j < h; ++j) {
                        const cpx<T> keep = up ? v[j + h] : v[j], give = up ? v[j] : v[j + h];
                        v[j].re = keep.re + xor_lane(give.re, m);
                        v[j].im = keep.im + xor_lane(give.im, m);
                    }
                }
#pragma unroll
                for (int m = 64 / PACK / 2; m >= 1; m /= 2) {
                    v[0].re += xor_lane(v[0].re, m);
                    v[0].im += xor_lane(v[0].im, m);
                }
                if ((lane & (64 / PACK - 1)) == 0) mine[r0 + lane / (64 / PACK)][k] = v[0];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (p.on) {
            cpx<T> sk[NC];
#pragma unroll
            for (int k = 0; k < NC; ++k) sk[k] = mine[lane][k];
            finish(d, sm, p, f, sk, acc);
        }
    }
    store(d, sm, acc);
}

// Which kernel sums the taps.  Measured against sixteen lanes a sample (us a call, 512^2 grids,
// w-kernels of up to 7, 15, 31 and 63 taps a side, samples in thousands):
//   one correlation, FP32:  238: 47/37, 56/66, 99/108, 285/325   499: 101/63, 124/107, 192/168,
//                           431/390; FP64 the wavefronts lead from 238 on (499: 159/86 .. 672/501)
//   two correlations:       126: 32/33 and 238: 57/46 up to 7 a side; above, 499: 146/140, 218/234,
//                           490/621   2064: 559/466, 814/730, 1807/1649
//   four, FP32:             238: 88/84 up to 7; above, 980: 388/373, 571/600, 1239/1550   4128:
//                           1531/1400, 2252/2142, 5324/5273; FP64 never (4128: 2468/2656 ..
//                           14894/15147)
// so wavefronts take the calls that are large enough to fill the GPU with them.  A lane a sample
// (AA) lags only where its few wavefronts leave each with a long chain: 7 thousand samples of four
// correlations 10/12 (W = 7) and 11/18 (W = 11), 15 thousand 12/12 and 15/18, 30 thousand 17/12 and
// 24/19; two correlations 10/12, 13/12 and 18/13 at W = 11.
template <int MODE, int PATH> static uint64_t wave_samples(uint32_t S) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    if (NC == 4 && PATH == PATH_FP64) return ~0ull;
    if (S <= 3) return 1u << 17;   // a footprint in one load
    return NC == 1 ? (PATH == PATH_FP64 ? 1u << 18 : 3u << 17) : NC == 2 ? 1u << 20 : 1u << 21;
}

template <int MODE, int PATH> static hipError_t launch_t(DArgs d, hipStream_t st) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    const uint64_t samples = d.rows * d.g.chan;
    const size_t smem = (size_t)d.g.csz * sizeof(typename PathTraits<PATH>::acc_t);
    const bool wave = d.wproj && samples >= wave_samples<MODE, PATH>(d.g.S);
    const bool lane = !d.wproj && smem <= 32768 && (d.g.W & 1) && d.g.W >= 3 && d.g.W <= 11 &&
                      (NC == 1 || samples >= 5120u * NC);
    // a launch holds fewer than 2^32 work items
    const uint64_t piece = wave || lane ? 1ull << 31 : 1ull << 27;
    const dim3 b(BLOCK);
    for (d.first = 0; d.first < samples; d.first += piece) {
        const uint64_t n = samples - d.first < piece ? samples - d.first : piece;
        const uint64_t lanes = wave || lane ? n : n * GL;
        const dim3 g((uint32_t)((lanes + BLOCK - 1) / BLOCK));
        if (wave) {
            if constexpr (NC != 4 || PATH != PATH_FP64)
                degrid_wave_kernel<MODE, PATH><<<g, b, 0, st>>>(d);
        } else if (lane) {
            switch (d.g.W) {
                case 3: degrid_aa_kernel<MODE, PATH, 3><<<g, b, smem, st>>>(d); break;
                case 5: degrid_aa_kernel<MODE, PATH, 5><<<g, b, smem, st>>>(d); break;
                case 7: degrid_aa_kernel<MODE, PATH, 7><<<g, b, smem, st>>>(d); break;
                case 9: degrid_aa_kernel<MODE, PATH, 9><<<g, b, smem, st>>>(d); break;
                case 11: degrid_aa_kernel<MODE, PATH, 11><<<g, b, smem, st>>>(d); break;
            }
        } else if (d.wproj) {
            degrid_group_kernel<MODE, PATH, true><<<g, b, 0, st>>>(d);
        } else {
            degrid_group_kernel<MODE, PATH, false><<<g, b, 0, st>>>(d);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int MODE> static hipError_t launch_m(const DArgs &d, int path, hipStream_t st) {
    switch (path) {
        case PATH_FP64: return launch_t<MODE, PATH_FP64>(d, st);
        case PATH_F32K: return launch_t<MODE, PATH_F32K>(d, st);
        case PATH_F32: return launch_t<MODE, PATH_F32>(d, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace dg

hipError_t launch_degrid(const GridArgs &a, const void *model, void *out, uint64_t rows,
                         uint32_t P, const void *taps, const uint64_t *plane_off,
                         const uint32_t *plane_half, uint32_t wplanes, uint32_t nf,
                         uint32_t fbase, float wmax_f, int mode, int path, hipStream_t st) {
    dg::DArgs d;
    d.g = a;
    d.model = (const grid_base_type *)model;
    d.out = (visibility_base_type *)out;
    d.taps = taps;
    d.plane_off = plane_off;
    d.plane_half = plane_half;
    d.wplanes = wplanes;
    d.nf = nf;
    d.fbase = fbase;
    d.wproj = wplanes > 1 ? 1u : 0u;
    d.wmax_f = wmax_f;
    d.P = P;
    d.rows = rows;
    switch (mode) {
        case MODE_1: return dg::launch_m<MODE_1>(d, path, st);
        case MODE_2: return dg::launch_m<MODE_2>(d, path, st);
        case MODE_4: return dg::launch_m<MODE_4>(d, path, st);
        case MODE_4J: return dg::launch_m<MODE_4J>(d, path, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace bam
