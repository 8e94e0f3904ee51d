// wtile.hip -- w-projection gridding through on-chip tiles of the uv-grid.
//
// Semantics: those of wproj.hip (cpu_algorithm/convolution_policies.h:231-289).  The samples of
// a call are binned by (plane width, grid slice, tile of TILE x TILE footprint origins); a
// workgroup then takes the samples of one bin, adds their taps into an FP64 image of the tile
// (plus the W - 1 halo cells of the footprints) in LDS and adds the tile to the grid once.
//
// Why: the class kernels of wproj.hip keep the footprint in registers and flush cells as it
// moves, 0.05 grid atomics per tap, and this GPU's FP64 atomics run at 23.7 G requests/s on the
// memory side whatever they carry.  Here a tile of 4096 samples of 49 taps costs about 400
// requests (0.002 per tap), the adds are LDS atomics (ds_add_f64: 8.7 cycles per wavefront on
// consecutive doubles, 4.5 T adds/s over the chip), and no lane owns or moves anything.
// Measured: 125 M samples on 4096^2 (supports 7..63) 41 -> 11.2 ms a call, of which the LDS adds
// take 6.2 ms and the two preparing passes 2.9 ms; 0.4 M samples into two facets 1.64 -> 0.50 ms.
//
//   k_count    bin of every sample, counted (one atomic per bin and wavefront)
//   scan       first record of every bin
//   k_scatter  the sample's weighted, rotated visibility and first tap, written to its bin;
//              normalisation sums and counters
//   k_items    bins cut into work items of at most `chunk` records, listed per width
//   wtile_kernel  persistent, one launch per list of widths: LDS tile per item
//
// The bank layout fixes TILE: with rows of W + 32 cells the taps t = row * W + column of a
// footprint fall on the doubles t + 32 * row, so the 64 lanes of an instruction touch 64
// consecutive banks pairs modulo the LDS width whatever the row breaks (7-wide rows 48 doubles
// apart: 24 cycles per instruction against 8.7).
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "wtile.h"

namespace bam {
namespace wt {

constexpr int BLOCK = 256;

// Position of one sample on its facet's grid.
struct Spot {
    int x0, y0;        // first cell of the W_p x W_p footprint
    int plane, half;   // w-plane and its half support
    uint32_t q;        // (frac_v, frac_u) block of the plane
    bool neg;          // w < 0: the visibility is conjugated
};

// rint(ww / wmax * (planes - 1)), operation by operation.  The quotient is first taken by the
// reciprocal (a few ulp off); the division, 12 instructions, runs only where those could change
// the rounding.
__device__ __forceinline__ double plane_of(double ww, const wp::WArgs &w) {
#pragma clang fp contract(off)
    const double n = (double)(w.wplanes - 1);
    const double x = ww * w.inv_wmax * n;
    double pl = rint(x);
    if (!(fabs(x - pl) < 0.499999)) pl = rint(ww / (double)w.wmax_f * n);
    return pl;
}

// The rounding of every operation is fixed here (no contraction), so that k_count and k_scatter
// agree on every sample's bin.
__device__ __forceinline__ bool locate(const wp::WArgs &w, const FacetGeom *gp, double u, double v,
                                       double ww, Spot &s) {
#pragma clang fp contract(off)
    const GridArgs &a = w.g;
    if (a.transform) {
        u = fma(-ww, gp->u_term, u);
        v = fma(-ww, gp->v_term, v);
    }
    u *= a.u_scale;
    v *= a.v_scale;
    s.neg = ww < 0;
    if (s.neg) {   // convolution_policies.h:248-253
        u = -u;
        v = -v;
        ww = -ww;
    }
    const double ru = rint(u), rv = rint(v);
    const int dx = (int)rint(u + a.off_x), dy = (int)rint(v + a.off_y);
    const int fu = (int)((1.0 - u + ru) * a.OS);
    const int fv = (int)((1.0 - v + rv) * a.OS);
    const double pl = plane_of(ww, w);
    const int padded = 2 * (int)a.S + 3;
    if (dx < 0 || dy < 0 || dx >= (int)a.nx - padded || dy >= (int)a.ny - padded ||
        pl >= (double)w.wplanes)
        return false;
    const uint32_t ru_ = (uint32_t)(fu - (int)w.fbase), rv_ = (uint32_t)(fv - (int)w.fbase);
    if (ru_ >= w.nf || rv_ >= w.nf) return false;   // only a coordinate that is not a number
    s.plane = (int)pl;
    s.half = (int)w.plane_half[s.plane];
    s.x0 = dx + (int)a.S - s.half;
    s.y0 = dy + (int)a.S - s.half;
    s.q = rv_ * w.nf + ru_;
    return true;
}

// What one (sorted row, channel) of a facet reads before it is known to count.  All of it is in
// range whatever the checks find, so the loads of a step leave together.
template <int MODE, bool VIS> struct Input {
    static constexpr int NC = MODE == MODE_PSF ? 0 : ModeTraits<MODE>::NCORR;
    ChanRec ch;
    visibility_weights_base_type wt[NC ? NC : 1];
    uint8_t fl[NC ? NC : 1];
    visibility_base_type vis[VIS && NC ? 2 * NC : 1];
    __device__ __forceinline__ void load(const GridArgs &a, const RowRec &rr, uint32_t c) {
        if (rr.spw < a.spw_count) ch = a.chanrec[rr.spw * a.chan + c];
        const size_t base = ((size_t)rr.row * a.chan + c) * a.npol;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const size_t idx = base + a.pol_idx[k];
            wt[k] = a.weights[idx];
            fl[k] = a.flags[idx];
            if constexpr (VIS) {
                vis[2 * k] = a.vis[2 * idx];
                vis[2 * k + 1] = a.vis[2 * idx + 1];
            }
        }
    }
};

// One (sorted row, channel) of a facet: the checks of the class kernels in their order, the
// weights, and the position.  Errors are raised only in the scattering pass.  The arrays shared by
// the facets come from the launch's arguments (t.w.g), the facet's own from w.
template <int MODE, bool RAISE, bool BATCH>
__device__ __forceinline__ bool find(const TArgs &t, const wp::WArgs &w, const FacetGeom *gp,
                                     uint32_t ri, const RowRec &rr,
                                     const Input<MODE, RAISE> &in, uint32_t c,
                                     uint32_t &cgi, double &u, double &v, double &ww, Spot &s) {
    const GridArgs &a = t.w.g;
    if (rr.spw >= a.spw_count) {
        if (RAISE) atomicOr(a.error_flag, 4);
        return false;
    }
    const ChanRec &ch = in.ch;
    if (!ch.enabled) return false;
    if (ch.cgi >= w.g.cube) {
        if (RAISE) atomicOr(a.error_flag, 4);
        return false;
    }
    cgi = ch.cgi;
    if (!(rr.state & ROW_USABLE)) return false;
    if constexpr (MODE == MODE_4J) {
        if (rr.state & ROW_BAD_IDS) {
            if (RAISE) atomicOr(a.error_flag, 4);
            return false;
        }
    }
    u = rr.u * ch.rw;
    v = rr.v * ch.rw;
    ww = rr.w * ch.rw;
    if constexpr (MODE != MODE_PSF) {
        bool any = false;
#pragma unroll
        for (int k = 0; k < ModeTraits<MODE>::NCORR; ++k) any |= !in.fl[k] && in.wt[k] != 0;
        if (!any) return false;
    }
    if (!locate(w, gp, u, v, ww, s)) return false;
    if constexpr (BATCH) {
        // a plan is of the data it was made from: a sample wider than the class its stream had
        // then is dropped and reported, as the class kernels do
        const uint32_t seg = (ri - a.bl_start[rr.bl]) / w.base_rows;
        const uint64_t entry =
            ((uint64_t)rr.bl * a.n_chan_blocks + c / a.chan_per_stream) * w.nseg_base + seg;
        if (2 * s.half + 1 > (int)w.seg_cls[entry]) {
            if (RAISE) atomicOr(a.error_flag, 8);
            return false;
        }
    }
    return true;
}

// Bin of a located sample of the pass's facet f: widths, then slices of the facets, then tiles.
__device__ __forceinline__ uint32_t bin_of(const TArgs &t, const wp::WArgs &w, uint32_t f,
                                           uint32_t cgi, const Spot &s) {
    const uint32_t tx = (uint32_t)s.x0 / TILE, ty = (uint32_t)s.y0 / TILE;
    const uint32_t nx = tiles_of(w.g.nx), ny = tiles_of(w.g.ny);
    const uint32_t spot = (t.spot_base ? t.spot_base[f] : f * w.g.cube * nx * ny) +
                          (cgi * ny + ty) * nx + tx;
    return (uint32_t)(s.half - (int)t.half_lo) * t.nspots + spot;
}

// Lanes of the wavefront that share this lane's bin (0 for lanes without a sample).
__device__ __forceinline__ uint64_t same_bin(bool live, uint32_t bin) {
    uint64_t mine = 0;
    uint64_t pend = __ballot(live);
    while (pend) {
        const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)bin, __ffsll((unsigned long long)pend) - 1);
        const uint64_t m = __ballot(live && bin == b0);
        if (live && bin == b0) mine = m;
        pend &= ~m;
    }
    return mine;
}

__device__ __forceinline__ uint32_t lane_rank(uint64_t m) {   // set bits of m below this lane
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Samples of the wavefront's next step: consecutive (row, channel) pairs over consecutive lanes,
// so the samples of a wavefront lie on one or two tracks and share a few bins.
struct Walk {
    uint32_t row, chan, drow, dchan, chans;
    uint32_t at;   // index of the sample in the pass
    __device__ __forceinline__ Walk(uint32_t first, uint32_t row0, uint32_t C, uint32_t base) {
        chans = C;
        row = first / C;
        chan = first - row * C;
        row += row0;
        drow = 64 / C;
        dchan = 64 - drow * C;
        at = base + first;
    }
    __device__ __forceinline__ void next() {
        row += drow;
        chan += dchan;
        if (chan >= chans) {
            chan -= chans;
            ++row;
        }
        at += 64;
    }
};

// Places in the bins are reserved by k_count: per step one atomic per bin of the wavefront, or,
// while all its samples stay in one bin, one for the whole run of steps.  (Atomics on one
// address run at about 0.5 us each here, and the bins of the short baselines hold tracks that
// never leave them: without the runs k_count took 2.5 ms on 125 M samples.)  The
// reservation's first place is left at the sample that opened it, where k_scatter, which
// walks alike, finds it.
constexpr uint32_t NO_BIN = 0xffffffffu;

// The row record of the next step, loaded while this one is worked on.  What bounds both passes
// is the chain of loads of a step (row, then channel, weights and visibility, then the plane's
// table, then the place): with this, the loads of Input together and a run's places kept, 125 M
// samples are counted in 0.97 ms and scattered in 1.95 ms (1.19 and 2.39 one load after another).
__device__ __forceinline__ void ahead(const TArgs &t, Walk k, RowRec &rn) {
    k.next();
    if (k.row < t.row1) rn = load_row_record(t.w.g.rowrec + k.row);
}

template <int MODE, bool BATCH> __global__ __launch_bounds__(BLOCK) void k_count(TArgs t) {
    const uint32_t f = BATCH ? t.facet_list[blockIdx.y] : t.f0 + blockIdx.y;
    const wp::WArgs &w = BATCH ? t.w.facet_args[f] : t.w;
    const FacetGeom *gp = w.g.geom + (BATCH ? 0 : f);
    const uint32_t lane = threadIdx.x & 63, copy = blockIdx.x % t.copies;
    const uint32_t wave = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    uint32_t run = NO_BIN, run_n = 0, run_at = 0;
    Walk k(wave * 64 * t.iters + lane, t.row0, t.w.g.chan,
           blockIdx.y * (t.row1 - t.row0) * t.w.g.chan);
    RowRec rn;
    if (k.row < t.row1) rn = load_row_record(t.w.g.rowrec + k.row);
    for (uint32_t it = 0; it < t.iters; ++it, k.next()) {
        const RowRec rr = rn;
        const bool in_pass = k.row < t.row1;
        Input<MODE, false> in;
        if (in_pass) in.load(t.w.g, rr, k.chan);
        ahead(t, k, rn);
        uint32_t cgi, bin = 0;
        double u, v, ww;
        Spot s;
        const bool live =
            in_pass && find<MODE, false, BATCH>(t, w, gp, k.row, rr, in, k.chan, cgi, u, v, ww,
                                                     s);
        if (live) bin = bin_of(t, w, blockIdx.y, cgi, s);
        const uint64_t any = __ballot(live);
        if (!any) continue;
        const int lead = __ffsll((unsigned long long)any) - 1;
        const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)bin, lead);
        const bool one = __ballot(live && bin == b0) == any;
        if (one && b0 == run) {
            run_n += (uint32_t)__popcll(any);
            continue;
        }
        if (run != NO_BIN && lane == 0)
            t.first[run_at] = atomicAdd(t.count + (size_t)run * t.copies + copy, run_n);
        run = NO_BIN;
        if (one) {
            run = b0;
            run_n = (uint32_t)__popcll(any);
            run_at = (uint32_t)__builtin_amdgcn_readlane((int)k.at, lead);
        } else {
            const uint64_t m = same_bin(live, bin);
            if (m && lane_rank(m) == 0)
                t.first[k.at] = atomicAdd(t.count + (size_t)bin * t.copies + copy,
                                          (uint32_t)__popcll(m));
        }
    }
    if (run != NO_BIN && lane == 0)
        t.first[run_at] = atomicAdd(t.count + (size_t)run * t.copies + copy, run_n);
}

template <int MODE, typename T, bool BATCH>
__global__ __launch_bounds__(BLOCK) void k_scatter(TArgs t) {
    constexpr int NC = ModeTraits<MODE>::NCORR;
    const uint32_t f = BATCH ? t.facet_list[blockIdx.y] : t.f0 + blockIdx.y;
    const wp::WArgs &w = BATCH ? t.w.facet_args[f] : t.w;
    const FacetGeom *gp = w.g.geom + (BATCH ? 0 : f);
    const GridArgs &a = t.w.g;
    const bool phase = w.g.phase != 0;
    const uint32_t lane = threadIdx.x & 63, copy = blockIdx.x % t.copies;
    const uint32_t wave = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    struct __align__(sizeof(T) == 4 && NC == 1 ? 16 : 8) Rec {
        Head h;
        cpx<T> vis[NC];
    };
    static_assert(sizeof(Rec) == sizeof(Head) + NC * sizeof(cpx<T>), "packed records");
    Rec *recs = reinterpret_cast<Rec *>(t.recs);
    int ncgi = -1;
    double nacc[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) nacc[k] = 0;
    unsigned long long cnt = 0, taps = 0;
    const int kbase = (int)(f * t.w.g.cube);   // normalisation key: slice of the facet
    uint32_t run = NO_BIN, run_next = 0, run_end = 0;   // the run's next place, its bin's end
    Walk k(wave * 64 * t.iters + lane, t.row0, a.chan, blockIdx.y * (t.row1 - t.row0) * a.chan);
    RowRec rn;
    if (k.row < t.row1) rn = load_row_record(a.rowrec + k.row);
    for (uint32_t it = 0; it < t.iters; ++it, k.next()) {
        const RowRec rr = rn;
        const bool in_pass = k.row < t.row1;
        Input<MODE, true> in;
        if (in_pass) in.load(a, rr, k.chan);
        ahead(t, k, rn);
        uint32_t cgi = 0, bin = 0;
        double u = 0, v = 0, ww = 0;
        Spot s;
        const bool live =
            in_pass && find<MODE, true, BATCH>(t, w, gp, k.row, rr, in, k.chan, cgi, u, v, ww,
                                                     s);
        cpx<T> vis[NC];
        if (live) {
            bin = bin_of(t, w, blockIdx.y, cgi, s);
            T wt[NC];
            if constexpr (MODE == MODE_PSF) {
                vis[0] = {T(1), T(0)};
                wt[0] = T(1);
            } else {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    vis[c] = {(T)in.vis[2 * c], (T)in.vis[2 * c + 1]};
                    wt[c] = in.fl[c] ? T(0) : (T)in.wt[c];
                }
            }
            if constexpr (MODE == MODE_4J) {
                const uint64_t jf = ((uint64_t)f * a.spw_count + rr.spw) * a.chan + k.chan;
                const cpx<T> *P = reinterpret_cast<const cpx<T> *>(a.jones_inv) + 4 * (rr.j1 + jf);
                const cpx<T> *Q = reinterpret_cast<const cpx<T> *>(a.jones_inv) + 4 * (rr.j2 + jf);
                const cpx<T> t0 = cmac_conj(cmul_conj(vis[0], Q[0]), vis[1], Q[1]);
                const cpx<T> t1 = cmac_conj(cmul_conj(vis[0], Q[2]), vis[1], Q[3]);
                const cpx<T> t2 = cmac_conj(cmul_conj(vis[2], Q[0]), vis[3], Q[1]);
                const cpx<T> t3 = cmac_conj(cmul_conj(vis[2], Q[2]), vis[3], Q[3]);
                vis[0] = cmac(cmul(P[0], t0), P[1], t2);
                vis[1] = cmac(cmul(P[0], t1), P[1], t3);
                vis[2] = cmac(cmul(P[2], t0), P[3], t2);
                vis[3] = cmac(cmul(P[2], t1), P[3], t3);
            }
            T sn = T(0), cs = T(1);
            if (phase) {   // phase_transform_policies.h:138-146, argument in turns, FP64
                const double turns = u * gp->dl + v * gp->dm + ww * gp->dn;
                const double fr = 2.0 * (turns - rint(turns));
                if constexpr (sizeof(T) == 8) {
                    sincospi(fr, &sn, &cs);
                } else {
                    sincospi_unit((float)fr, &sn, &cs);
                }
            }
            const double ts = w.plane_norm[(size_t)s.plane * w.nf * w.nf + s.q];
            if constexpr (MODE != MODE_PSF) {
                if ((int)cgi != ncgi) {
                    if (ncgi >= 0) flush_norm_lane<NC>(t.w.g, kbase + ncgi, nacc);
                    ncgi = (int)cgi;
                }
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                vis[c].re *= wt[c];
                vis[c].im *= wt[c];
                if (phase) vis[c] = cmul(vis[c], cpx<T>{cs, sn});
                if (s.neg) vis[c].im = -vis[c].im;
                nacc[c] += (double)wt[c] * ts;
            }
            ++cnt;
            taps += (unsigned long long)((2 * s.half + 1) * (2 * s.half + 1));
        }
        const uint64_t any = __ballot(live);
        if (!any) continue;
        const int lead = __ffsll((unsigned long long)any) - 1;
        const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)bin, lead);
        const bool one = __ballot(live && bin == b0) == any;
        uint32_t at, end;
        if (one) {
            if (b0 != run) {
                const uint32_t from = (uint32_t)__builtin_amdgcn_readlane((int)k.at, lead);
                const size_t slot = (size_t)b0 * t.copies + copy;
                run_next = t.start[slot] + t.first[from];
                run_end = t.start[slot + 1];
            }
            at = run_next + lane_rank(any);
            end = run_end;
            run_next += (uint32_t)__popcll(any);
        } else {
            const uint64_t m = same_bin(live, bin);
            uint32_t first = 0;
            if (live && lane_rank(m) == 0) first = t.first[k.at];
            first = __shfl(first, m ? __ffsll((unsigned long long)m) - 1 : 0, 64);
            const size_t slot = (size_t)bin * t.copies + copy;
            if (live) {
                at = t.start[slot] + first + lane_rank(m);
                end = t.start[slot + 1];
            }
        }
        run = one ? b0 : NO_BIN;
        if (live) {
            // both passes locate a sample alike, so it lies inside what k_count reserved
            if (at < end) {
                const uint32_t wp_ = (uint32_t)(2 * s.half + 1);
                Rec r;
                r.h.tap = (uint32_t)(w.plane_off[s.plane] + (uint64_t)s.q * (wp_ * wp_));
                r.h.cell = (uint32_t)(s.y0 % TILE) * (wp_ + TILE - 1) + (uint32_t)(s.x0 % TILE);
#pragma unroll
                for (int c = 0; c < NC; ++c) r.vis[c] = vis[c];
                recs[at] = r;
            }
        }
    }
    if constexpr (MODE != MODE_PSF) publish_norm<NC>(t.w.g, ncgi >= 0 ? kbase + ncgi : -1, nacc);
    publish_counts(t.w.g, cnt, taps);
}

// Widths are listed apart up to 11 and together above, where items are few: 13-15, then four
// widths a list (an empty launch costs as much as a small one).
constexpr int NLIST = 13;
__host__ __device__ constexpr uint32_t list_of(uint32_t half) {
    return half < 6 ? half : half < 8 ? 6 : 7 + (half - 8) / 4;
}
__host__ __device__ constexpr uint32_t list_first(uint32_t list) {   // its narrowest half support
    return list < 7 ? list : 8 + (list - 7) * 4;
}
// Widths of the call that a list holds, and the start of its items.
__host__ __device__ __forceinline__ uint32_t list_widths(const TArgs &t, uint32_t list) {
    const uint32_t a = list_first(list) > t.half_lo ? list_first(list) : t.half_lo;
    const uint32_t e = list_first(list + 1), hi = t.half_lo + t.ncls;
    const uint32_t b = e < hi ? e : hi;
    return b > a ? b - a : 0;
}
__host__ __device__ __forceinline__ size_t list_base(const TArgs &t, uint32_t list) {
    const uint32_t a = list_first(list);
    return a > t.half_lo ? (size_t)(a - t.half_lo) * t.item_cap : 0;
}

// Work items: every bin in pieces of at most t.chunk records, listed per width.
__global__ __launch_bounds__(BLOCK) void k_items(TArgs t) {
    const uint32_t spot = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t cls = blockIdx.y, half = t.half_lo + cls;
    const uint32_t list = list_of(half);
    uint32_t n = 0, first = 0, count = 0;
    if (spot < t.nspots) {
        const size_t slot = ((size_t)cls * t.nspots + spot) * t.copies;
        first = t.start[slot];
        count = t.start[slot + t.copies] - first;
        n = (count + t.chunk - 1) / t.chunk;
    }
    // one reservation per wavefront
    const uint32_t lane = threadIdx.x & 63;
    uint32_t sum = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t up = __shfl_up(sum, o, 64);
        if ((int)lane >= o) sum += up;
    }
    uint32_t at = 0;
    if (lane == 63 && sum) at = atomicAdd(t.item_count + list, sum);
    at = __shfl(at, 63, 64) + sum - n;
    uint32_t f = 0, in = spot;
    if (t.spot_base && n) {   // the facet whose spots hold this one
        uint32_t hi = t.nfacets;
        while (hi - f > 1) {
            const uint32_t mid = (f + hi) / 2;
            if (t.spot_base[mid] <= spot)
                f = mid;
            else
                hi = mid;
        }
        in -= t.spot_base[f];
    }
    const wp::WArgs &w = t.spot_base ? t.w.facet_args[t.facet_list[f]] : t.w;
    const uint32_t nx = tiles_of(w.g.nx), ny = tiles_of(w.g.ny);
    if (!t.spot_base) {
        f = in / (w.g.cube * nx * ny);
        in -= f * w.g.cube * nx * ny;
    }
    Item it;
    it.facet = t.spot_base ? t.facet_list[f] : t.f0 + f;
    it.slice = in / (nx * ny);
    in -= it.slice * nx * ny;
    it.ty = (uint16_t)(in / nx);
    it.tx = (uint16_t)(in % nx);
    Item *out = t.items + list_base(t, list);
    const uint32_t cap = t.item_cap * list_widths(t, list);
    it.half = half;
    it.first = first;
    it.count = min(t.chunk, count);
    if (n && at < cap) out[at] = it;
    // the further pieces of a long bin are listed by the whole wavefront
    for (uint64_t more = __ballot(n > 1); more; more &= more - 1) {
        const int l = __ffsll((unsigned long long)more) - 1;
        const uint32_t ln = __shfl(n, l, 64), lat = __shfl(at, l, 64);
        const uint32_t lfirst = __shfl(first, l, 64), lcount = __shfl(count, l, 64);
        Item li;
        li.half = half;
        li.facet = __shfl(it.facet, l, 64);
        li.slice = __shfl(it.slice, l, 64);
        li.tx = (uint16_t)__shfl((uint32_t)it.tx, l, 64);
        li.ty = (uint16_t)__shfl((uint32_t)it.ty, l, 64);
        for (uint32_t j = 1 + lane; j < ln; j += 64) {
            li.first = lfirst + j * t.chunk;
            li.count = min(t.chunk, lcount - j * t.chunk);
            if (lat + j < cap) out[lat + j] = li;
        }
    }
}

template <typename T> __device__ __forceinline__ T lane_value(T v, int l);
template <> __device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
template <> __device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Taps in the global address space: a batch's pointers come from memory, and loads whose address
// space the compiler cannot see wait for the LDS adds in flight as well.
template <typename T> struct Taps {
    typedef T v2 __attribute__((ext_vector_type(2)));
    typedef const v2 __attribute__((address_space(1))) * ptr;
    ptr p;
    __device__ __forceinline__ explicit Taps(const void *q) : p((ptr)(uintptr_t)q) {}
    __device__ __forceinline__ cpx<T> operator[](uint32_t i) const {
        const v2 x = p[i];
        return {x.x, x.y};
    }
    __device__ __forceinline__ Taps at(uint32_t i) const {
        Taps t(*this);
        t.p += i;
        return t;
    }
};

__device__ __forceinline__ void grid_add(double *p, double v) {
    typedef __attribute__((address_space(1))) double gdouble;
    (void)__builtin_amdgcn_global_atomic_fadd_f64((gdouble *)(uintptr_t)p, v);
}

// One tap of a sample: the product in the path's precision, added in FP64.
template <int CELLS, typename T>
__device__ __forceinline__ void add_tap(double *tile, uint32_t at, cpx<T> v, cpx<T> tap) {
    const T re = fma(v.re, tap.re, -(v.im * tap.im));
    const T im = fma(v.re, tap.im, v.im * tap.re);
    unsafeAtomicAdd(tile + at, (double)re);
    unsafeAtomicAdd(tile + CELLS + at, (double)im);
}

constexpr int tile_block(int W) { return W <= 15 ? 256 : W <= 31 ? 512 : 1024; }

// One item of width W on a zero tile.  Per tap: an 8-byte tap load (a sample's W x W block is
// contiguous, so the wavefront's loads are too), 4 FMAs on the sample's visibility (one value
// per wavefront, in scalar registers) and two LDS adds; the two adds bound it.  FP32 products
// are added in FP64, so nothing is lost to the order or number of the samples.
template <typename T, int W, int BLK, bool BATCH>
__device__ __forceinline__ void add_item(const TArgs &t, const wp::WArgs &w, const Item &it,
                                         uint32_t corr, double *tile) {
    constexpr int ST = W + TILE - 1, CELLS = ST * ST, TAPS = W * W;
    constexpr int PACK = TAPS >= 33 ? 1 : 64 / TAPS;       // samples per instruction
    constexpr int K = (TAPS + 63) / 64;                    // instructions per sample
    constexpr int KU = K < 8 ? K : 8;                      // of them in flight together
    constexpr int U = PACK > 1 ? 2 : K == 1 ? 8 : K == 2 ? 4 : K < 4 ? 2 : 1;   // samples in flight
    const int lane = threadIdx.x & 63;
    const Taps<T> taps(w.taps);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // records a wavefront takes at a time: 64, or its share of a short item
    constexpr uint32_t WAVES = BLK / 64;
    const uint32_t step = min(64u, (it.count + WAVES - 1) / WAVES);
    const uint32_t rsize = sizeof(Head) + t.ncorr * sizeof(cpx<T>);
    const unsigned char *recs = static_cast<const unsigned char *>(t.recs) +
                                (size_t)it.first * rsize;
    Head hn = {0, 0};              // the next records, loaded while these are added
    cpx<T> vn = {T(0), T(0)};
    auto fetch = [&](uint32_t b) {
        if (b + lane < it.count && lane < (int)step) {
            const unsigned char *p = recs + (size_t)(b + lane) * rsize;
            hn = *reinterpret_cast<const Head *>(p);
            vn = *reinterpret_cast<const cpx<T> *>(p + sizeof(Head) + corr * sizeof(cpx<T>));
        }
    };
    fetch(wave * step);
    for (uint32_t b = wave * step; b < it.count; b += WAVES * step) {
        const int n = (int)min(step, it.count - b);
        const Head h = hn;
        const cpx<T> vv = vn;
        fetch(b + WAVES * step);
        if constexpr (PACK > 1) {
            const int q = lane / TAPS, tt = lane - q * TAPS;
            const uint32_t off = (uint32_t)(tt + (TILE - 1) * (tt / W));
            for (int r = 0; r < n; r += PACK * U) {
                cpx<T> tp[U], vr[U];
                uint32_t at[U];
                bool on[U];
#pragma unroll
                for (int j = 0; j < U; ++j) {
                    const int src = r + j * PACK + q;
                    on[j] = q < PACK && src < n;
                    const uint32_t tb = (uint32_t)__shfl((int)h.tap, src & 63, 64);
                    at[j] = (uint32_t)__shfl((int)h.cell, src & 63, 64) + off;
                    vr[j] = {__shfl(vv.re, src & 63, 64), __shfl(vv.im, src & 63, 64)};
                    tp[j] = on[j] ? taps[tb + (uint32_t)tt] : cpx<T>{T(0), T(0)};
                }
#pragma unroll
                for (int j = 0; j < U; ++j)
                    if (on[j]) add_tap<CELLS>(tile, at[j], vr[j], tp[j]);
            }
        } else if constexpr (K == 1) {
            if (lane < TAPS) {   // lanes without a tap sit out the whole loop
                const uint32_t off = (uint32_t)(lane + (TILE - 1) * (lane / W));
                const Taps<T> lt = taps.at((uint32_t)lane);
                int r = 0;
                for (; r + U <= n; r += U) {
                    cpx<T> tp[U];
#pragma unroll
                    for (int j = 0; j < U; ++j)
                        tp[j] = lt[(uint32_t)__builtin_amdgcn_readlane((int)h.tap, r + j)];
#pragma unroll
                    for (int j = 0; j < U; ++j)
                        add_tap<CELLS>(
                            tile, off + (uint32_t)__builtin_amdgcn_readlane((int)h.cell, r + j),
                            cpx<T>{lane_value(vv.re, r + j), lane_value(vv.im, r + j)}, tp[j]);
                }
                for (; r < n; ++r)
                    add_tap<CELLS>(tile,
                                   off + (uint32_t)__builtin_amdgcn_readlane((int)h.cell, r),
                                   cpx<T>{lane_value(vv.re, r), lane_value(vv.im, r)},
                                   lt[(uint32_t)__builtin_amdgcn_readlane((int)h.tap, r)]);
            }
        } else {
            for (int r = 0; r < n; r += U) {
#pragma unroll 1
                for (int k0 = 0; k0 < K; k0 += KU) {
                    cpx<T> tp[U][KU];
#pragma unroll
                    for (int j = 0; j < U; ++j) {
                        const uint32_t tb =
                            (uint32_t)__builtin_amdgcn_readlane((int)h.tap, min(r + j, n - 1));
                        const Taps<T> blk = taps.at(tb);
#pragma unroll
                        for (int k = 0; k < KU; ++k)   // beyond the block: its last tap
                            tp[j][k] =
                                blk[min((uint32_t)(lane + 64 * (k0 + k)), (uint32_t)(TAPS - 1))];
                    }
#pragma unroll
                    for (int j = 0; j < U; ++j) {
                        if (r + j >= n) break;
                        const uint32_t cell =
                            (uint32_t)__builtin_amdgcn_readlane((int)h.cell, r + j);
                        const cpx<T> v = {lane_value(vv.re, r + j), lane_value(vv.im, r + j)};
#pragma unroll
                        for (int k = 0; k < KU; ++k) {
                            const uint32_t tt = (uint32_t)(lane + 64 * (k0 + k));
                            if (tt < TAPS)
                                add_tap<CELLS>(tile, cell + tt + (TILE - 1) * (tt / W), v,
                                               tp[j][k]);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    // the tile's nonzero cells into the grid: the two doubles of a cell in adjacent lanes, a
    // row's cells together (one request per 64-byte segment); footprints lie in the grid, so
    // cells beyond it are zero
    const size_t stride = (size_t)w.g.pstride * 2;
    double *g = w.g.grid + ((((size_t)(BATCH ? 0 : it.facet) * w.g.cube + it.slice) * w.g.ny +
                             (size_t)it.ty * TILE) * w.g.nx + (size_t)it.tx * TILE) * stride +
                2 * corr;
    for (int i = threadIdx.x; i < 2 * CELLS; i += BLK) {
        const int cell = i >> 1, comp = i & 1;
        const int y = cell / ST, x = cell - y * ST;
        const double val = tile[comp * CELLS + cell];
        tile[comp * CELLS + cell] = 0.0;
        if (val != 0.0) grid_add(g + ((size_t)y * w.g.nx + x) * stride + comp, val);
    }
}

// The items of widths W0, W0 + 2, .. W0 + 2 (N - 1).
template <typename T, int W0, int N, bool BATCH>
__global__ __launch_bounds__(tile_block(W0)) void wtile_kernel(TArgs t, uint32_t list) {
    constexpr int WM = W0 + 2 * (N - 1), CELLS = (WM + TILE - 1) * (WM + TILE - 1);
    constexpr int BLK = tile_block(W0);
    extern __shared__ __align__(16) double tile[];   // real parts, then imaginary parts
    __shared__ uint32_t s_item;
    const uint32_t NC = t.ncorr;
    const uint32_t total = t.item_count[list] * NC;
    if (blockIdx.x >= total) return;   // fewer items than workgroups
    for (int i = threadIdx.x; i < 2 * CELLS; i += BLK) tile[i] = 0.0;
    const Item *items = t.items + list_base(t, list);
    for (;;) {
        __syncthreads();   // the tile is zero
        if (threadIdx.x == 0) s_item = atomicAdd(t.queue + list, 1u);
        __syncthreads();
        const uint32_t id = __builtin_amdgcn_readfirstlane(s_item);
        if (id >= total) break;
        const Item it = items[id / NC];
        const uint32_t corr = id % NC;
        const wp::WArgs &w = BATCH ? t.w.facet_args[it.facet] : t.w;
        switch (it.half - W0 / 2) {
            case 0: add_item<T, W0, BLK, BATCH>(t, w, it, corr, tile); break;
            case 1: if constexpr (N > 1) add_item<T, W0 + 2, BLK, BATCH>(t, w, it, corr, tile); break;
            case 2: if constexpr (N > 2) add_item<T, W0 + 4, BLK, BATCH>(t, w, it, corr, tile); break;
            case 3: if constexpr (N > 3) add_item<T, W0 + 6, BLK, BATCH>(t, w, it, corr, tile); break;
        }
    }
}

template <typename T, int W0, int N, bool BATCH>
static hipError_t launch_w(const TArgs &t, uint32_t list, hipStream_t st) {
    constexpr int ST = W0 + 2 * (N - 1) + TILE - 1;
    const size_t smem = (size_t)2 * ST * ST * sizeof(double);
    static int per = 0;
    static int cus = 0;
    if (!per) {
        int dev = 0;
        (void)hipGetDevice(&dev);
        (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (cus <= 0) cus = 1;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, wtile_kernel<T, W0, N, BATCH>,
                                                         tile_block(W0), smem) != hipSuccess ||
            per <= 0)
            per = 1;
    }
    const uint64_t cap = (uint64_t)t.item_cap * list_widths(t, list) * t.ncorr;
    const uint64_t blocks = std::min<uint64_t>((uint64_t)per * cus, cap);
    wtile_kernel<T, W0, N, BATCH>
        <<<dim3((uint32_t)blocks), dim3(tile_block(W0)), smem, st>>>(t, list);
    return hipGetLastError();
}

template <typename T, bool BATCH>
static hipError_t launch_list(const TArgs &t, uint32_t list, hipStream_t st) {
    switch (list) {
        case 0: return launch_w<T, 1, 1, BATCH>(t, list, st);
        case 1: return launch_w<T, 3, 1, BATCH>(t, list, st);
        case 2: return launch_w<T, 5, 1, BATCH>(t, list, st);
        case 3: return launch_w<T, 7, 1, BATCH>(t, list, st);
        case 4: return launch_w<T, 9, 1, BATCH>(t, list, st);
        case 5: return launch_w<T, 11, 1, BATCH>(t, list, st);
        case 6: return launch_w<T, 13, 2, BATCH>(t, list, st);
        case 7: return launch_w<T, 17, 4, BATCH>(t, list, st);
        case 8: return launch_w<T, 25, 4, BATCH>(t, list, st);
        case 9: return launch_w<T, 33, 4, BATCH>(t, list, st);
        case 10: return launch_w<T, 41, 4, BATCH>(t, list, st);
        case 11: return launch_w<T, 49, 4, BATCH>(t, list, st);
        case 12: return launch_w<T, 57, 4, BATCH>(t, list, st);
    }
    return hipErrorInvalidValue;
}

template <int MODE, bool BATCH> static hipError_t prep_mode(const TArgs &t, bool fp64, uint32_t blocks,
                                                hipStream_t st, int pass) {
    const dim3 g(blocks, t.nfacets);
    if (pass == 0)
        k_count<MODE, BATCH><<<g, BLOCK, 0, st>>>(t);
    else if (fp64)
        k_scatter<MODE, double, BATCH><<<g, BLOCK, 0, st>>>(t);
    else
        k_scatter<MODE, float, BATCH><<<g, BLOCK, 0, st>>>(t);
    return hipGetLastError();
}

template <bool BATCH>
static hipError_t prep(const TArgs &t, int mode, bool fp64, uint32_t blocks, hipStream_t st,
                       int pass) {
    switch (mode) {
        case MODE_1: return prep_mode<MODE_1, BATCH>(t, fp64, blocks, st, pass);
        case MODE_2: return prep_mode<MODE_2, BATCH>(t, fp64, blocks, st, pass);
        case MODE_4: return prep_mode<MODE_4, BATCH>(t, fp64, blocks, st, pass);
        case MODE_4J: return prep_mode<MODE_4J, BATCH>(t, fp64, blocks, st, pass);
        case MODE_PSF: return prep_mode<MODE_PSF, BATCH>(t, fp64, blocks, st, pass);
    }
    return hipErrorInvalidValue;
}

}  // namespace wt

hipError_t fill_u32(uint32_t *p, uint32_t n, uint32_t v, hipStream_t st);

static size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

// Widths fix the bins: half supports lo .. hi of the call's planes.
bool wtile_plan(wt::Plan &p, uint64_t samples, uint64_t spots, uint32_t half_lo, uint32_t half_hi,
                int ncorr, bool fp64) {
    p.samples = samples;
    p.spots = spots;
    p.half_lo = half_lo;
    p.ncls = half_hi - half_lo + 1;
    if (samples >= (1ull << 31) || spots >= (1ull << 31)) return false;
    // fewer counters per bin where the bins are many (their samples are spread anyway)
    p.copies = wt::COPIES;
    uint64_t slots = spots * p.ncls * p.copies + 1;
    while (slots > wt::MAX_SLOTS / 4 && p.copies > 1) {
        p.copies /= 2;
        slots = spots * p.ncls * p.copies + 1;
    }
    if (slots > wt::MAX_SLOTS) return false;
    p.slots = (uint32_t)slots;
    // pieces small enough to fill the GPU, large enough to pay for clearing and adding a tile
    p.chunk = (uint32_t)std::min<uint64_t>(4096, std::max<uint64_t>(256, samples / 4096));
    p.item_cap = (uint32_t)std::min<uint64_t>(samples + 1, spots + samples / p.chunk + 1);
    size_t scan = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, scan, (uint32_t *)nullptr, (uint32_t *)nullptr,
                                           (int)p.slots);
    p.scan_bytes = scan;
    size_t o = 0;
    p.off_count = o;   o += up256((size_t)p.slots * 4);
    p.off_start = o;   o += up256(((size_t)p.slots + 1) * 4);
    p.off_meta = o;    o += up256(2 * 64 * 4);
    p.off_items = o;   o += up256((size_t)p.item_cap * p.ncls * sizeof(wt::Item));
    p.off_first = o;   o += up256(samples * 4);
    p.off_recs = o;    o += up256(samples * (sizeof(wt::Head) + (size_t)ncorr * (fp64 ? 16 : 8)));
    p.off_scan = o;    o += up256(scan);
    p.total = o;
    return true;
}

template <bool BATCH>
static hipError_t grid_pass(wt::TArgs t, const wt::Plan &p, void *ws, int mode, bool fp64,
                            const uint8_t *widths, hipStream_t st, hipStream_t *side, int nside,
                            hipEvent_t fork, hipEvent_t *join) {
    unsigned char *b = static_cast<unsigned char *>(ws);
    t.nspots = (uint32_t)p.spots;
    t.half_lo = p.half_lo;
    t.copies = p.copies;
    t.ncls = p.ncls;
    t.chunk = p.chunk;
    t.item_cap = p.item_cap;
    t.ncorr = (uint32_t)((mode == MODE_2) ? 2 : (mode == MODE_4 || mode == MODE_4J) ? 4 : 1);
    t.count = reinterpret_cast<uint32_t *>(b + p.off_count);
    t.first = reinterpret_cast<uint32_t *>(b + p.off_first);
    t.start = reinterpret_cast<uint32_t *>(b + p.off_start);
    t.item_count = reinterpret_cast<uint32_t *>(b + p.off_meta);
    t.queue = t.item_count + 64;
    t.items = reinterpret_cast<wt::Item *>(b + p.off_items);
    t.recs = b + p.off_recs;
    const uint64_t samples = (uint64_t)(t.row1 - t.row0) * t.w.g.chan;
    if (!samples || !t.nfacets) return hipSuccess;
    // samples a preparing lane takes before its sums are published: as many as leave the GPU
    // full (16384 wavefronts), at most 32
    t.iters = (uint32_t)std::min<uint64_t>(32, std::max<uint64_t>(1, samples * t.nfacets >> 20));
    const uint32_t per = wt::BLOCK * t.iters;
    const uint32_t blocks = (uint32_t)((samples + per - 1) / per);
    hipError_t e = fill_u32(t.count, p.slots, 0u, st);
    if (e == hipSuccess) e = fill_u32(t.item_count, 128, 0u, st);
    if (e == hipSuccess) e = wt::prep<BATCH>(t, mode, fp64, blocks, st, 0);
    if (e != hipSuccess) return e;
    size_t bytes = p.scan_bytes;
    e = hipcub::DeviceScan::ExclusiveSum(b + p.off_scan, bytes, t.count, t.start, (int)p.slots, st);
    if (e != hipSuccess) return e;
    wt::k_items<<<dim3((t.nspots + wt::BLOCK - 1) / wt::BLOCK, p.ncls), wt::BLOCK, 0, st>>>(t);
    e = hipGetLastError();
    if (e == hipSuccess) e = wt::prep<BATCH>(t, mode, fp64, blocks, st, 1);
    if (e != hipSuccess) return e;
    // one persistent launch per list, widest first, dealt over the streams
    if (nside) {
        e = hipEventRecord(fork, st);
        for (int i = 0; i < nside && e == hipSuccess; ++i) e = hipStreamWaitEvent(side[i], fork, 0);
        if (e != hipSuccess) return e;
    }
    int turn = 0;
    for (int l = wt::NLIST - 1; l >= 0 && e == hipSuccess; --l) {
        bool any = false;
        for (uint32_t h = wt::list_first(l); h < wt::list_first(l + 1) && h < 32; ++h)
            any |= widths[h] != 0;
        if (!any) continue;
        const int on = turn++ % (nside + 1);
        e = fp64 ? wt::launch_list<double, BATCH>(t, (uint32_t)l, on ? side[on - 1] : st)
                 : wt::launch_list<float, BATCH>(t, (uint32_t)l, on ? side[on - 1] : st);
    }
    // joined also after a failed launch: later work on the stream must not overtake these
    for (int i = 0; i < nside; ++i) {
        hipError_t j = hipEventRecord(join[i], side[i]);
        if (j == hipSuccess) j = hipStreamWaitEvent(st, join[i], 0);
        if (e == hipSuccess) e = j;
    }
    return e;
}

hipError_t wtile_grid(const wt::TArgs &t, const wt::Plan &p, void *ws, int mode, bool fp64,
                      const uint8_t *widths, hipStream_t st, hipStream_t *side, int nside,
                      hipEvent_t fork, hipEvent_t *join) {
    return t.w.facet_args
               ? grid_pass<true>(t, p, ws, mode, fp64, widths, st, side, nside, fork, join)
               : grid_pass<false>(t, p, ws, mode, fp64, widths, st, side, nside, fork, join);
}

}  // namespace bam
