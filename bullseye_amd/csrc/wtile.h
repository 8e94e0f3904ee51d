// wtile.h -- arguments and plan of the tiled w-projection gridder (csrc/wtile.hip).
#pragma once
#include "wproj_args.h"

namespace bam {
namespace wt {

constexpr int TILE = 33;          // footprint origins per tile and axis (32 + 1: see the bank layout)
constexpr uint32_t COPIES = 16;   // counters per bin (at most), so a busy bin's atomics spread
// Counters of one pass at most.  The workspace beside the records is then 0.5 GiB of counters, as
// much of first places, and up to 3 GiB of work items.
constexpr uint64_t MAX_SLOTS = 1ull << 27;

__host__ __device__ constexpr uint32_t tiles_of(uint32_t n) { return (n + TILE - 1) / TILE; }

struct Head {
    uint32_t tap;    // first tap of the sample's W x W block
    uint32_t cell;   // first cell of the footprint in the tile (rows of W + TILE - 1 cells)
};

struct Item {        // up to TArgs::chunk consecutive records of one bin
    uint32_t facet, slice, half;
    uint16_t tx, ty;
    uint32_t first, count;
};

struct TArgs {
    wp::WArgs w;                 // call arguments; w.facet_args: per-facet arguments of a batch
    uint32_t f0, nfacets;        // facets of this pass
    const uint32_t *facet_list;  // batch: the pass's facets
    uint32_t row0, row1;         // sorted rows of this pass
    const uint32_t *spot_base;   // batch: first spot (slice, tile) of each facet of the pass
    uint32_t nspots;             // spots of the pass's facets
    uint32_t half_lo, ncls;      // half supports half_lo .. half_lo + ncls - 1
    uint32_t chunk, item_cap, ncorr, copies;
    uint32_t iters;              // samples per preparing lane
    uint32_t *count, *start;            // [bin][copies]; start has one more
    uint32_t *first;                    // [sample] reservations of k_count
    uint32_t *item_count, *queue;       // [list of widths]
    Item *items;                        // [width][item_cap], a list's widths together
    void *recs;                         // [record]: Head, then ncorr complex values
};

struct Plan {
    uint64_t samples, spots;
    uint32_t half_lo, ncls, copies, slots, chunk, item_cap;
    size_t off_count, off_start, off_meta, off_items, off_first, off_recs, off_scan, scan_bytes,
        total;
};

}  // namespace wt

// Workspace layout for at most `samples` samples (rows x channels x facets) over `spots` (facet,
// slice, tile) places and the half supports half_lo .. half_hi.  False when the bins or samples
// exceed what one pass can number.
bool wtile_plan(wt::Plan &p, uint64_t samples, uint64_t spots, uint32_t half_lo, uint32_t half_hi,
                int ncorr, bool fp64);
// One pass: t.w, facets, rows and (batch) facet_list and spot_base set by the caller, the rest from the plan's
// workspace.  widths[h] != 0: some plane has half support h.  The width launches are dealt over
// st and the side streams, forked and joined by events.
hipError_t wtile_grid(const wt::TArgs &t, const wt::Plan &p, void *ws, int mode, bool fp64,
                      const uint8_t *widths, hipStream_t st, hipStream_t *side, int nside,
                      hipEvent_t fork, hipEvent_t *join);

}  // namespace bam
