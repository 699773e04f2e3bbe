// pa_split.h - the cut of a prefill row block into ranges of its cells, shared by
// the kernels and the plan.  Plain C++ on the host as on the device.
#pragma once

#include <math.h>
#include <stdint.h>

#include "pa_gen_layout.h"   // IIAN_PA_HD

namespace iian_pa {

constexpr int kSplitMinCells = 1024;
constexpr int kMaxSplits = 16;   // p.n_split at most, for any head size
// Lanes of a merge that take a row of dv floats, 4 each; a row's (m, l) pairs
// must fit them (split_merge_rows).
inline int merge_lpr(int dv) { return dv <= 64 ? 16 : dv <= 128 ? 32 : 64; }

// Whether a launch of workgroups that have their CU alone is worth cutting for
// balance: uncut, it takes the longest of them, or its rounds of average ones,
// and that is well above an even share of the cells (records and the pieces'
// starts cost an even batch 12%: 8 chunks of 256 tokens over 6000 cells each 356
// against 400 us; over 4K-16K cells 784 us uncut, 627 cut).  blocks: the batch's
// row blocks; cells: the sum over them of their sequence's cells; longest: of
// one sequence.
IIAN_PA_HD inline bool prefill_uneven(float blocks, float cells, float longest, float heads, float cus) {
    const float share = cells * heads / cus;
    const float uncut = fmaxf(longest, ceilf(blocks * heads / cus) * (cells / fmaxf(blocks, 1.f)));
    return uncut > 1.2f * share;
}

struct SplitRange {
    int n;        // ranges of this row block
    int lo, hi;   // cells of range z (empty when z >= n)
};
// Range z of the cells [c_lo, c_hi) in whole tiles of `tile` cells.
IIAN_PA_HD inline SplitRange split_range(int c_lo, int c_hi, int z, int n_split, int tile) {
    const int cells = c_hi > c_lo ? c_hi - c_lo : 0, most = (cells + kSplitMinCells - 1) / kSplitMinCells;
    SplitRange r;
    r.n = most <= 1 ? 1 : most < n_split ? most : n_split;
    const int nt = (cells + tile - 1) / tile, per = (nt + r.n - 1) / r.n;
    const int lo = c_lo + z * per * tile, hi = lo + per * tile;
    r.lo = lo < c_hi ? lo : c_hi;
    r.hi = z >= r.n ? r.lo : hi < c_hi ? hi : c_hi;
    return r;
}

}  // namespace iian_pa
