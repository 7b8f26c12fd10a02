// How the bins of a multihistogram run are cut over workgroups, and the LDS a
// workgroup asks for: plain host arithmetic, so that it can be checked without
// a device.
#pragma once
#include <algorithm>
#include <cstddef>

namespace ptmc {

constexpr int MH_THREADS = 256;
constexpr int MH_BINS = 128;                   // bins of a block, whose sums are formed together
constexpr size_t MH_LARGE = 96 * 1024;         // bytes of a slice above which few runs are cut

// LDS of mh_iterate_kernel in doubles: the temperatures' terms, and with KEEP
// a slice of `bins` bins (matrix, histogram sums, offsets, ratios)
constexpr size_t mh_lds(int R, bool keep, bool totals)
{
    return (size_t)3 * R + (keep || R <= MH_THREADS ? MH_THREADS : 0) + (totals ? R : 0);
}
constexpr size_t mh_slice(int R, size_t bins) { return bins * ((size_t)R + 3); }

struct MhCut {
    int n_blk, wg_blk, n_wg;  // blocks of a run, blocks of a workgroup, workgroups of a run
    bool keep;                // the slices fit LDS
    size_t lds;               // bytes
};

// Workgroups of a run of `bins` bins and R temperatures, one of `runs` runs, on
// a device of `cus` compute units with max_lds bytes of LDS that a workgroup can
// ask for.  Up to 512 bins (NVT histograms) one, if its slice fits LDS: an
// iteration (4 us) is not worth a barrier between workgroups (about 3 us), unless
// the slice is large and the runs few (20 iterations of one run of 32 x 500 bins
// on one workgroup 259 us, on four 233; of 16 runs 363, 404; 300 runs of 40 x 400
// 2197, 2416).  Else the bins are cut so that every slice fits LDS, and over more
// workgroups while the runs leave compute units idle (48 x 10^4 NPT bins: 79
// workgroups of one block each).  Where even one workgroup per compute unit would
// hold too much (20 x 400^2 bins fit, 48 x 400^2 do not) the slices are not kept.
inline MhCut mh_cut(int R, size_t bins, int runs, int cus, size_t max_lds)
{
    MhCut c{};
    c.n_blk = (int)((bins + MH_BINS - 1) / MH_BINS);
    auto cut = [&](int n) {
        c.wg_blk = (c.n_blk + n - 1) / n;
        c.n_wg = (c.n_blk + c.wg_blk - 1) / c.wg_blk;
    };
    auto slice = [&]() { return 8 * mh_slice(R, std::min(bins, (size_t)c.wg_blk * MH_BINS)); };
    cut(1);
    const size_t base = 8 * mh_lds(R, true, false);
    const size_t room = max_lds > base ? max_lds - base : 0;
    if (bins > 512 || slice() > room || (slice() > MH_LARGE && runs < 16)) {
        const size_t fit = room / (8 * mh_slice(R, MH_BINS));  // blocks of a slice
        const int need = fit > 0 ? (int)((c.n_blk + fit - 1) / fit) : c.n_blk;
        cut(std::max({1, std::min(c.n_blk, cus / runs), need <= cus ? need : 0}));
    }
    c.keep = slice() <= room;
    c.lds = c.keep ? base + slice() : 8 * mh_lds(R, false, false);
    return c;
}

}  // namespace ptmc
