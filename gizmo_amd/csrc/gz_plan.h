// gz_plan.h -- launch arithmetic of the host: grid sizes and the rules that choose between kernels
// by sizes.  Plain C++ (no HIP), so that the CPU tests compile it as it is.
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace gz {

constexpr int kXcds = 8;  // MI355X: 8 XCDs, each with its own L2
inline unsigned xcd_grid(long nblocks) { return (unsigned)(((nblocks + kXcds - 1) / kXcds) * kXcds); }

// Workgroups of 256 threads that find the stencils of ncell cells, 32 threads per cell.  A launch holds
// fewer than 2^32 threads along x, and a grid of 512^3 cells would take just that many: at most a
// quarter of them run, each striding over the cells (grids up to 256^3: one cell per 32 threads).
constexpr int kStencilThreads = 32;
inline unsigned stencil_grid(long ncell)
{
    const long most = 1L << 22, blocks = (kStencilThreads * ncell + 255) / 256;
    return (unsigned)(blocks < most ? blocks : most);
}

// Workgroups along y of the walk of ngroups row groups (k_build_sym_groups, whose time grows with a group's
// rows): while the groups do not fill the chip's 4096 places for its wavefronts, several share a group.  The
// list stage of 19,472 particles of a shock tube searched over many levels 1014 -> 447 us (with a lane per
// row 483), of a 33^3 lattice 457 -> 295; from 4096 groups on one workgroup each, as before.
inline unsigned group_parts(long ngroups)
{
    const long p = 4096 / (ngroups > 0 ? ngroups : 1);
    return (unsigned)(p < 1 ? 1 : (p > 8 ? 8 : p));
}

// Density rounds after the first of a batch's pass over many rows: whether the rows still iterating are
// taken one workgroup each, from the list that the closing kernel wrote, or by a walk of every group
// (the rows of one cell) again.  By row a row takes 2 to 4 ns (FP64 3 to 6).  A walk takes nearly as long for
// one row of a group as for all, and longer the more particles the cells hold: 28 to 35 ns a group
// at 16 to 64 particles per cell, 80 to 100 at 125, 200 at 244; each XCD walks a contiguous eighth
// of the groups, so the boxes of the fullest cells set the time; and below some 3000 groups it takes as long
// as one wavefront, 120 to 300 us.  The line: 5 rows per group and a sixth of the particles per cell in the
// fullest eighth of the cells, of at least 3072 groups.  24 batches (equal boxes of 20^3 to 128^3,
// mixtures of 12^3 to 110^3, both forms), their later rounds of 10 to 12 steps together: always the walk
// 428 ms, always by row up to half of the rows 375, this line 338, the faster way of each round 336; up to
// half of the rows, two boxes of 128^3 took 29.2 ms where the walk takes 19.8.  One box on one
// grid keeps nearly all rows or none after its first round: no list there.
constexpr long kFewGroups = 3072;
struct BoxCells { long particles, cells; };
// the mean number of particles per cell in the fullest eighth of the boxes' cells
inline double fullest_cells(std::vector<BoxCells> boxes)
{
    std::sort(boxes.begin(), boxes.end(), [](const BoxCells &a, const BoxCells &b) {
        return (double)a.particles * (double)b.cells > (double)b.particles * (double)a.cells;
    });
    double cells = 0;
    for (const BoxCells &b : boxes) cells += (double)b.cells;
    const double eighth = cells > 8 ? cells / 8 : 1;
    double left = eighth, held = 0;
    for (const BoxCells &b : boxes) {
        const double part = (double)b.cells < left ? (double)b.cells : left;
        held += part * (double)b.particles / (double)b.cells;
        left -= part;
    }
    return held / eighth;
}
inline bool density_by_row(long remaining, long ngroups, double per_cell)
{
    return (double)remaining <= (double)(ngroups > kFewGroups ? ngroups : kFewGroups) * (5.0 + per_cell / 6.0);
}

// The force pass over many rows (k_force): 64 rows of four lanes each per workgroup at a time.
constexpr int kForceRowsPerBlock = 64;
// at most this many list entries of a row between two rounds of queued faces: the lists of 64
// neighbours (at most ~90 entries) in one segment, and a queue that leaves room for the LDS of
// two workgroups on a CU
constexpr int kForceSegment = 96;
// workgroups of the fixed grid: two per CU of 256, by their registers (and, FP64, their LDS)
constexpr int kForceBlocks = 2 * 256;
// The launch of a pass over nrows rows with at most `room` bytes for the stored fluxes (a segment's
// entries x rows x 4 per workgroup; the whole grid with whole segments takes up to 100 MB).  Less
// room: shorter segments, down to eight entries, then fewer workgroups, and for eight workgroups still
// shorter segments.  segment 0: the room does not hold one entry for each of them (16 KB in FP64), and
// the pass cannot be launched.
struct ForcePlan {
    int blocks, segment;
    size_t bytes;
};
template <typename R> inline ForcePlan force_plan(long nrows, size_t room)
{
    const long nrb = (nrows + kForceRowsPerBlock - 1) / kForceRowsPerBlock;
    const size_t entry = (size_t)kForceRowsPerBlock * 4 * sizeof(R);
    long blocks = (long)xcd_grid(nrb < kForceBlocks ? nrb : kForceBlocks);
    long seg = (long)(room / ((size_t)blocks * entry));
    if (seg > kForceSegment) seg = kForceSegment;
    if (seg < 8) {
        seg = 8;
        blocks = (long)(room / (seg * entry)) / kXcds * kXcds;
        if (blocks < kXcds) {
            blocks = kXcds;
            seg = (long)(room / (blocks * entry));
        }
    }
    return ForcePlan{(int)blocks, (int)seg, (size_t)blocks * seg * entry};
}

// How even the lists of a pass are in the rows' plain order: their sum over 64 times the sum of the
// wavefronts' longest.  Below this the FP32 form sorts its rows by list length, block by block.
constexpr double kPlainEven = 0.75;
// Whether a pass over many rows of the FP32 form goes through one lane per row first (k_force_lanes), the rows
// with a face past the Riemann ladder's common case behind it through k_force: by the share of such
// rows and the evenness of the lists in the pass before (a guess of speed alone: every row's sums are
// the same; a context's first pass takes k_force).  Lanes first against k_force alone, 2M rows: no such
// rows 3.3 and 4.7 ms (a blast) or 3.4 and 5.5, 5% 3.9 and 6.6, 24% 5.2 and 7.1, 40% 6.4 and 7.3, 73% 8.8 and 7.5; 262K
// rows: none 0.46 and 0.69, 24% 0.72 and 0.88, 40% 0.93 and 0.90; 141K rows, two workgroups of lanes per CU: none
// 0.36 and 0.40, but 0.04% of the rows 0.46 and 0.41 (the few rows' own launch), 24% 0.61 and 0.51.  512K rows, no such
// rows, lists of evenness 0.92 0.92 and 1.39, 0.79 0.94 and 1.43, 0.71 1.37 and 1.20 (a wavefront of lanes lasts as long
// as its longest list); 1M rows of a lognormal field (0.53) 3.7 and 3.0.
constexpr long kLaneRows = 196608;
constexpr double kLaneShare = 0.25;
inline bool force_by_lanes(long nrows, double rare_share, double list_even)
{
    return nrows >= kLaneRows && rare_share <= kLaneShare && list_even >= kPlainEven;
}

}  // namespace gz
