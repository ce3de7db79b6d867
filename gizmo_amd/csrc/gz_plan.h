// gz_plan.h -- launch arithmetic of the host: grid sizes and the rules that choose between kernels
// by sizes.  Plain C++ (no HIP), so that the CPU tests compile it as it is.
#pragma once
#include <cstddef>

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

}  // namespace gz
