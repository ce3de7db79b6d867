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

}  // namespace gz
