// gz_kernels_f32.hip -- FP32-mixed instantiations.  Built with FMA contraction and the fast FP32
// divide/square root: this form is held to the stated tolerance against the FP64 oracle, not to
// its rounding order.  The FP64 pieces it keeps (positions, radius test, 3x3 inverse) follow
// the same source.
#include "gz_kernels_impl.h"
#include "gz_rows_impl.h"

namespace gz {

// ---------------------------------------------------------------------------------------
// instantiations
// ---------------------------------------------------------------------------------------

#define GZ_INST_LANES(KERN, R, BOXES)                                                                                           \
    template __global__ void k_gradients<KERN, R, BOXES>(DevParams, int, const int *, const double *, const GradLaneRec<R> *,   \
                                                         const double *, const double *,                                         \
                                                         long, const int *, long, const int *, double *, double *, double *,    \
                                                         BoxTable);                                                              \
    template __global__ void k_force<KERN, R, BOXES, false>(DevParams, Gam<R>, ForceView, const Cell<R> *, ForceRows, BoxTable);

#define GZ_INST_DROWS(KERN, R, TPB)                                                                                             \
    template __global__ void k_density_rows<KERN, R, TPB>(DevParams, GridView, int, const int *, const uint8_t *,               \
                                                          const uint32_t *, const double *, const double *, const double *,     \
                                                          const double *, const double *, const double *, const double *,       \
                                                          const double *, double *, BoxTable, int *, const int *, int);

#define GZ_INST_DCELLS(KERN, R, FD)                                                                                             \
    template __global__ void k_density_cells<KERN, R, FD>(DevParams, GridView, CellRows, const int *, const uint8_t *,          \
                                                          const double *, const double *, const double *, const double *,       \
                                                          const double *, const double *, const double *, const double *,       \
                                                          double *);

#define GZ_INST(KERN, R)                                                                                                         \
    GZ_INST_DCELLS(KERN, R, false)                                                                                               \
    GZ_INST_DCELLS(KERN, R, true)                                                                                                \
    GZ_INST_LANES(KERN, R, false)                                                                                                \
    GZ_INST_LANES(KERN, R, true)                                                                                                 \
    GZ_INST_DROWS(KERN, R, 64)                                                                                                   \
    GZ_INST_DROWS(KERN, R, kRowThreads)                                                                                          \
    template __global__ void k_gradients_rows<KERN, R>(DevParams, int, const int *, const double *, const double *,             \
                                                       const double *, const double *, const GradRec<R> *, GradSrc, const double *,             \
                                                       const double *, long, const int *, long, const int *, double *, double *,\
                                                       double *, BoxTable, int *);                                              \
    template __global__ void k_force_rows<KERN, R>(DevParams, Gam<R>, int, const int *, ForceView, const Cell<R> *,            \
                                                   const int *, long, const int *, const uint8_t *, const int *,                \
                                                   const double *, int *, double *, double *, double *, int *, int *,           \
                                                   unsigned long long *, BoxTable, const int *);                                \
    template __global__ void k_force_rows<KERN, R, false, kListThreads, true>(DevParams, Gam<R>, int, const int *, ForceView,  \
                                                   const Cell<R> *, const int *, long, const int *, const uint8_t *,            \
                                                   const int *, const double *, int *, double *, double *, double *, int *,     \
                                                   int *, unsigned long long *, BoxTable, const int *);
GZ_INST(3, float)
GZ_INST(6, float)
// the force kernel of quiet gas
#define GZ_INST_QUIET(KERN, BOXES)                                                                                               \
    template __global__ void k_force_lanes<KERN, BOXES>(DevParams, Gam<float>, ForceView, const Cell<float> *, ForceRows, BoxTable);
GZ_INST_QUIET(3, false)
GZ_INST_QUIET(6, false)
GZ_INST_QUIET(3, true)
GZ_INST_QUIET(6, true)
// the force kernels that count the Riemann rungs of their faces (one box)
#define GZ_INST_STATS(KERN, R)                                                                                                   \
    template __global__ void k_force<KERN, R, false, true>(DevParams, Gam<R>, ForceView, const Cell<R> *, ForceRows, BoxTable);     \
    template __global__ void k_force_rows<KERN, R, true>(DevParams, Gam<R>, int, const int *, ForceView, const Cell<R> *,      \
                                                         const int *, long, const int *, const uint8_t *, const int *,          \
                                                         const double *, int *, double *, double *, double *, int *, int *,     \
                                                         unsigned long long *, BoxTable, const int *);
GZ_INST_STATS(3, float)
GZ_INST_STATS(6, float)
template __global__ void k_riemann_probe<float>(int, Gam<float>, long, const double *, double *, unsigned *);
template __global__ void k_pack_grad<float, GradRec<float>>(long, const double *, const double *, const double *, const double *, const double *,
                                             const double *, const double *, GradRec<float> *, const double *, const double *,
                                             const double *, double, BoxTable);
template __global__ void k_pack_force<float>(double, ForceView, Cell<float> *, int *, double, BoxTable);
template __global__ void k_pack_grad_list<float, GradRec<float>>(int, const int *, const int *, long, const int *, const double *, const double *,
                                               const double *, const double *, const double *, const double *, const double *,
                                               GradRec<float> *, const double *, const double *, const double *, double, BoxTable);
template __global__ void k_pack_force_list<float>(int, const int *, const int *, long, const int *, double, ForceView, Cell<float> *,
                                                int *, double, BoxTable);
#undef GZ_INST

}  // namespace gz
