// gz_kernels_impl.h -- gfx950 kernels of the MFM hydro pipeline (templates; instantiated per
// arithmetic form in gz_kernels.hip (FP64, strict) and gz_kernels_f32.hip (FP32-mixed)).
//
// Layout: particles live on the device in structure-of-arrays form, ordered by a 30-bit
// Morton key of a fixed 1024^3 grid over the periodic box.  Any power-of-two search grid
// (cell side >= the search radius) is then a contiguous range of that order per cell, and
// the 27 neighbour-cell ranges of a cell, sorted by start, visit candidates in ascending
// device index: the canonical summation order, shared with the CPU oracle.
//
// Neighbour lists are ELLPACK: entry q of row r sits at ell[ell_at(ld, r, q)], four entries of a
// row side by side.  Wave64.
#pragma once
#include <type_traits>
#include "gz_kernels.h"

namespace gz {

// ---------------------------------------------------------------------------------------
// keys, gathers, scatters
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t spread10(uint32_t v)
{
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t compact10(uint32_t v)
{
    v &= 0x09249249u;
    v = (v | (v >> 2)) & 0x030c30c3u;
    v = (v | (v >> 4)) & 0x0300f00fu;
    v = (v | (v >> 8)) & 0x030000ffu;
    v = (v | (v >> 16)) & 0x000003ffu;
    return v;
}

__device__ __forceinline__ int fine_coord(double x, double box)
{
    double w = x - box * floor(x / box);
    int c = (int)(w * (double)kFine / box);
    return c < 0 ? 0 : (c >= kFine ? kFine - 1 : c);
}

#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_morton(long n, const double *__restrict__ pos, double box, uint32_t *__restrict__ key, int *__restrict__ val)
{
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t cx = fine_coord(pos[3 * i + 0], box), cy = fine_coord(pos[3 * i + 1], box), cz = fine_coord(pos[3 * i + 2], box);
    key[i] = (spread10(cx) << 2) | (spread10(cy) << 1) | spread10(cz);
    val[i] = (int)i;
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_morton_soa(long n, const double *__restrict__ X, const double *__restrict__ Y, const double *__restrict__ Z,
                             double box, uint32_t *__restrict__ key, int *__restrict__ val)
{
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t cx = fine_coord(X[i], box), cy = fine_coord(Y[i], box), cz = fine_coord(Z[i], box);
    key[i] = (spread10(cx) << 2) | (spread10(cy) << 1) | spread10(cz);
    val[i] = (int)i;
}

__global__ void k_permute_int(long n, const int *__restrict__ order, const int *__restrict__ in, int *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[s] = in[order[s]];
}

__global__ void k_permute_u8(long n, const int *__restrict__ order, const uint8_t *__restrict__ in, uint8_t *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[s] = in[order[s]];
}

// up to kPermCols 8-byte columns gathered by one order in one launch (every load of a lane
// issued before its stores: the columns are distinct buffers)
__global__ void __launch_bounds__(256) k_permute_many(long n, const int *__restrict__ order, PermCols P)
{
    const long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    const long u = order[s];
    unsigned long long v[kPermCols];
#pragma unroll
    for (int c = 0; c < kPermCols; c++)
        if (c < P.ncol) v[c] = P.in[c][u];
#pragma unroll
    for (int c = 0; c < kPermCols; c++)
        if (c < P.ncol) P.out[c][s] = v[c];
}

// the columns copied, in order (what k_permute_many left in a scratch area, back to its place)
__global__ void __launch_bounds__(256) k_copy_many(long n, PermCols P)
{
    const long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    unsigned long long v[kPermCols];
#pragma unroll
    for (int c = 0; c < kPermCols; c++)
        if (c < P.ncol) v[c] = P.in[c][s];
#pragma unroll
    for (int c = 0; c < kPermCols; c++)
        if (c < P.ncol) P.out[c][s] = v[c];
}

__global__ void k_gather_ll(long n, const int *__restrict__ perm, const long long *__restrict__ in, long long *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[s] = in[perm[s]];
}

__global__ void k_scatter_ll(long n, const int *__restrict__ perm, const long long *__restrict__ in, long long *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[perm[s]] = in[s];
}
#endif


// sorted field s <- user field perm[s] (width doubles per particle; interleaved in, SoA out
// when soa != 0 with column stride n)
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_gather(long n, int width, const int *__restrict__ perm, const double *__restrict__ in,
                         double *__restrict__ out, int soa)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    long u = perm[s];
    for (int c = 0; c < width; c++) {
        double v = in[(size_t)u * width + c];
        if (soa) out[(size_t)c * n + s] = v; else out[(size_t)s * width + c] = v;
    }
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_gather_int(long n, const int *__restrict__ perm, const int *__restrict__ in, int *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[s] = in[perm[s]];
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_gather_u8(long n, const int *__restrict__ perm, const uint8_t *__restrict__ in, uint8_t *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[s] = in[perm[s]];
}
#endif


// user field perm[s] <- sorted field s
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_scatter(long n, int width, const int *__restrict__ perm, const double *__restrict__ in,
                          double *__restrict__ out, int soa)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    long u = perm[s];
    for (int c = 0; c < width; c++) {
        double v = soa ? in[(size_t)c * n + s] : in[(size_t)s * width + c];
        out[(size_t)u * width + c] = v;
    }
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_scatter_int(long n, const int *__restrict__ perm, const int *__restrict__ in, int *__restrict__ out)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    out[perm[s]] = in[s];
}
#endif


// active rows: act[r] = sorted index of the r-th active particle (ascending)
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_flag_active(long n, const uint8_t *__restrict__ active, const double *__restrict__ mass, int *__restrict__ flag)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    flag[s] = (active == nullptr || active[s]) ? 1 : 0;
    (void)mass;
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_compact(long n, const int *__restrict__ flag, const int *__restrict__ scan, int *__restrict__ act)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    if (flag[s]) act[scan[s]] = (int)s;
}
#endif


// ---------------------------------------------------------------------------------------
// cell grid at level L (nc = 2^L): cells indexed by Morton code, [start, end) of the order
// ---------------------------------------------------------------------------------------
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_cell_clear(long ncell, int *__restrict__ cstart, int *__restrict__ cend, double *__restrict__ chmax)
{
    long c = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    cstart[c] = 0;
    cend[c] = 0;
    chmax[c] = 0;
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_cell_bounds(long n, const uint32_t *__restrict__ key, int shift, int *__restrict__ cstart, int *__restrict__ cend)
{
    long s = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (s >= n) return;
    uint32_t c = key[s] >> shift;
    if (s == 0 || (key[s - 1] >> shift) != c) cstart[c] = (int)s;
    if (s == n - 1 || (key[s + 1] >> shift) != c) cend[c] = (int)(s + 1);
}
#endif


// largest kernel radius per cell (the symmetric search reaches max(h_i, h_j))
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_cell_hmax(long ncell, const int *__restrict__ cstart, const int *__restrict__ cend,
                            const double *__restrict__ h, double *__restrict__ chmax)
{
    long c = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    double m = 0;
    for (int s = cstart[c]; s < cend[c]; s++) m = fmax(m, h[s]);
    chmax[c] = m;
}
#endif


// the (deduplicated) 27 neighbour cells of each cell, non-empty ones only, sorted by start;
// each entry packs start, end and the offset code (dx+1)*9+(dy+1)*3+(dz+1).  Half a wavefront per
// cell, one lane per neighbour: a lane's place is its rank among the kept starts, counted over
// shuffles.  (One thread per cell with its entries sorted in scratch took 145-175 us whatever the
// grid, all of it the chain of 27 dependent loads and the insertion sort: a third of a pass over a
// few thousand particles.)
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(256) k_cell_stencil(int level, const int *__restrict__ cstart, const int *__restrict__ cend,
                                                      int4 *__restrict__ sten, int *__restrict__ nsten)
{
    const long ncell = 1L << (3 * level);
    const int lane = threadIdx.x & 31;
    const int nc = 1 << level;
    const int none = 0x7fffffff;
    // (whole halves of a wavefront run and leave together: the shuffles stay within one half)
    for (long c = (blockIdx.x * (long)blockDim.x + threadIdx.x) >> 5; c < ncell; c += (gridDim.x * (long)blockDim.x) >> 5) {
        const int cx = compact10((uint32_t)c >> 2), cy = compact10((uint32_t)c >> 1), cz = compact10((uint32_t)c);
        int st = none, en = 0;
        uint32_t code = 0;
        if (lane < 27) {
            const int dx = lane / 9 - 1, dy = (lane / 3) % 3 - 1, dz = lane % 3 - 1;
            const int a = (cx + dx + nc) % nc, b = (cy + dy + nc) % nc, d = (cz + dz + nc) % nc;
            code = (spread10(a) << 2) | (spread10(b) << 1) | spread10(d);
            st = cstart[code];
            en = cend[code];
            if (en <= st) st = none;
        }
        if (nc < 3) {
            // neighbours coincide on such grids: the first lane of each start stays
            bool dup = false;
            for (int q = 0; q < 27; q++) dup |= __shfl(st, q, 32) == st && q < lane;
            if (dup) st = none;
        }
        int rank = 0, m = 0;
        for (int q = 0; q < 27; q++) {
            const int s = __shfl(st, q, 32);
            rank += s < st;
            m += s != none;
        }
        if (st != none) sten[c * 27 + rank] = make_int4(st, en, lane, (int)code);
        if (lane == 0) nsten[c] = m;
    }
}
#endif


// ---------------------------------------------------------------------------------------
// neighbour lists (gpu_ngb_list_build, src/mesh/gpu_neighbor_list.cc:1950, exact FP64 accept)
//   SYMMETRIC = false: rows r2 < (scale*h_i)^2, self included (density, scale = 1.3 buffer)
//   SYMMETRIC = true : rows r2 < max(h_i,h_j)^2, self excluded (gradients, force)
// rows: the slots listed in rows[0..nrows) (row r of the list is slot rows[k]); act[slot] =
// sorted index of that slot's particle.
// ---------------------------------------------------------------------------------------
template <bool SYMMETRIC>
__global__ void __launch_bounds__(256) k_build_ell(int nrows, const int *__restrict__ rows, const int *__restrict__ act,
                                                   const double *__restrict__ hrow, double scale, const double *__restrict__ X,
                                                   const double *__restrict__ Y, const double *__restrict__ Z, const double *__restrict__ H,
                                                   const uint32_t *__restrict__ key, GridView g, int *__restrict__ ell, long ld, int cap,
                                                   int *__restrict__ cnt, int *__restrict__ overflow)
{
    const long k = xcd_block() * blockDim.x + threadIdx.x;
    if (k >= nrows) return;
    const int r = rows ? rows[k] : (int)k;
    const int i = act[r];
    const double xi = X[i], yi = Y[i], zi = Z[i];
    const double hi = hrow ? hrow[r] * scale : H[i];
    const uint32_t home = key[i] >> g.shift;
    const int nc = 1 << g.level;
    const int cx = compact10(home >> 2), cy = compact10(home >> 1), cz = compact10(home);
    const bool prune = nc >= 3;
    const int m = g.nsten[home];
    int c = 0;
    for (int q = 0; q < m; q++) {
        const int4 e = g.sten[(size_t)home * 27 + q];
        if (prune) {
            double reach = hi;
            if (SYMMETRIC) reach = fmax(hi, g.chmax[e.w]);
            reach = reach * (1.0 + 1e-9) + 1e-6 * g.cell;
            const int dx = e.z / 9 - 1, dy = (e.z / 3) % 3 - 1, dz = e.z % 3 - 1;
            const double lx = (cx + dx) * g.cell, ly = (cy + dy) * g.cell, lz = (cz + dz) * g.cell;
            const double xw = xi - g.box * floor(xi / g.box), yw = yi - g.box * floor(yi / g.box), zw = zi - g.box * floor(zi / g.box);
            double ex = fmax(fmax(lx - xw, xw - (lx + g.cell)), 0.0);
            double ey = fmax(fmax(ly - yw, yw - (ly + g.cell)), 0.0);
            double ez = fmax(fmax(lz - zw, zw - (lz + g.cell)), 0.0);
            if (ex * ex + ey * ey + ez * ez > reach * reach) continue;
        }
        for (int j = e.x; j < e.y; j++) {
            if (SYMMETRIC && j == i) continue;
            if (accept_pair<SYMMETRIC>(xi, yi, zi, X[j], Y[j], Z[j], hi, H[j], g.box, g.half)) {
                if (c < cap) ell[ell_at(ld, r, c)] = j;
                c++;
            }
        }
    }
    cnt[r] = min(c, cap);  // readers stay inside the list; the overflow carries the full length
    if (c > cap) atomicMax(overflow, c);
}

// ---------------------------------------------------------------------------------------
// density: fused pair sums (DensitySpec::pair_kernel, src/hydro/density_loop.h:1141-1385),
// after_iter_body (:516-961) and, on convergence, density_finalize_post_runner
// (src/hydro/density_loop.cc:303-733)
// ---------------------------------------------------------------------------------------
__device__ inline void density_finalize(const DevParams &P, const DensityOut &o, int i, double h, const double *acc, const DensityNorm &dn,
                                        double mass, double u)
{
    o.h[i] = h;
    const double nn = dn.nn, normalizer = dn.normalizer;
    o.drk[i] = dn.dr;
    o.divv[i] = dn.dv;
    for (int k = 0; k < 3; k++) o.fw[(size_t)k * o.n + i] = acc[10 + k];
    o.t[0 * o.n + i] = dn.Ti[0] / normalizer;
    o.t[1 * o.n + i] = dn.Ti[4] / normalizer;
    o.t[2 * o.n + i] = dn.Ti[8] / normalizer;
    o.t[3 * o.n + i] = dn.Ti[1] / normalizer;
    o.t[4 * o.n + i] = dn.Ti[5] / normalizer;
    o.t[5 * o.n + i] = dn.Ti[2] / normalizer;
    o.cn[i] = dn.cn;
    o.fce[i] = dn.fce;
    double rho = acc[1];
    if (mass > 0) {
        if ((h > 0) && (nn > 0)) rho = mass * nn / (kVolNorm * pow(h, 3.0));
        else if (h <= 0) rho = 0;
        else rho = mass / (kVolNorm * pow(h, 3.0));
        if (P.fd4alpha > 0 && acc[16] != 0) {
            // the first-derivative partition-of-unity volume correction (src/hydro/density_loop.cc:622-633):
            // grad H = -GradH_numer / GradH_denom, the density divided by 1 + 4 alpha |grad H|^2
            const double inv_denom = -1.0 / acc[16];
            const double g0 = acc[13] * inv_denom, g1 = acc[14] * inv_denom, g2 = acc[15] * inv_denom;
            rho /= 1.0 + P.fd4alpha * (g0 * g0 + g1 * g1 + g2 * g2);
        }
        o.p[i] = (P.gamma - 1) * u * rho;
    }
    o.rho[i] = rho;
    o.nn[i] = (nn > 0) ? pow(nn, 1.0 / 3.0) : 0.0;
}

// ---------------------------------------------------------------------------------------
// per-cell active rows: the active slots of one grid cell are a contiguous range of act[]
// (act ascends in device order, cells are contiguous in it); one entry per occupied cell
// ---------------------------------------------------------------------------------------
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_cell_rows_mark(int nact, const int *__restrict__ act, const uint32_t *__restrict__ key, int shift,
                                 int *__restrict__ ca0, int *__restrict__ ca1, int *__restrict__ flag)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nact) return;
    const uint32_t c = key[act[r]] >> shift;
    const bool first = (r == 0) || ((key[act[r - 1]] >> shift) != c);
    const bool last = (r == nact - 1) || ((key[act[r + 1]] >> shift) != c);
    if (first) ca0[c] = r;
    if (last) ca1[c] = r + 1;
    flag[r] = first ? 1 : 0;
}
#endif


#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void k_cell_rows_list(int nact, const int *__restrict__ act, const uint32_t *__restrict__ key, int shift,
                                 const int *__restrict__ flag, const int *__restrict__ scan, int *__restrict__ cells)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nact) return;
    if (flag[r]) cells[scan[r]] = (int)(key[act[r]] >> shift);
}
#endif


__device__ __forceinline__ bool wave_any(bool v) { return __builtin_amdgcn_ballot_w64(v) != 0; }

// ---------------------------------------------------------------------------------------
// leaf culling for the cell walks.  A wavefront's particles (one leaf) have a bounding box in
// coordinates relative to the home cell's origin; a candidate farther from that box than the
// reach of the pair test cannot be accepted by any lane and is dropped while its tile is
// staged, keeping the survivors in ascending order (stable compaction over the ballot mask).
// The test is conservative: the slack covers rounding of the relative coordinates.
// ---------------------------------------------------------------------------------------
struct LeafBox {
    double ox, oy, oz;          // home cell origin
    double lo[3], hi[3];        // leaf box, relative to the origin
    bool cull;                  // false on grids too coarse for relative coordinates
};

__device__ __forceinline__ double wave_min(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ float wave_minf(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ LeafBox leaf_box(const GridView &g, int c, bool on, double xi, double yi, double zi)
{
    LeafBox b;
    const int cx = compact10((uint32_t)c >> 2), cy = compact10((uint32_t)c >> 1), cz = compact10((uint32_t)c);
    b.ox = cx * g.cell; b.oy = cy * g.cell; b.oz = cz * g.cell;
    const double rx = wrap(xi - b.ox, g.box, g.half), ry = wrap(yi - b.oy, g.box, g.half), rz = wrap(zi - b.oz, g.box, g.half);
    b.lo[0] = wave_min(on ? rx : 1e300); b.hi[0] = wave_max(on ? rx : -1e300);
    b.lo[1] = wave_min(on ? ry : 1e300); b.hi[1] = wave_max(on ? ry : -1e300);
    b.lo[2] = wave_min(on ? rz : 1e300); b.hi[2] = wave_max(on ? rz : -1e300);
    b.cull = (1 << g.level) >= 4;
    return b;
}

__device__ __forceinline__ bool leaf_reach(const GridView &g, const LeafBox &b, double xj, double yj, double zj, double reach)
{
    if (!b.cull) return true;
    const double rx = wrap(xj - b.ox, g.box, g.half), ry = wrap(yj - b.oy, g.box, g.half), rz = wrap(zj - b.oz, g.box, g.half);
    const double ex = fmax(fmax(b.lo[0] - rx, rx - b.hi[0]), 0.0);
    const double ey = fmax(fmax(b.lo[1] - ry, ry - b.hi[1]), 0.0);
    const double ez = fmax(fmax(b.lo[2] - rz, rz - b.hi[2]), 0.0);
    const double rr = reach * (1.0 + 1e-9) + 1e-12 * g.box;
    return ex * ex + ey * ey + ez * ez <= rr * rr;
}

// a lane's value in every lane (a: the same lane for all)
__device__ __forceinline__ int lane_value(int v, int a) { return __builtin_amdgcn_readlane(v, a); }
__device__ __forceinline__ float lane_value(float v, int a) { return __int_as_float(lane_value(__float_as_int(v), a)); }
__device__ __forceinline__ double lane_value(double v, int a)
{
    return __hiloint2double(lane_value(__double2hiint(v), a), lane_value(__double2loint(v), a));
}

// position of this lane among the kept lanes below it (stable compaction)
__device__ __forceinline__ int kept_rank(bool keep, int &count)
{
    const unsigned long long m = __ballot(keep ? 1 : 0);
    count = __popcll(m);
    const unsigned lane = threadIdx.x & 63;
    return __popcll(m & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
}

// The difference of two coordinates of a pair closer than half a box: d brought to the nearest
// image, d - box * rint(d / box).  The product is exact (the factor is -1, 0 or 1), so the bits
// are those of wrap() in three instructions instead of eight; only a difference that rounds
// onto half a box may take the other image, which no pair within reach of a kernel has.
__device__ __forceinline__ double wrap_near(double d, double box, double inv_box)
{
    return __builtin_fma(-__builtin_rint(d * inv_box), box, d);
}

// the square of the distance of two points in units of the cell side on a periodic grid of nc cells
// a side (for grids so coarse that positions relative to a cell may wrap).  Small boxes live on such
// grids: this mask took the density walk of twelve boxes of 16^3 to 64^3 from 901 to 800 us and their
// symmetric list from 1101 to 796, against testing every candidate in FP64 by 78 instructions.
__device__ __forceinline__ float wrapped_r2(float ux, float uy, float uz, const float4 &v, float nc, float inv_nc)
{
    float dx = ux - v.x, dy = uy - v.y, dz = uz - v.z;
    dx = __builtin_fmaf(-__builtin_rintf(dx * inv_nc), nc, dx);
    dy = __builtin_fmaf(-__builtin_rintf(dy * inv_nc), nc, dy);
    dz = __builtin_fmaf(-__builtin_rintf(dz * inv_nc), nc, dz);
    return dx * dx + dy * dy + dz * dz;
}

// m = 2 m + (t <= lim): one candidate's bit into a lane's mask in two instructions
__device__ __forceinline__ void mask_push(uint32_t &m, float t, float lim)
{
    __asm__("v_cmp_le_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(t), "v"(lim) : "vcc");
}

// ---------------------------------------------------------------------------------------
// Cell walk's candidate window.  Most candidates a wavefront stages lie outside a given row's
// radius (72 of 432 on a 64-neighbour lattice), so testing each of them with the pair body
// behind the test runs the body for every candidate that any lane accepts: all of them.
// Instead a tile of 64 culled candidates is tested first in FP32 (coordinates in units of the
// cell side around the cell's centre: |x_j|^2 - 2 x_i.x_j against h_i^2 - |x_i|^2, four
// instructions a candidate, with a slack that covers every rounding, so no partner is missed),
// each lane keeping one bit per candidate; the lanes then take their own candidates one by one
// through the exact test and the body.  The last kWinWords tiles stay in LDS, and a new one is
// taken only when every lane is done with the oldest: lanes with few candidates in one tile
// run ahead into the next ones, so the body runs nearly as often as the longest lane needs it
// (78 times for rows of 77 partners among 432 culled candidates; 115 with a window of three
// tiles, 203 with one).  Each lane takes its candidates in ascending order.
// ---------------------------------------------------------------------------------------
constexpr int kWinWords = 5;                     // tiles in the window
constexpr int kWinRing = 64 * (kWinWords + 1);   // staged candidates: the window and the tile being filled
// r^2 in units of the cell side squared: |x| <= 2 along each axis (a stencil cell and the
// distance a particle may have moved, at most half a cell), |x|^2 <= 12, a dozen roundings of
// 2^-24 each of at most 24: below 2e-5
constexpr float kWinSlack = 3e-5f;

// A lane's queue of masks: m[0] belongs to the tile at ring slot `at`, `behind` tiles before the
// newest, the others to the tiles after it.
struct Window {
    unsigned long long m[kWinWords];
    int at = 0, behind = -1;
    __device__ __forceinline__ Window()
    {
        for (int w = 0; w < kWinWords; w++) m[w] = 0;
    }
    // a new tile's mask (behind < kWinWords - 1 in every lane)
    __device__ __forceinline__ void push(unsigned long long mask)
    {
        behind++;
        for (int w = 0; w < kWinWords; w++) m[w] = behind == w ? mask : m[w];
    }
    // on to the next tile when this lane is done with its oldest; whether it has a candidate now
    __device__ __forceinline__ bool ready()
    {
        const bool done = m[0] == 0 && behind >= 0;
        for (int w = 0; w + 1 < kWinWords; w++) m[w] = done ? m[w + 1] : m[w];
        m[kWinWords - 1] = done ? 0 : m[kWinWords - 1];
        behind -= done;
        at += done ? 64 : 0;
        at = at == kWinRing ? 0 : at;
        return m[0] != 0;
    }
    // the ring slot of this lane's next candidate (ready() holds)
    __device__ __forceinline__ int next()
    {
        const int slot = at + (int)__builtin_ctzll(m[0]);
        m[0] &= m[0] - 1;
        return slot;
    }
};

// ---------------------------------------------------------------------------------------
// density as a cell walk: one wavefront per occupied cell, its active particles one per lane;
// the candidates of the cell's 27 neighbour ranges are staged through LDS after leaf culling
// and go through the candidate window above, every lane taking its own in ascending order (the
// oracle's summation order).  need[r] marks the rows still iterating.  The 13 pair sums of
// DensitySpec::pair_kernel (src/hydro/density_loop.h:1141-1385) go to acc[13*r];
// k_density_after closes the round.  Bound by the body's VALU instructions (140 per candidate taken
// in FP64, a third of them the square root and the division).  2M rows: FP64 3.45 -> 1.52 ms, FP32
// 1.64 -> 1.11 ms against the body behind the test of every candidate; a window of three tiles
// with branches around the sums (each copied all of them) took 2.12 and 1.45 ms.
// ---------------------------------------------------------------------------------------
template <int KERN, typename R, bool FD>
__global__ void __launch_bounds__(64) k_density_cells(DevParams P, GridView g, CellRows cr, const int *__restrict__ act,
                                                      const uint8_t *__restrict__ need, const double *__restrict__ X,
                                                      const double *__restrict__ Y, const double *__restrict__ Z,
                                                      const double *__restrict__ VX, const double *__restrict__ VY,
                                                      const double *__restrict__ VZ, const double *__restrict__ M,
                                                      const double *__restrict__ hcur, double *__restrict__ accout)
{
    // the staged candidates: positions in FP64 (FP32 form on grids of 8 cells a side or more: as
    // floats relative to the cell's origin, in the same memory), velocities and masses, and the
    // tile being filled in cell units for the FP32 test
    __shared__ double sx[kWinRing], sy[kWinRing], sz[kWinRing];
    __shared__ R svx[kWinRing], svy[kWinRing], svz[kWinRing], sm[kWinRing];
    __shared__ float4 st[64];
    const long cb = xcd_block();
    if (cb >= (cr.ncells_dev ? *cr.ncells_dev : cr.ncells)) return;
    int c, a0, a1, nst;
    const int4 *sten;
    if (cr.gsten) {
        c = cr.gcode[cb]; a0 = cr.gstart[cb]; a1 = cr.gstart[cb + 1]; nst = cr.gnst[cb]; sten = cr.gsten + (size_t)27 * cb;
        if (cr.bt.b) {
            resolve_box(cr.bt, act[cr.grow ? cr.grow[a0] : a0], P, g);
        } else {
            g.level = cr.glev[cb];
            g.cell = g.box / (double)(1 << g.level);
        }
    } else {
        c = cr.cells[cb]; a0 = cr.ca0[c]; a1 = cr.ca1[c]; nst = g.nsten[c]; sten = g.sten + (size_t)c * 27;
    }
    const int t = threadIdx.x;
    const double inv_box = 1.0 / P.box;
    // a lane without a candidate reads ring slots that may not be staged yet: zeros
    for (int k = t; k < kWinRing; k += 64) {
        sx[k] = sy[k] = sz[k] = 0;
        svx[k] = svy[k] = svz[k] = sm[k] = 0;
    }
    // a cell's rows in equal parts of at most 64, dealt to the workgroups along y
    const int parts = (a1 - a0 + 63) / 64, part_rows = (a1 - a0 + parts - 1) / parts;
    for (int part = blockIdx.y; part < parts; part += gridDim.y) {
        const int base = a0 + part * part_rows;
        const bool in = t < part_rows && base + t < a1;
        const int r = in ? (cr.grow ? cr.grow[base + t] : base + t) : 0;
        const bool on = in && need[r];
        if (!wave_any(on)) continue;
        int i = 0;
        double xi = 0, yi = 0, zi = 0, h = 0;
        R vxi = 0, vyi = 0, vzi = 0;
        if (on) {
            i = act[r];
            xi = X[i]; yi = Y[i]; zi = Z[i];
            vxi = (R)VX[i]; vyi = (R)VY[i]; vzi = (R)VZ[i];
            h = hcur[r];
        }
        const LeafBox lb = leaf_box(g, c, on, xi, yi, zi);
        const double reach = wave_max(on ? h : 0.0);
        // grids of at least 8 cells a side: every partner lies within half a box of the home
        // cell's origin, so relative positions (one FP64 difference and wrap per row and per
        // staged candidate) give the pairs' differences: the FP32 test of the window, and the
        // FP32 form's pair differences
        const bool small = (1 << g.level) >= 8;
        const bool rel = std::is_same<R, float>::value && small;
        const R rxi = (R)wrap(xi - lb.ox, g.box, g.half), ryi = (R)wrap(yi - lb.oy, g.box, g.half),
                rzi = (R)wrap(zi - lb.oz, g.box, g.half);
        const double inv_cell = 1.0 / g.cell;
        const float ux = (float)(wrap(xi - lb.ox, g.box, g.half) * inv_cell - 0.5), uy = (float)(wrap(yi - lb.oy, g.box, g.half) * inv_cell - 0.5),
                    uz = (float)(wrap(zi - lb.oz, g.box, g.half) * inv_cell - 0.5), uh = (float)(h * inv_cell);
        const float qx = -2.0f * ux, qy = -2.0f * uy, qz = -2.0f * uz;
        // (small: the limit of |x_j|^2 - 2 x_i.x_j, else that of the distance's square)
        const float lim = on ? (small ? uh * uh - (ux * ux + uy * uy + uz * uz) : uh * uh) + kWinSlack : -1e30f;
        constexpr int nsum = FD ? kDensSumsFD : kDensSums;
        R a[nsum];
        for (int q = 0; q < nsum; q++) a[q] = 0;
        const R hR = (R)(on ? h : 1.0);
        const R h2 = hR * hR;
        R hinv, hinv3, hinv4;
        kernel_hinv(hR, hinv, hinv3, hinv4);
        Window win;
        int head = 0;  // ring slot of the tile being filled
        int q = 0, ts = nst > 0 ? sten[0].x : 0, te = nst > 0 ? sten[0].y : 0;  // the next candidates
        int fill = 0;       // candidates in the tile being filled
        bool keep = false;  // this lane holds a candidate for the next tile, at place pos
        int pos = 0, j = 0;
        double xj = 0, yj = 0, zj = 0;
        bool more = nst > 0, left = false;
        // the next 64 candidates' positions, loaded while the last are tested and staged (with the
        // walk in parts along y: twelve boxes of 16^3 to 64^3 800 -> 718 us; 128^3, where six other
        // wavefronts on the CU hide the loads already, 1490 either way)
        double xn = 0, yn = 0, zn = 0;
        auto load_next = [&]() {
            if (ts + t < te) {
                xn = X[ts + t]; yn = Y[ts + t]; zn = Z[ts + t];
            }
        };
        load_next();
        // a candidate into the tile being filled
        auto stage = [&](int k) {
            const int s = head + k;
            const double ux = wrap(xj - lb.ox, g.box, g.half), uy = wrap(yj - lb.oy, g.box, g.half), uz = wrap(zj - lb.oz, g.box, g.half);
            if (rel) {
                ((float *)sx)[s] = (float)ux; ((float *)sy)[s] = (float)uy; ((float *)sz)[s] = (float)uz;
            } else {
                sx[s] = xj; sy[s] = yj; sz[s] = zj;
            }
            const double mj = M[j];
            svx[s] = (R)VX[j]; svy[s] = (R)VY[j]; svz[s] = (R)VZ[j]; sm[s] = (R)mj;
            // (FP32 form: a mass may round to 0 that is not, so a retired particle is dropped here, as no
            // comparison with a NaN holds; the FP64 form tests the staged mass, 1.44 ms instead of 1.50)
            const float fx = std::is_same<R, float>::value && mj <= 0 ? __builtin_nanf("") : (float)(ux * inv_cell - 0.5), fy = (float)(uy * inv_cell - 0.5), fz = (float)(uz * inv_cell - 0.5);
            st[k] = make_float4(fx, fy, fz, fx * fx + fy * fy + fz * fz);
        };
        while (more || left) {
            __syncthreads();  // the lanes are done with the tile before the last and its test values
            if (keep) stage(pos);  // what the last tile had no room for
            keep = false;
            left = false;
            while (more && fill < 64) {
                const bool in_range = ts + t < te;
                j = ts + t;
                xj = xn; yj = yn; zj = zn;
                ts += 64;
                if (ts >= te) {
                    q++;
                    more = q < nst;
                    if (more) { ts = sten[q].x; te = sten[q].y; }
                }
                if (more) load_next();
                keep = in_range && leaf_reach(g, lb, xj, yj, zj, reach);
                int nt;
                pos = fill + kept_rank(keep, nt);
                if (keep && pos < 64) {
                    stage(pos);
                    keep = false;
                }
                fill += nt;
            }
            const int nt = fill < 64 ? fill : 64;
            fill -= nt;
            left = fill > 0;
            pos -= 64;
            if (t >= nt) st[t] = make_float4(0.0f, 0.0f, 0.0f, 1e30f);  // no candidate
            __syncthreads();
            uint32_t mlo = 0, mhi = 0;
            if (small) {
#pragma unroll 4
                for (int k = 31; k >= 0; k--) {
                    const float4 u = st[k], v = st[k + 32];
                    mask_push(mlo, __builtin_fmaf(qx, u.x, __builtin_fmaf(qy, u.y, __builtin_fmaf(qz, u.z, u.w))), lim);
                    mask_push(mhi, __builtin_fmaf(qx, v.x, __builtin_fmaf(qy, v.y, __builtin_fmaf(qz, v.z, v.w))), lim);
                }
            } else {
                // coarse grids: the nearest image of each difference (a candidate beyond nt lies at
                // the cell's centre: masked off)
                const float nc = (float)(1 << g.level), inv_nc = 1.0f / nc;
                for (int k = 31; k >= 0; k--) {
                    mask_push(mlo, wrapped_r2(ux, uy, uz, st[k], nc, inv_nc), lim);
                    mask_push(mhi, wrapped_r2(ux, uy, uz, st[k + 32], nc, inv_nc), lim);
                }
                const unsigned long long valid = nt == 64 ? ~0ull : (1ull << nt) - 1ull;
                mlo &= (uint32_t)valid;
                mhi &= (uint32_t)(valid >> 32);
            }
            win.push(((unsigned long long)mhi << 32) | mlo);
            head = head == kWinRing - 64 ? 0 : head + 64;
            // until the next tile has room (the last tile: until every candidate is taken)
            const int room = more || left ? kWinWords - 2 : -1;
            do {
                // one region without branches (a branch around the sums would copy all of them): a
                // lane without a candidate, a candidate that is no partner, and the row itself
                // (rr = 0) add zeros, which leave a sum that starts at +0 as it is bit for bit
                const bool got = win.ready();
                const int k = got ? win.next() : 0;
                const R mj = sm[k];
                R dp0, dp1, dp2;
                if (rel) {
                    dp0 = rxi - (R)((float *)sx)[k]; dp1 = ryi - (R)((float *)sy)[k]; dp2 = rzi - (R)((float *)sz)[k];
                } else {
                    dp0 = (R)wrap_near(xi - sx[k], P.box, inv_box);
                    dp1 = (R)wrap_near(yi - sy[k], P.box, inv_box);
                    dp2 = (R)wrap_near(zi - sz[k], P.box, inv_box);
                }
                const R r2 = dp0 * dp0 + dp1 * dp1 + dp2 * dp2;
                const bool ok = got && (std::is_same<R, float>::value || !(mj <= 0)) && !(r2 >= h2);
                const R rr = sqrt(r2);
                const R u = rr * hinv;
                R wk = 0, dwk = 0;
                kernel_main<KERN, 0>(u, hinv3, hinv4, wk, dwk);
                wk = ok ? wk : R(0);
                dwk = ok ? dwk : R(0);
                const R mj_wk = mj * wk;
                a[0] += rounded(wk);
                a[1] += rounded(mj_wk);
                a[2] += rounded(-(R(3.0) * hinv * wk + u * dwk));
                a[4] += rounded(wk * (dp0 * dp0));
                a[5] += rounded(wk * (dp1 * dp1));
                a[6] += rounded(wk * (dp2 * dp2));
                a[7] += rounded(wk * (dp0 * dp1));
                a[8] += rounded(wk * (dp1 * dp2));
                a[9] += rounded(wk * (dp0 * dp2));
                a[10] += rounded(wk * dp0);
                a[11] += rounded(wk * dp1);
                a[12] += rounded(wk * dp2);
                const R dv0 = vxi - svx[k], dv1 = vyi - svy[k], dv2 = vzi - svz[k];
                const R rs = rr > 0 ? rr : R(1);
                const R dwr = rounded(dwk * (dp0 * dv0 + dp1 * dv1 + dp2 * dv2) / rs);
                a[3] -= ok && rr > 0 ? dwr : R(0);
                if constexpr (FD) {  // GradH_numer, GradH_denom (src/hydro/density_loop.h:1281-1286)
                    a[13] += rounded((dwk / rs) * dp0);
                    a[14] += rounded((dwk / rs) * dp1);
                    a[15] += rounded((dwk / rs) * dp2);
                    a[16] += rounded(u * dwk);
                }
            } while (wave_any(win.behind > room));
        }
        __syncthreads();  // before the next rows' candidates take the ring
        if (on)
            for (int k = 0; k < nsum; k++) accout[(size_t)k * cr.nrows + r] = (double)a[k];
    }
}

// the maximum of v over the block into *dst (one conditional atomic per block)
__device__ __forceinline__ void block_max_to(double v, unsigned long long *dst)
{
    __shared__ double wv[16];
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    if ((threadIdx.x & 63) == 0) wv[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < (int)((blockDim.x + 63) >> 6); k++) v = fmax(v, wv[k]);
        if (v > 0) atomic_max_bits(dst, v);
    }
}

// density()'s pre-iteration radius clamp (src/hydro/density_loop.cc:818-838) and the start of
// the iteration: radius of each row, empty bracket, round counters, the largest radius (the
// bits of a positive double order like the double)
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(256) k_density_init(int na, const int *__restrict__ act, double *__restrict__ H, double hclamp,
                                                      double *__restrict__ hcur, double *__restrict__ left, double *__restrict__ right,
                                                      double *__restrict__ cn_cur, int *__restrict__ cn_init, int *__restrict__ iter,
                                                      uint8_t *__restrict__ need, int *__restrict__ counters,
                                                      unsigned long long *__restrict__ hmax, unsigned long long *__restrict__ hfinal,
                                                      BoxTable bt)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < 8) counters[r] = 0;
    if (r == 0) *hfinal = 0;
    double h = 0;
    if (r < na) {
        const int i = act[r];
        if (bt.b) hclamp = 0.99 * bt.b[bt.BOX[i]].max_h;
        h = H[i];
        if ((h < 0) || !isfinite(h) || (h > hclamp)) { h = hclamp; H[i] = h; }
        hcur[r] = h;
        left[r] = 0; right[r] = 0; cn_cur[r] = 0; cn_init[r] = 0; iter[r] = 0;
        need[r] = 1;
    }
    if (!hmax) return;
    block_max_to(h, hmax);
}
#endif

// the maximum of v over the wave into slot (one atomic when the wave holds one box; the bits of
// a positive double order like the double)
__device__ __forceinline__ void wave_max_to(double v, bool valid, int box, unsigned long long *single, const BoxTable &bt, int slot)
{
    if (!bt.b) {
        for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
        if ((threadIdx.x & 63) == 0 && v > 0) atomic_max_bits(single, v);
        return;
    }
    const unsigned long long vm = __ballot(valid);
    if (!vm) return;
    const int b0 = __shfl(box, __ffsll((long long)vm) - 1, 64);
    if (__all(!valid || box == b0)) {
        double w = valid ? v : 0.0;
        for (int o = 32; o > 0; o >>= 1) w = fmax(w, __shfl_xor(w, o, 64));
        if ((threadIdx.x & 63) == 0 && w > 0) atomic_max_bits(&bt.slot[(size_t)b0 * kBoxSlots + slot], w);
    } else if (valid && v > 0) {
        atomic_max_bits(&bt.slot[(size_t)box * kBoxSlots + slot], v);
    }
}

// the sum of the list lengths (the pairs a force pass evaluates): one atomic per block
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(256) k_sum_counts(int nrows, const int *__restrict__ cnt, unsigned long long *__restrict__ out,
                                                    const int *__restrict__ gate)
{
    if (gate && *gate) return;
    __shared__ unsigned long long part[4];
    unsigned long long s = 0;
    for (long r = blockIdx.x * (long)blockDim.x + threadIdx.x; r < nrows; r += (long)gridDim.x * blockDim.x) s += (unsigned long long)cnt[r];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        s = part[0] + part[1] + part[2] + part[3];
        if (s) atomicAdd(out, s);
    }
}

#endif

// after_iter_body (src/hydro/density_loop.h:516-961) on the sums of the round and, on
// convergence, density_finalize_post_runner (src/hydro/density_loop.cc:303-733)
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(256) k_density_after(DevParams P, int nrows, const int *__restrict__ act, uint8_t *__restrict__ need,
                                                       const double *__restrict__ accin, const double *__restrict__ M,
                                                       const double *__restrict__ U, double cell, DensityIter it, DensityOut out,
                                                       int *__restrict__ nnext, int *__restrict__ rebuild, int *__restrict__ err,
                                                       unsigned long long *__restrict__ hfinal, BoxTable bt, double hlim,
                                                       int *__restrict__ gate, unsigned int *__restrict__ done,
                                                       const int *__restrict__ rows, int nlist, int *__restrict__ next_rows)
{
    // every lane reaches the wave-wide counts and maxima at the end.  Lane t takes row t, or the
    // t-th row of the list of rows of this round (rows, nlist); next_rows (may be null) receives
    // the rows that iterate again, in any order (each row's sums do not depend on the others)
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = rows ? (t < nlist ? rows[t] : nrows) : t;
    const bool row = r < nrows && need[r];
    double h_final = 0, h_grow = 0;
    bool cont = false;
    int box = 0;
    if (row) {
        const int i = act[r];
        if (bt.b) {
            GridView g{};
            resolve_box(bt, i, P, g);
            box = bt.BOX[i];
            cell = bt.b[box].rowlim;
        }
        double acc[kDensSumsFD];
        for (int q = 0; q < kDensSums; q++) acc[q] = accin[(size_t)q * nrows + r];
        if (P.fd4alpha > 0)
            for (int q = kDensSums; q < kDensSumsFD; q++) acc[q] = accin[(size_t)q * nrows + r];
        else
            for (int q = kDensSums; q < kDensSumsFD; q++) acc[q] = 0;
        const double h = it.hcur[r];
        IterState sc;
        sc.left = it.left[r]; sc.right = it.right[r]; sc.cn_cur = it.cn_cur[r]; sc.cn_init = it.cn_init[r];
        const int iter = it.iter[r];
        double nh = h;
        DensityNorm dn;
        density_norm(acc, h, dn);
        const int rc = density_after_iter(P, out.cn[i], iter, h, dn, sc, nh);
        it.iter[r] = iter + 1;
        if (rc <= 0 || iter + 1 >= kMaxIter) {
            if (rc < 0) atomicMax(err, 90001009);
            else if (rc > 0) atomicMax(err, 1155);
            density_finalize(P, out, i, h, acc, dn, M[i], U[i]);
            need[r] = 0;
            if (h > 0) h_final = h;
        } else {
            it.left[r] = sc.left; it.right[r] = sc.right; it.cn_cur[r] = sc.cn_cur; it.cn_init[r] = sc.cn_init;
            it.hcur[r] = nh;
            if (nh * (1.0 + 1e-6) > cell) h_grow = nh;
            cont = true;
        }
    }
    // rows still iterating and the grid flag: one atomic per block
    const unsigned long long cm = __ballot(cont), gm = __ballot(h_grow > 0);
    __shared__ int wcont[16], wgrow[16];
    if ((threadIdx.x & 63) == 0) { wcont[threadIdx.x >> 6] = (int)__popcll(cm); wgrow[threadIdx.x >> 6] = gm != 0; }
    if (bt.b) {
        wave_max_to(h_final, row, box, hfinal, bt, kSlotHfinal);
        if (gm) wave_max_to(h_grow, row, box, nullptr, bt, kSlotHgrow);
        __syncthreads();
    } else {
        block_max_to(h_final, hfinal);  // synchronises the block
    }
    __shared__ int wbase[16];
    if (threadIdx.x == 0) {
        int c = 0, g = 0;
        for (int k = 0; k < (int)((blockDim.x + 63) >> 6); k++) { wbase[k] = c; c += wcont[k]; g |= wgrow[k]; }
        if (next_rows) {
            const int base = c ? atomicAdd(nnext, c) : 0;
            for (int k = 0; k < (int)((blockDim.x + 63) >> 6); k++) wbase[k] += base;
        } else if (c) {
            atomicAdd(nnext, c);  // no result: no wait for it
        }
        if (g) atomicOr(rebuild, 1);
        if (gate) {
            // the last block to finish, when every block's counts and maxima are in, writes
            // whether the passes launched behind this round before its counters are read stand:
            // the round's stop code; else -1 while rows still iterate; else -2 when a final
            // radius exceeds hlim, the bound every radius was taken under when the symmetric
            // list's grid was sized; else 0.  The passes' kernels with effects that a second
            // run would not undo (wake-up flags, pair counts) read it and do nothing unless 0.
            __threadfence();
            if (atomicAdd(done, 1u) == gridDim.x - 1) {
                __threadfence();
                const int e = atomicOr(err, 0), nrem = atomicOr(nnext, 0);
                const double hf = __longlong_as_double((long long)atomicOr(hfinal, 0ull));
                *gate = e ? e : (nrem ? -1 : (hf > hlim ? -2 : 0));
                *done = 0u;
            }
        }
    }
    if (next_rows) {
        // the rows that iterate again, each wave's at the place its block reserved
        __syncthreads();
        if (cont) {
            const unsigned long long below = (1ull << (threadIdx.x & 63)) - 1ull;
            next_rows[wbase[threadIdx.x >> 6] + (int)__popcll(cm & below)] = r;
        }
    }
}
#endif



// ---------------------------------------------------------------------------------------
// records: the neighbour-side fields of a pass, packed per particle (device order)
// ---------------------------------------------------------------------------------------
// the gradient record of particle j, from the state (the record a pass packs, or builds where it
// reads it)
template <typename R>
__device__ __forceinline__ GradRec<R> make_grad_rec(long j, const GradSrc &s, const double *__restrict__ X, const double *__restrict__ Y,
                                                    const double *__restrict__ Z, const BoxTable &bt)
{
    GradRec<R> g;
    g.h = (R)s.H[j]; g.m = (R)s.M[j]; g.rho = s.RHO[j]; g.p = s.PR[j];
    g.v0 = s.VX[j]; g.v1 = s.VY[j]; g.v2 = s.VZ[j];
    if constexpr (std::is_same<R, float>::value) g.fp = fine_pos(X[j], Y[j], Z[j], bt.b ? bt.b[bt.BOX[j]].box : s.box);
    return g;
}

// the gradient record of particle j
template <typename R, typename Rec>
__device__ __forceinline__ void pack_grad_one(long j, const GradSrc &s, Rec *__restrict__ rec, const double *__restrict__ X,
                                              const double *__restrict__ Y, const double *__restrict__ Z, const BoxTable &bt)
{
    if constexpr (std::is_same<Rec, GradRec<R>>::value) rec[j] = make_grad_rec<R>(j, s, X, Y, Z, bt);
    else rec[j] = GradPosRec{s.H[j], s.M[j], s.RHO[j], s.PR[j], s.VX[j], s.VY[j], s.VZ[j], X[j], Y[j], Z[j]};
}

// every record (passes over many rows)
template <typename R, typename Rec>
__global__ void k_pack_grad(long n, const double *__restrict__ H, const double *__restrict__ M,
                            const double *__restrict__ RHO, const double *__restrict__ PR, const double *__restrict__ VX,
                            const double *__restrict__ VY, const double *__restrict__ VZ, Rec *__restrict__ rec,
                            const double *__restrict__ X, const double *__restrict__ Y, const double *__restrict__ Z, double box,
                            BoxTable bt)
{
    const long j = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (j >= n) return;
    pack_grad_one<R>(j, GradSrc{H, M, RHO, PR, VX, VY, VZ, box}, rec, X, Y, Z, bt);
}

// the force record of particle j (effective_soundspeed, src/declarations/cell_data.h:703-712)
template <typename R>
__device__ __forceinline__ Cell<R> force_rec_of(long j, double gamma, const ForceView &F, double box, const BoxTable &bt)
{
    const long n = F.n;
    Cell<R> c;
    c.h = F.H[j]; c.m = (R)F.M[j]; c.rho = (R)F.RHO[j]; c.p = (R)F.PR[j];
    c.cn = (R)F.CN[j]; c.fce = (R)F.FCE[j]; c.drk = (R)F.DRK[j];
    c.v0 = (R)F.VX[j]; c.v1 = (R)F.VY[j]; c.v2 = (R)F.VZ[j];
    c.gr0 = (R)F.GR[j]; c.gr1 = (R)F.GR[n + j]; c.gr2 = (R)F.GR[2 * n + j];
    c.gp0 = (R)F.GP[j]; c.gp1 = (R)F.GP[n + j]; c.gp2 = (R)F.GP[2 * n + j];
    for (int k = 0; k < 9; k++) c.gv[k] = (R)F.GV[(size_t)k * n + j];
    for (int k = 0; k < 6; k++) c.t[k] = (R)F.T[(size_t)k * n + j];
    const double rho = F.RHO[j];
    c.cs = (R)((rho > 0) ? sqrt(gamma * F.PR[j] / rho) : sqrt(gamma * (gamma - 1.) * F.U[j]));
    if constexpr (std::is_same<R, float>::value) c.fp = fine_pos(F.X[j], F.Y[j], F.Z[j], bt.b ? bt.b[bt.BOX[j]].box : box);
    return c;
}

template <typename R>
__device__ __forceinline__ void pack_force_one(long j, double gamma, const ForceView &F, Cell<R> *__restrict__ rec, double box,
                                               const BoxTable &bt)
{
    rec[j] = force_rec_of<R>(j, gamma, F, box, bt);
}

// the force pass's error and wake-up flags, the first pair without a Riemann solution and the
// count of rows left to the whole Riemann ladder
__device__ __forceinline__ void force_flags_clear(int *zero2)
{
    zero2[0] = 0; zero2[2] = 0; zero2[10] = -1; zero2[11] = -1; zero2[12] = 0;
}

template <typename R>
__global__ void k_pack_force(double gamma, ForceView F, Cell<R> *__restrict__ rec, int *__restrict__ zero2, double box, BoxTable bt)
{
    const long j = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (j == 0 && zero2) force_flags_clear(zero2);
    if (j >= F.n) return;
    pack_force_one<R>(j, gamma, F, rec, box, bt);
}

// Few rows: the records of the rows and of their list entries only, one wavefront per row
// (a record shared by several rows is written several times with the same bytes)
template <typename R, typename Rec>
__global__ void __launch_bounds__(64) k_pack_grad_list(int nrows, const int *__restrict__ act, const int *__restrict__ ell, long ld,
                                                       const int *__restrict__ cnt, const double *__restrict__ H,
                                                       const double *__restrict__ M, const double *__restrict__ RHO,
                                                       const double *__restrict__ PR, const double *__restrict__ VX,
                                                       const double *__restrict__ VY, const double *__restrict__ VZ,
                                                       Rec *__restrict__ rec, const double *__restrict__ X,
                                                       const double *__restrict__ Y, const double *__restrict__ Z, double box,
                                                       BoxTable bt)
{
    const long r = xcd_block();
    if (r >= nrows) return;
    const int c = cnt[r];
    for (int q = threadIdx.x; q <= c; q += 64) {
        const int j = q == 0 ? act[r] : ell[ell_at(ld, r, q - 1)];
        pack_grad_one<R>(j, GradSrc{H, M, RHO, PR, VX, VY, VZ, box}, rec, X, Y, Z, bt);
    }
}

template <typename R>
__global__ void __launch_bounds__(64) k_pack_force_list(int nrows, const int *__restrict__ act, const int *__restrict__ ell, long ld,
                                                        const int *__restrict__ cnt, double gamma, ForceView F,
                                                        Cell<R> *__restrict__ rec, int *__restrict__ zero2, double box, BoxTable bt)
{
    const long r = xcd_block();
    if (r == 0 && threadIdx.x == 0 && zero2) force_flags_clear(zero2);
    if (r >= nrows) return;
    const int c = cnt[r];
    for (int q = threadIdx.x; q <= c; q += 64) {
        const int j = q == 0 ? act[r] : ell[ell_at(ld, r, q - 1)];
        pack_force_one<R>(j, gamma, F, rec, box, bt);
    }
}

// ---------------------------------------------------------------------------------------
// gradients: gradient_accumulate_neighbor (src/hydro/gradient_functions.h:305-665),
// construct_gradient (src/hydro/gradients_loop.cc:129-136) and the limiter block
// (:1077-1130), fused per active particle
// ---------------------------------------------------------------------------------------
// construct_gradient (NV_T^-1 times the sums) and the limiter block of one particle
template <typename R, typename Rec>
__device__ inline void gradients_tail(const Rec &I, bool enabled, const R (&G)[3][5], const R (&mx)[5], const R (&mn)[5],
                                      R maxd, const double *__restrict__ T, const double *__restrict__ CN, long n, int i,
                                      double *__restrict__ GR, double *__restrict__ GP, double *__restrict__ GV)
{
    const R hi = I.h;
    const R t0 = (R)T[0 * n + i], t1 = (R)T[1 * n + i], t2 = (R)T[2 * n + i], t3 = (R)T[3 * n + i], t4 = (R)T[4 * n + i], t5 = (R)T[5 * n + i];
    R o[5][3];
    for (int b = 0; b < 5; b++) {
        const R v0 = G[0][b], v1 = G[1][b], v2 = G[2][b];
        o[b][0] = t0 * v0 + t3 * v1 + t5 * v2;
        o[b][1] = t3 * v0 + t1 * v1 + t4 * v2;
        o[b][2] = t5 * v0 + t4 * v1 + t2 * v2;
    }
    if (enabled) {
        const R stol = R(0.1);
        const R dmaxv = dmax(hi, maxd);
        const double cni = CN[i];
        R alim = R(0.25);
        if (cni > 100) alim = (R)dmin(0.5, 0.25 + 0.25 * (cni - 100) / 100);
        slopelimiter<R>(o[0], mx[0], mn[0], alim, hi, R(0), 1, dmaxv, (R)I.rho);
        slopelimiter<R>(o[1], mx[1], mn[1], alim, hi, stol, 1, dmaxv, (R)I.p);
        for (int kk = 0; kk < 3; kk++) slopelimiter<R>(o[2 + kk], mx[2 + kk], mn[2 + kk], alim, hi, stol, 0, R(0), R(0));
    }
    for (int kk = 0; kk < 3; kk++) {
        GR[(size_t)kk * n + i] = (double)o[0][kk];
        GP[(size_t)kk * n + i] = (double)o[1][kk];
        for (int b = 0; b < 3; b++) GV[(size_t)(3 * b + kk) * n + i] = (double)o[2 + b][kk];
    }
}

// 16 bytes from src to LDS at lds + 16 x lane; complete after wait_staged
__device__ __forceinline__ void lds_load16(const char *src, unsigned char *lds)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}
__device__ __forceinline__ void wait_staged() { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// One lane per row, an entry of each row's list at a time.  A lane that reads its own partner's record
// touches a cache line per lane with each of its seven loads; instead the wavefront loads the 64
// records piece by piece (16 bytes a lane, so a record is one line for its four or five
// lanes) straight into LDS, those of the next entry while this one is added.  2M rows FP64 1.86 -> 1.13 ms, FP32 1.68
// -> 1.07.  Rows sorted by list length, over 2048 rows as the force pass has them or over the workgroup's
// 256: 1.74 and 1.13 ms, 4M lognormal rows 4.48 and 3.65 against 3.85, so they stay in order.
template <int KERN, typename R, bool BOXES>
__global__ void __launch_bounds__(256, 4) k_gradients(DevParams P, int nrows, const int *__restrict__ act, const double *__restrict__ H,
                                                   const GradLaneRec<R> *__restrict__ rec, const double *__restrict__ T,
                                                   const double *__restrict__ CN, long n, const int *__restrict__ ell, long ld,
                                                   const int *__restrict__ cnt, double *__restrict__ GR, double *__restrict__ GP,
                                                   double *__restrict__ GV, BoxTable bt)
{
    using Rec = GradLaneRec<R>;
    constexpr int kPieces = (int)sizeof(Rec) / 16;
    static_assert(sizeof(Rec) % 16 == 0, "whole pieces");
    __shared__ __align__(16) unsigned char staged[4][2][64 * sizeof(Rec)];
    const int lane = threadIdx.x & 63;
    const int r = (int)(xcd_block() * blockDim.x + threadIdx.x);
    const bool row = r < nrows;
    const int i = row ? act[r] : 0;
    if (BOXES && row) {
        GridView g{};
        resolve_box(bt, i, P, g);
    }
    R G[3][5];
    for (int a = 0; a < 3; a++) for (int b = 0; b < 5; b++) G[a][b] = 0;
    R mx[5], mn[5];
    for (int b = 0; b < 5; b++) { mx[b] = 0; mn[b] = 0; }
    R maxd = 0;
    const Rec I = rec[i];
    const bool enabled = row && I.m > 0 && I.rho > 0;
    const R hi = I.h;
    // the row's radius in FP64 (the kernel's edge factor, pair_kernel)
    const double hid = std::is_same<R, double>::value ? (double)hi : H[i];
    const double h2i = hid * hid;
    const double inv_box = 1.0 / P.box;
    const int c = enabled ? cnt[r] : 0;
    int cmax = c;
    for (int o = 32; o > 0; o >>= 1) cmax = max(cmax, __shfl_xor(cmax, o, 64));
    unsigned char *const area = staged[threadIdx.x >> 6][0];
    // the records of the lanes' j (a lane without an entry: any record) into area + at
    auto stage = [&](int j, int at) {
        // the reads of the area's last contents are done
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int k = 0; k < kPieces; k++) {
            const int piece = k * 64 + lane, owner = piece / kPieces;
            const int jo = __shfl(j, owner, 64);
            lds_load16((const char *)rec + (size_t)(unsigned)jo * sizeof(Rec) + (piece - owner * kPieces) * 16, area + at + k * 1024);
        }
    };
    int jn = 0;
    if (cmax > 0) {
        stage(c > 0 ? ell[ell_at(ld, r, 0)] : i, 0);
        jn = c > 1 ? ell[ell_at(ld, r, 1)] : i;
    }
    for (int q = 0; q < cmax; q++) {
        const int at = (q & 1) * 64 * (int)sizeof(Rec);
        wait_staged();
        if (q + 1 < cmax) {
            stage(jn, 64 * (int)sizeof(Rec) - at);
            jn = q + 2 < c ? ell[ell_at(ld, r, q + 2)] : i;
        }
        const Rec &J = *(const Rec *)(area + at + lane * (int)sizeof(Rec));
        if (q >= c || !(J.m > 0) || !(J.rho > 0) || !(J.h > 0)) continue;
        R dp[3];
        if constexpr (std::is_same<R, float>::value) {
            fine_dp(I.fp, J.fp, (float)(P.box * (1.0 / 1024.0)), dp[0], dp[1], dp[2]);
        } else {
            dp[0] = wrap_near(I.x - J.x, P.box, inv_box);
            dp[1] = wrap_near(I.y - J.y, P.box, inv_box);
            dp[2] = wrap_near(I.z - J.z, P.box, inv_box);
        }
        const R r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
        if (r2 <= 0) continue;
        const double r2d = pair_r2d<R>(dp[0], dp[1], dp[2], r2);
        if ((r2d >= h2i) && (r2d >= (double)J.h * (double)J.h)) continue;
        const R rr = sqrt(r2);
        const double rd = std::is_same<R, double>::value ? 0.0 : sqrt(r2d);
        const bool inside = std::is_same<R, double>::value ? (rr < hi) : (rd < hid);
        R wk = 0, dwk = 0;
        pair_kernel<KERN, -1, R>(rr, rd, hid, wk, dwk);
        if (rr > maxd) maxd = rr;
        R d[5];
        d[0] = (R)(J.rho - I.rho);
        d[1] = (R)(J.p - I.p);
        d[2] = (R)(J.v0 - I.v0);
        d[3] = (R)(J.v1 - I.v1);
        d[4] = (R)(J.v2 - I.v2);
        for (int b = 0; b < 5; b++) {
            if (d[b] < mn[b]) mn[b] = d[b];
            else if (d[b] > mx[b]) mx[b] = d[b];
        }
        if (inside) {
            for (int kk = 0; kk < 3; kk++) {
                const R w = -wk * dp[kk];
                for (int b = 0; b < 5; b++) G[kk][b] += rounded(w * d[b]);
            }
        }
    }
    if (row) gradients_tail<R>(I, enabled, G, mx, mn, maxd, T, CN, n, i, GR, GP, GV);
}

// Running sum of a conserved flux total.  FP32: Neumaier-compensated (the lost low bits of each
// addition are kept in c, so sums that cancel to a small net keep their accuracy); FP64: the
// plain sum in list order (the oracle's additions).
template <typename R>
struct CSum {
    R s = 0, c = 0;
    __device__ __forceinline__ void add(R x)
    {
        const R t = s + x;
        c += (fabs(s) >= fabs(x)) ? ((s - t) + x) : ((x - t) + s);
        s = t;
    }
    __device__ __forceinline__ double value() const { return (double)s + (double)c; }
};
template <>
struct CSum<double> {
    double s = 0;
    __device__ __forceinline__ void add(double x) { s += x; }
    __device__ __forceinline__ double value() const { return s; }
};

// x_i - x_j of a pair of records: FP32 form from the records' fine cells and offsets (no FP64
// position reads); FP64 form the wrapped FP64 difference of the positions
template <typename R, typename Rec>
__device__ __forceinline__ void record_dp(const DevParams &P, const Rec &I, const Rec &J, double xi, double yi, double zi,
                                          const double *__restrict__ X, const double *__restrict__ Y,
                                          const double *__restrict__ Z, int j, R &dp0, R &dp1, R &dp2)
{
    if constexpr (std::is_same<R, float>::value) {
        fine_dp(I.fp, J.fp, (float)(P.box * (1.0 / 1024.0)), dp0, dp1, dp2);
    } else {
        double d0 = xi - X[j], d1 = yi - Y[j], d2 = zi - Z[j];
        d1 = wrap(d1, P.box, P.half);
        d0 = wrap(d0, P.box, P.half);
        d2 = wrap(d2, P.box, P.half);
        dp0 = (R)d0; dp1 = (R)d1; dp2 = (R)d2;
    }
}

// ---------------------------------------------------------------------------------------
// force: the pair loop of hydro_force() (src/hydro/hydro_force_loop.cc:423-480), two-sided
// (each active particle accumulates its own side of every pair), then the writeback
// (:227-321) and hydro_final_operations_and_cleanup (src/hydro/hydro_toplevel.cc:133-250).
// ---------------------------------------------------------------------------------------
// the writeback (src/hydro/hydro_force_loop.cc:302-321) and hydro_final_operations_and_cleanup
// (src/hydro/hydro_toplevel.cc:133-250, non-comoving MFM) of one particle
__device__ inline void force_tail(const DevParams &P, const ForceView &F, int i, bool enabled, double sound_i, double A0, double A1,
                                  double A2, double dE, double msv, double *__restrict__ ACC, double *__restrict__ DTU,
                                  double *__restrict__ MSV)
{
    const long n = F.n;
    const double mi = F.M[i];
    // MaxSignalVel = max(accumulated, c_s) over MIN_REAL_NUMBER (hydro_force_loop.cc:318-321)
    double ms = kMinReal;
    double mxs = fmax(msv, sound_i);
    if (ms < mxs) ms = mxs;
    double e = dE;
    if (enabled) {
        const double inv1 = 1.0 / 1.0;
        const double vp0 = F.VX[i] * inv1, vp1 = F.VY[i] * inv1, vp2 = F.VZ[i] * inv1;
        e -= vp0 * A0 + vp1 * A1 + vp2 * A2;
        const double invm = 1.0 / mi;
        A0 *= invm; A1 *= invm; A2 *= invm;
        e /= mi;
        if (F.H[i] >= 0.99 * P.max_kernel_radius) e = 0;
    }
    ACC[i] = A0; ACC[n + i] = A1; ACC[2 * n + i] = A2;
    DTU[i] = e;
    MSV[i] = ms;
}

// The records of the lanes' partners into LDS: the four lanes of a quad load one record after the
// other, 16 bytes per lane and instruction, straight into LDS (a lane loading its own record
// would touch one cache line per lane and instruction).  Every lane of the wavefront calls it;
// want: the lane's j is to be loaded.  The caller waits for the loads (wait_staged) before it
// reads them, and has read what it needs of the area's last contents.
template <typename R, int K>
__device__ __forceinline__ void stage_quad_row(const Cell<R> *__restrict__ rec, int j, int want, unsigned char *wave_lds)
{
    using S = StagedRec<R>;
    const int jk = __builtin_amdgcn_mov_dpp(j, K * 0x55, 0xf, 0xf, true);  // lane K of the quad
    const int wk = __builtin_amdgcn_mov_dpp(want, K * 0x55, 0xf, 0xf, true);
    const char *src = (const char *)(rec + jk) + (threadIdx.x & 3) * 16;
    if (wk) {
#pragma unroll
        for (int b = 0; b < S::kBlocks; b++) lds_load16(src + b * 64, wave_lds + K * S::kQuadRow + b * S::kBlock);
    }
}
// the half blocks of the quad's rows 2 K (lanes 0 and 1) and 2 K + 1 (lanes 2 and 3)
template <typename R, int K>
__device__ __forceinline__ void stage_quad_half(const Cell<R> *__restrict__ rec, int j, int want, unsigned char *wave_lds)
{
    using S = StagedRec<R>;
    constexpr int perm = 2 * K | (2 * K) << 2 | (2 * K + 1) << 4 | (2 * K + 1) << 6;
    const int jk = __builtin_amdgcn_mov_dpp(j, perm, 0xf, 0xf, true);
    const int wk = __builtin_amdgcn_mov_dpp(want, perm, 0xf, 0xf, true);
    if (wk) lds_load16((const char *)(rec + jk) + S::kBlocks * 64 + (threadIdx.x & 1) * 16, wave_lds + S::kHalfAt + K * S::kBlock);
}
template <typename R>
__device__ __forceinline__ void stage_records(const Cell<R> *__restrict__ rec, int j, bool want, unsigned char *wave_lds)
{
    // reads and writes of the area's last contents are done
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    stage_quad_row<R, 0>(rec, j, want, wave_lds);
    stage_quad_row<R, 1>(rec, j, want, wave_lds);
    stage_quad_row<R, 2>(rec, j, want, wave_lds);
    stage_quad_row<R, 3>(rec, j, want, wave_lds);
    if constexpr (StagedRec<R>::kHalf) {
        stage_quad_half<R, 0>(rec, j, want, wave_lds);
        stage_quad_half<R, 1>(rec, j, want, wave_lds);
    }
}

// the difference of a pair's positions from the staged record of j (FP32 form) or the position
// arrays (FP64 form)
template <typename R>
__device__ __forceinline__ void staged_dp(const DevParams &P, const Cell<R> &I, const StagedCell<R> &J, double xi, double yi, double zi,
                                          double xj, double yj, double zj, R &dp0, R &dp1, R &dp2)
{
    if constexpr (std::is_same<R, float>::value) {
        fine_dp(I.fp, J.fp(), (float)(P.box * (1.0 / 1024.0)), dp0, dp1, dp2);
    } else {
        const double inv_box = 1.0 / P.box;
        dp0 = wrap_near(xi - xj, P.box, inv_box);
        dp1 = wrap_near(yi - yj, P.box, inv_box);
        dp2 = wrap_near(zi - zj, P.box, inv_box);
    }
}

// What a pair's fluxes leave besides the sums: a failed solve, and the wake-up of an inactive
// neighbour (rc, vts: force_pair's)
template <bool BOXES, typename R>
__device__ __forceinline__ void pair_flags(const ForceRows &a, const BoxTable &bt, int i, int j, int rc, R vts)
{
    if (rc < 0) {
        atomicMax(a.err, 1234);
        if (atomicCAS(a.err + 10, -1, i) == -1) a.err[11] = j;
    }
    if (rc == 1 && a.active && !a.active[j] && a.wakeup) {
        if ((double)vts > kWakeup * a.msv_in[j]) {
            atomicMax(&a.wakeup[j], (a.timebin ? a.timebin[i] : 0) + 1);
            if (BOXES) bt.b[bt.BOX[i]].need_wakeup = 1;
            else *a.need_wakeup = 1;
        }
    }
}

// The force pass over many rows: four lanes (a quad) per row, 64 rows per workgroup, the quad's
// lanes on four consecutive list entries at a time.  A fixed number of workgroups (kForceBlocks)
// walks the rows, each XCD through its own contiguous part, so that the rows in flight on an XCD
// are consecutive and few (4096) and their partners' records (2.6 MB FP64) stay in its L2; one
// lane per row had 16K rows in flight, whose records (7 MB) did not.
//
// The fluxes are added in list order: the quad's four entries go through LDS, and lane t of the
// quad keeps sum t (momentum, energy) and adds the four in turn.  A face past the Riemann ladder's
// common case (riemann_common; one in 14 to 300 on moving gas, but nearly every row has some) is
// not taken where it comes up, where it would hold the other 63 lanes through the exact solver:
// it goes to the workgroup's queue, and from there on its row's fluxes go to the workgroup's part
// of `flux` instead of the sums.  After a segment of every row's list the queued faces are
// taken together, 256 at a time, with the whole ladder, and the rows that wait for them add the
// stored fluxes in list order.  Each row's sums are those of one loop over its list, bit for bit.
// STATS: the faces' RiemannRung bits are counted.
//
// 2M rows of a box at Mach 0.3 (7% of the faces past the common case, 97% of the rows): FP64 22.7
// -> 11.4 ms, FP32 12.3 -> 8.5 ms; 1M rows of a lognormal field (0.3% of the faces) FP64 10.4 ->
// 5.4 ms; 15,625 rows FP32 1,120 -> 130 us (one lane per row left most of the chip idle).  The two
// kernels before took a row again from its start at its first such face.  Waiting lanes in one
// lane per row's loop (until 8, 24, 40 of 64 waited) took 18.9, 24.9, 36.9 ms: rows with many such
// faces hold their wavefront.  Two wavefronts per SIMD: the record of the row and the whole
// ladder take 256 registers (FP32 at three: spills, 10.8 ms).  Bound now by its VALU instructions
// (half of the time) and the wait for the records between them.
template <int KERN, typename R, bool BOXES, bool STATS>
__global__ void __launch_bounds__(256, 2)
    k_force(DevParams P0, Gam<R> G, ForceView F, const Cell<R> *__restrict__ rec, ForceRows a, BoxTable bt)
{
    using S = StagedRec<R>;
    __shared__ __align__(16) unsigned char staged[4][S::kWave];
    __shared__ unsigned short queue[kForceRowsPerBlock * kForceSegment];  // (list entry in the segment) * rows + row
    __shared__ unsigned long long mrow[kForceRowsPerBlock];               // signal speeds of the queued faces (bits)
    __shared__ int nqueue, cwave[2][4];  // (two: a wavefront may be one row block ahead)
    const int tid = threadIdx.x, lane = tid & 63, t = tid & 3;
    unsigned char *wave_lds = staged[tid >> 6];
    const StagedCell<R> J(wave_lds + S::lane_at(lane), wave_lds + S::half_at(lane));
    R(*flux)[kForceRowsPerBlock][4] = (R(*)[kForceRowsPerBlock][4])a.flux + (size_t)blockIdx.x * a.segment;
    // the row blocks of this workgroup: one of every (grid / 8) of its XCD's contiguous eighth, its
    // place among them shifted each turn (the row order repeats from long lists to short ones)
    const int nrows = std::is_same<R, float>::value && a.nrows_dev ? *a.nrows_dev : a.nrows;
    const int nrb = (nrows + kForceRowsPerBlock - 1) / kForceRowsPerBlock;
    const int per = (nrb + kXcds - 1) / kXcds, xcd = blockIdx.x % kXcds, nx = gridDim.x / kXcds;
    int rare_rows = 0;
    if (tid == 0) nqueue = 0;
    for (int b0 = 0, place = blockIdx.x / kXcds, turn = 0; b0 < per; b0 += nx, turn ^= 1) {
        const int b = b0 + place, rb = xcd * per + b;
        place += 13;
        while (place >= nx) place -= nx;
        if (b >= per || rb >= nrb) continue;
        const int k = rb * kForceRowsPerBlock + (tid >> 2);
        const bool row = k < nrows;
        const int r = row ? (a.sched ? a.sched[k] : k) : 0;
        const int i = row ? a.act[r] : 0;
        DevParams P = P0;
        if (BOXES && row) {
            GridView g{};
            resolve_box(bt, i, P, g);
        }
        // hydro_force_initial_operations_preloop (src/hydro/hydro_toplevel.cc:457-565): an active
        // particle's own flag is cleared; only inactive neighbours are flagged below
        if (row && t == 0 && a.wakeup) a.wakeup[i] = 0;
        const double mi = row ? F.M[i] : 0, rhoi = row ? F.RHO[i] : 0;
        const bool enabled = row && mi > 0 && rhoi > 0;
        const int c = enabled ? a.cnt[r] : 0;
        {
            int cm = c;
            for (int o = 32; o >= 4; o >>= 1) cm = max(cm, __shfl_xor(cm, o, 64));
            if (lane == 0) cwave[turn][tid >> 6] = cm;
        }
        if (t == 0) mrow[tid >> 2] = 0;
        __syncthreads();
        const int cmax = max(max(cwave[turn][0], cwave[turn][1]), max(cwave[turn][2], cwave[turn][3]));
        CSum<R> sum;
        R m = 0;
        bool had_rare = false;
        for (int seg = 0; seg < cmax; seg += a.segment) {
            const int cs = min(c - seg, a.segment);  // this row's entries of the segment
            int first_rare = -1;                         // the first queued entry of the row
            {
                const Cell<R> I = rec[i];
                const double xi = F.X[i], yi = F.Y[i], zi = F.Z[i];
                if (cs > 0 && m < I.cs) m = I.cs;
                int jn = t < cs ? a.ell[ell_at(a.ld, r, seg + t)] : 0;
                for (int q0 = 0; __any(q0 < cs); q0 += 4) {
                    const int q = q0 + t, j = jn;
                    const bool go = q < cs;
                    stage_records<R>(rec, j, go, wave_lds);
                    double xj = 0, yj = 0, zj = 0;
                    if (go) {
                        if constexpr (std::is_same<R, double>::value) { xj = F.X[j]; yj = F.Y[j]; zj = F.Z[j]; }
                        if (q + 4 < cs) jn = a.ell[ell_at(a.ld, r, seg + q + 4)];
                    }
                    wait_staged();
                    int rc = 0;
                    R f0 = 0, f1 = 0, f2 = 0, fp = 0;
                    if (go) {
                        R dp0, dp1, dp2, vts;
                        unsigned rung;
                        staged_dp<R>(P, I, J, xi, yi, zi, xj, yj, zj, dp0, dp1, dp2);
                        rc = force_pair<KERN, R, true>(P, G, I, J, dp0, dp1, dp2, dp0 * dp0 + dp1 * dp1 + dp2 * dp2, f0, f1, f2, fp, vts, rung);
                        if constexpr (STATS) {
                            if (rc != 2) count_rungs(F.rungs, rung);
                        }
                        if (rc == 1 && vts > m) m = vts;
                        pair_flags<BOXES>(a, bt, i, j, rc, vts);
                    }
                    // faces of this round that wait; the quad's first one closes its row
                    const unsigned long long waits = __ballot(rc == 2);
                    if (waits) {
                        int base = 0;
                        const int lead = __ffsll((long long)waits) - 1;
                        if (lane == lead) base = atomicAdd(&nqueue, (int)__popcll(waits));
                        base = __shfl(base, lead, 64);
                        if (rc == 2) queue[base + __popcll(waits & ((1ull << lane) - 1ull))] = (unsigned short)(q * kForceRowsPerBlock + (tid >> 2));
                        const unsigned mine = (unsigned)(waits >> (lane & ~3)) & 15u;
                        if (first_rare < 0 && mine) first_rare = q0 + __ffs((int)mine) - 1;
                    }
                    const bool open = first_rare < 0 || q < first_rare;
                    if (go && !open && rc != 2) {
                        R *w = flux[q][tid >> 2];
                        w[0] = rounded(f0); w[1] = rounded(f1); w[2] = rounded(f2); w[3] = rounded(fp);
                    }
                    // lane t adds component t of the quad's entries, in order (an entry that is not
                    // added here counts as zeros, which leave a sum as it is)
                    R *w = (R *)(wave_lds + (lane >> 2) * (16 * (int)sizeof(R) + 16)) + 4 * t;
                    const bool add = rc == 1 && open;
                    w[0] = add ? rounded(f0) : R(0); w[1] = add ? rounded(f1) : R(0);
                    w[2] = add ? rounded(f2) : R(0); w[3] = add ? rounded(fp) : R(0);
                    __builtin_amdgcn_wave_barrier();
                    const R *v = (const R *)(wave_lds + (lane >> 2) * (16 * (int)sizeof(R) + 16)) + t;
                    const R x0 = v[0], x1 = v[4], x2 = v[8], x3 = v[12];
                    __builtin_amdgcn_wave_barrier();
                    sum.add(x0); sum.add(x1); sum.add(x2); sum.add(x3);
                }
            }
            __syncthreads();  // the queue and the stored fluxes are written
            const int nq = nqueue;
            __syncthreads();  // before a wavefront goes on to queue the next segment's faces
            if (nq) {
                // the queued faces with the whole ladder
                for (int e0 = 0; e0 < nq; e0 += 256) {
                    const bool go = e0 + tid < nq;
                    const int e = go ? queue[e0 + tid] : 0, er = e % kForceRowsPerBlock, q = e / kForceRowsPerBlock;
                    const int ek = min(rb * kForceRowsPerBlock + er, nrows - 1);
                    const int rr = a.sched ? a.sched[ek] : ek, ii = a.act[rr];
                    const int j = go ? a.ell[ell_at(a.ld, rr, seg + q)] : 0;
                    stage_records<R>(rec, j, go, wave_lds);
                    if (!__any(go)) break;
                    const Cell<R> I = rec[ii];
                    wait_staged();
                    if (go) {
                        DevParams Q = P0;
                        if (BOXES) {
                            GridView g{};
                            resolve_box(bt, ii, Q, g);
                        }
                        R dp0, dp1, dp2, f0, f1, f2, fp, vts;
                        unsigned rung;
                        double xi = 0, yi = 0, zi = 0, xj = 0, yj = 0, zj = 0;
                        if constexpr (std::is_same<R, double>::value) {
                            xi = F.X[ii]; yi = F.Y[ii]; zi = F.Z[ii];
                            xj = F.X[j]; yj = F.Y[j]; zj = F.Z[j];
                        }
                        staged_dp<R>(Q, I, J, xi, yi, zi, xj, yj, zj, dp0, dp1, dp2);
                        const int rc = force_pair<KERN, R, false>(Q, G, I, J, dp0, dp1, dp2, dp0 * dp0 + dp1 * dp1 + dp2 * dp2, f0, f1, f2, fp, vts, rung);
                        if constexpr (STATS) count_rungs(F.rungs, rung);
                        const bool add = rc == 1;
                        R *w = flux[q][er];
                        w[0] = add ? rounded(f0) : R(0); w[1] = add ? rounded(f1) : R(0);
                        w[2] = add ? rounded(f2) : R(0); w[3] = add ? rounded(fp) : R(0);
                        if (add && vts > 0) atomicMax(&mrow[er], (unsigned long long)__double_as_longlong((double)vts));
                        pair_flags<BOXES>(a, bt, ii, j, rc, vts);
                    }
                }
                __syncthreads();
                if (tid == 0) nqueue = 0;
                // the rows that waited: the rest of the segment in list order
                if (first_rare >= 0) {
                    had_rare = true;
                    const R *f = &flux[0][tid >> 2][t];
                    int q = first_rare;
                    for (; q + 4 <= cs; q += 4) {
                        const R x0 = f[(size_t)q * 4 * kForceRowsPerBlock], x1 = f[(size_t)(q + 1) * 4 * kForceRowsPerBlock],
                                x2 = f[(size_t)(q + 2) * 4 * kForceRowsPerBlock], x3 = f[(size_t)(q + 3) * 4 * kForceRowsPerBlock];
                        sum.add(x0); sum.add(x1); sum.add(x2); sum.add(x3);
                    }
                    for (; q < cs; q++) sum.add(f[(size_t)q * 4 * kForceRowsPerBlock]);
                }
                __syncthreads();  // the next segment's entries take the queue and the flux rows
            }
        }
        // lane 0 of the quad closes the row: the quad's sums and its largest signal speed
        const double v = sum.value();
        const int l0 = lane & ~3;
        const double A0 = __shfl(v, l0, 64), A1 = __shfl(v, l0 + 1, 64), A2 = __shfl(v, l0 + 2, 64), dE = __shfl(v, l0 + 3, 64);
        m = dmax(m, __shfl_xor(m, 1, 64));
        m = dmax(m, __shfl_xor(m, 2, 64));
        if (row && t == 0) {
            const double mq = __longlong_as_double((long long)mrow[tid >> 2]);
            // effective_soundspeed of i, src/declarations/cell_data.h:703-712 (floor of MaxSignalVel)
            const double sound_i = (rhoi > 0) ? sqrt(P.gamma * F.PR[i] / rhoi) : sqrt(P.gamma * (P.gamma - 1.) * F.U[i]);
            force_tail(P, F, i, enabled, sound_i, A0, A1, A2, dE, dmax((double)m, mq), a.ACC, a.DTU, a.MSV);
            rare_rows += had_rare;
        }
    }
    // rows with a face past the common case (one atomic per wavefront of the fixed grid)
    if (a.count_rare) {
        for (int o = 32; o > 0; o >>= 1) rare_rows += __shfl_xor(rare_rows, o, 64);
        if (lane == 0 && rare_rows) atomicAdd(a.err + 12, rare_rows);
    }
}

// The same pass over many rows of quiet gas in the FP32 form (force_by_lanes): one lane per row through the
// Riemann ladder's common case alone, which takes a third of the whole ladder's registers (four
// wavefronts per SIMD hide the loads of the records where k_force's two wait for them).  A row with a face
// past that case is listed for k_force, and nothing of it is written but its neighbours' wake-up
// flags, which k_force sets again to the same values.  Each row's sums are k_force's, bit for bit.
// 2M rows at rest or nearly so 5.5 -> 3.4 ms.  Bound by its VALU instructions (0.19 of an issue rate of 0.25;
// the quads' 0.16), with 8.3 GB from beyond the L2 (a lane reads its own partner's record, 16K rows in flight on an XCD).
template <int KERN, bool BOXES>
__global__ void __launch_bounds__(256) k_force_lanes(DevParams P0, Gam<float> G, ForceView F, const Cell<float> *__restrict__ rec,
                                                     ForceRows a, BoxTable bt)
{
    const int k = (int)(xcd_block() * blockDim.x + threadIdx.x);
    const bool row = k < a.nrows;
    const int r = row ? (a.sched ? a.sched[k] : k) : 0;
    bool rare = false;
    if (row) {
        DevParams P = P0;
        const int i = a.act[r];
        if (BOXES) {
            GridView g{};
            resolve_box(bt, i, P, g);
        }
        if (a.wakeup) a.wakeup[i] = 0;  // (as k_force)
        const double mi = F.M[i], rhoi = F.RHO[i];
        // effective_soundspeed of i, src/declarations/cell_data.h:703-712 (floor of MaxSignalVel)
        const double sound_i = (rhoi > 0) ? sqrt(P.gamma * F.PR[i] / rhoi) : sqrt(P.gamma * (P.gamma - 1.) * F.U[i]);
        const bool enabled = mi > 0 && rhoi > 0;
        CSum<float> a0, a1, a2, ae;
        float m = 0;
        const int c = enabled ? a.cnt[r] : 0;
        if (c > 0) {
            const Cell<float> I = rec[i];
            if (m < I.cs) m = I.cs;
            for (int q = 0; q < c; q++) {
                const int j = a.ell[ell_at(a.ld, r, q)];
                const Cell<float> J = rec[j];
                float dp0, dp1, dp2, f0, f1, f2, fp, vts;
                fine_dp(I.fp, J.fp, (float)(P.box * (1.0 / 1024.0)), dp0, dp1, dp2);
                unsigned rung;
                const int rc = force_pair<KERN, float, true>(P, G, I, J, dp0, dp1, dp2, dp0 * dp0 + dp1 * dp1 + dp2 * dp2, f0, f1, f2, fp, vts, rung);
                if (rc == 2) {
                    rare = true;
                    break;
                }
                if (rc == 1) {
                    a0.add(rounded(f0)); a1.add(rounded(f1)); a2.add(rounded(f2)); ae.add(rounded(fp));
                    if (vts > m) m = vts;
                }
                pair_flags<BOXES>(a, bt, i, j, rc, vts);
            }
        }
        if (!rare) force_tail(P, F, i, enabled, sound_i, a0.value(), a1.value(), a2.value(), ae.value(), (double)m, a.ACC, a.DTU, a.MSV);
    }
    // a wavefront's listed rows together and in lane order, by one atomic
    const unsigned long long left = __ballot(rare);
    if (!left) return;
    const int lane = threadIdx.x & 63, lead = __ffsll((long long)left) - 1;
    int base = 0;
    if (lane == lead) base = atomicAdd(a.err + 12, (int)__popcll(left));
    base = __shfl(base, lead, 64);
    if (rare) a.rare[base + __popcll(left & ((1ull << lane) - 1ull))] = r;
}

// ---------------------------------------------------------------------------------------
// The Riemann functions on given face states, one lane per case (a diagnostic with no
// counterpart in the reference; the force pass reaches the same functions through the pair
// body).  Case k reads kProbeIn values from in + k*kProbeIn: the left state (rho, p, v[3]), the
// right state, the face normal n[3], the pressure limiter, then the first-order states the
// ladder retries with (p_i, p_j, rho_i, rho_j, v_i[3], v_j[3]); it writes P_M, S_M, the momentum
// flux[3], the energy flux and 1 (0: the ladder found no positive pressure) to
// out + k*kProbeOut, and the RiemannRung bits taken to rung[k].  Modes: 0 the ladder of the pair
// body with its two retries (hydro_core_meshless_functions.h:351-427), 1 Riemann_solver
// (reimann.h:282-370), 2 get_wavespeeds_and_pressure_star alone (:485-549), 3
// Riemann_solver_KurganovTadmor_PWK alone (:445-477), 4 Riemann_solver_exact alone (:625-668).
// ---------------------------------------------------------------------------------------
template <typename R>
__global__ void __launch_bounds__(256) k_riemann_probe(int mode, Gam<R> G, long n, const double *__restrict__ in,
                                                       double *__restrict__ out, unsigned *__restrict__ rung)
{
    const long k = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double *c = in + k * kProbeIn;
    RState<R> L, Rs;
    L.rho = (R)c[0]; L.p = (R)c[1]; L.v0 = (R)c[2]; L.v1 = (R)c[3]; L.v2 = (R)c[4];
    Rs.rho = (R)c[5]; Rs.p = (R)c[6]; Rs.v0 = (R)c[7]; Rs.v1 = (R)c[8]; Rs.v2 = (R)c[9];
    const R nv[3] = {(R)c[10], (R)c[11], (R)c[12]};
    const R ptl = (R)c[13];
    ROut<R> o;
    o.P_M = o.S_M = o.f0 = o.f1 = o.f2 = o.fp = 0;
    unsigned rb = 0;
    bool ok = true;
    if (mode == 0) {
        ok = riemann_ladder<R>(G, L, Rs, nv, ptl, (R)c[14], (R)c[15], (R)c[16], (R)c[17], (R)c[18], (R)c[19], (R)c[20], (R)c[21],
                               (R)c[22], (R)c[23], o, rb);
    } else if (mode == 1) {
        rb = riemann(G, L, Rs, nv, ptl, o);
    } else {
        const RPrep<R> q = riemann_prep(G, L, Rs, nv);
        if (mode == 2) rb = wavespeeds(G, L, Rs, nv, q.vL, q.vR, q.csL, q.csR, q.hL, q.hR, o, ptl);
        else if (mode == 3) { kt_flux(L, Rs, nv, q.vL, q.vR, q.csL, q.csR, q.hL, q.hR, o); rb = kRungKt; }
        else rb = exact_riemann(G, L, Rs, q.vL, q.vR, q.csL, q.csR, o);
    }
    double *w = out + k * kProbeOut;
    w[0] = (double)o.P_M; w[1] = (double)o.S_M; w[2] = (double)o.f0; w[3] = (double)o.f1; w[4] = (double)o.f2; w[5] = (double)o.fp;
    w[6] = ok ? 1.0 : 0.0;
    w[7] = 0.0;
    rung[k] = rb;
}

#ifdef GZ_DEFINE_COMMON_KERNELS
// per block of 1024 rows: the sum of the list lengths and the sum of each wave's longest
__global__ void __launch_bounds__(1024) k_sched_stats(int nrows, const int *__restrict__ cnt, unsigned long long *__restrict__ partial)
{
    __shared__ unsigned long long ss[16], sm[16];
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    int c = r < nrows ? cnt[r] : 0;
    int mx = c;
    unsigned long long sum = (unsigned long long)c;
    for (int o = 32; o > 0; o >>= 1) {
        mx = max(mx, __shfl_xor(mx, o, 64));
        sum += __shfl_xor(sum, o, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { ss[w] = sum; sm[w] = (unsigned long long)mx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long a = 0, b = 0;
        for (int k = 0; k < (int)(blockDim.x >> 6); k++) { a += ss[k]; b += sm[k]; }
        partial[2 * blockIdx.x] = a;
        partial[2 * blockIdx.x + 1] = b;
    }
}

// the totals of the partial sums, and how even the waves of the plain order are (in millionths; one block)
__global__ void __launch_bounds__(1024) k_sched_total(int nparts, const unsigned long long *__restrict__ partial,
                                                      unsigned long long *__restrict__ total, int *__restrict__ even)
{
    __shared__ unsigned long long ss[16], sm[16];
    unsigned long long a = 0, b = 0;
    for (int k = threadIdx.x; k < nparts; k += blockDim.x) { a += partial[2 * k]; b += partial[2 * k + 1]; }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { ss[w] = a; sm[w] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long x = 0, y = 0;
        for (int k = 0; k < (int)(blockDim.x >> 6); k++) { x += ss[k]; y += sm[k]; }
        total[0] = x;
        total[1] = y;
        *even = (int)(1e6 * (double)x / (64.0 * (double)(y > 0 ? y : 1)));
    }
}

// The force pass's order of each block of span rows (span a power of two, at most
// kSchedMaxSpan): longest list first, ties in row order (lengths above 2047 tie), by a bitonic
// sort of (2047 - length, row) keys in LDS; the plain order when the waves are even.  The rows
// of a block stay close in space; their waves even out.
__global__ void __launch_bounds__(1024) k_sched_sort(int nrows, int span, const int *__restrict__ cnt,
                                                     const unsigned long long *__restrict__ total, double min_even,
                                                     int *__restrict__ sched)
{
    __shared__ unsigned int key[kSchedMaxSpan];
    const int base = blockIdx.x * span;
    const int m = min(span, nrows - base);  // rows of this block
    const double even = (double)total[0] / (64.0 * (double)(total[1] > 0 ? total[1] : 1));
    if (!(even < min_even)) {
        for (int k = threadIdx.x; k < m; k += blockDim.x) sched[base + k] = base + k;
        return;
    }
    for (int k = threadIdx.x; k < span; k += blockDim.x) {
        // rows past the end sort last
        const unsigned c = k < m ? (unsigned)min(cnt[base + k], 2047) : 0u;
        key[k] = k < m ? (((2047u - c) << 11) | (unsigned)k) : 0xffffffffu;
    }
    __syncthreads();
    for (int size = 2; size <= span; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int k = threadIdx.x; k < span / 2; k += blockDim.x) {
                // the pair (lo, hi) of this compare-exchange, ascending within blocks of size
                const int lo = 2 * k - (k & (stride - 1));
                const int hi = lo + stride;
                const bool up = (lo & size) == 0;
                const unsigned a = key[lo], b2 = key[hi];
                if ((a > b2) == up) { key[lo] = b2; key[hi] = a; }
            }
            __syncthreads();
        }
    }
    for (int k = threadIdx.x; k < m; k += blockDim.x) sched[base + k] = base + (int)(key[k] & 2047u);
}
#endif

}  // namespace gz
