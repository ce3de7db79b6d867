// gz_rows_impl.h -- the hot-path passes with one wavefront per active row, for steps in which
// few particles are active (the usual case of adaptive time bins: a few hundred hot particles
// in a resting medium).  The 64 lanes of the row's wavefront evaluate 64 candidates or list
// entries at once; each lane's pair terms go to LDS, and then lane k keeps running sum k (one
// lane per accumulated quantity) over the accepted entries in ascending order, so every sum is
// the same chain of additions as in the lane-per-row kernels (and the oracle).  One wavefront
// per workgroup: the block barrier is a wave barrier.
#pragma once
#include "gz_kernels_impl.h"

namespace gz {

// The candidates of a row: the non-empty cells of its home cell's 27-stencil in ascending cell
// code (cells are consecutive ranges of the Morton order, so this is ascending start: the
// candidates come in ascending particle index whatever the grid level), laid end to end.
// Virtual index v maps to the particle of range k with pref[k] <= v < pref[k+1].
constexpr int kMarked = 1024;  // candidates whose range is found by counting bits (row_candidate_marked)
// the sum of the values of lanes 0 .. lane, for lanes below 32
__device__ __forceinline__ int scan32(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1, 2, 4, 8
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    return x;
}

struct RangeMarks {
    unsigned long long first[kMarked / 64];  // a bit per candidate: the first of its range
    int range[kMarked / 64];                 // for each word: the range of the word's first candidate, less bit 0 of the word
    // candidate v's range, where the wavefront's lanes hold 64 consecutive v from a multiple of 64:
    // the marks up to this lane's in its word
    __device__ __forceinline__ int range_of(int v) const
    {
        const unsigned long long word = first[v >> 6] >> 1;
        return range[v >> 6] + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(word >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)word, 0));
    }
    // built by one wavefront: cleared, each range's first candidate marked (no range is empty), counted
    __device__ __forceinline__ void clear(int lane)
    {
        if (lane < kMarked / 64) first[lane] = 0;
    }
    __device__ __forceinline__ void mark(int pref)
    {
        if (pref < kMarked) atomicOr(&first[pref >> 6], 1ull << (pref & 63));
    }
    __device__ __forceinline__ void count(int lane)
    {
        const unsigned long long word = lane < kMarked / 64 ? first[lane] : 0ull;
        const int marks = __popcll(word), upto = scan32(marks);
        if (lane < kMarked / 64) range[lane] = upto - marks + (int)(word & 1ull) - 1;
    }
};
struct RowStencil {
    int start[27];
    int pref[28];
    int len[27];
    int nst;
    int shift[27];  // start - pref
    RangeMarks marks;
};

// The ranges in ascending code, of a grid of nc cells a side.  The lanes of the first wavefront bring
// their cell's code (0x7fffffff: dropped, all lanes from 27 on) and range; of equal codes (grids under
// 3 cells a side) the first lane stays.  The ranks come from 27 lane broadcasts and the prefix of
// the lengths from a scan in registers: loops over LDS words here were a chain of 80 dependent
// reads (about 5000 cycles), a third of the time of a row.
__device__ __forceinline__ void stencil_finish(RowStencil &rs, int nc, int code, int st, int en)
{
    const int lane = threadIdx.x;
    int m = 0;
    if (lane < 64) {
        if (nc < 3) {
            for (int q = 0; q < 26; q++) {
                const int cq = lane_value(code, q);
                if (lane > q && code == cq) code = 0x7fffffff;
            }
        }
        const bool kept = code != 0x7fffffff;
        int rank = 0;  // kept codes below this one
#pragma unroll
        for (int q = 0; q < 27; q++) rank += lane_value(code, q) < code;
        m = __popcll(__ballot(kept));
        if (kept) {
            rs.start[rank] = st;
            rs.len[rank] = en - st;
        }
        rs.marks.clear(lane);
    }
    __syncthreads();
    if (lane < 64) {
        const int len = lane < m ? rs.len[lane] : 0;
        const int upto = scan32(len), pref = upto - len;
        if (lane <= m) rs.pref[lane] = pref;
        if (lane < m) {
            rs.shift[lane] = rs.start[lane] - pref;
            rs.marks.mark(pref);
        }
        if (lane == 0) rs.nst = m;
    }
    __syncthreads();
    if (lane < 64) rs.marks.count(lane);
    __syncthreads();
}


// The stencil of the row's home cell, built by 27 lanes (one per neighbour cell): periodic
// neighbours, duplicates of small grids dropped, cells beyond reach dropped (the row lies
// farther from the cell's box than its reach plus the distance any particle has moved from its
// cell; reach = h_i, or max(h_i, the cell's largest radius) for the symmetric test), ranks by
// code, then the prefix of the lengths.
template <bool SYM>
__device__ __forceinline__ void row_stencil(const GridView &g, uint32_t home, double xi, double yi, double zi, double hrow,
                                            RowStencil &rs)
{
    const int lane = threadIdx.x;
    const int nc = 1 << g.level;
    const int cx = compact10(home >> 2), cy = compact10(home >> 1), cz = compact10(home);
    int code = 0x7fffffff, st = 0, en = 0;
    if (lane < 27) {
        const int dx = lane / 9 - 1, dy = (lane / 3) % 3 - 1, dz = lane % 3 - 1;
        const int a = (cx + dx) & (nc - 1), b = (cy + dy) & (nc - 1), d = (cz + dz) & (nc - 1);
        const int c = (int)((spread10(a) << 2) | (spread10(b) << 1) | spread10(d));
        st = g.cstart[g.cell_off + c];
        en = g.cend[g.cell_off + c];
        bool keep = en > st;
        if (keep && nc >= 4) {
            const double ox = cx * g.cell, oy = cy * g.cell, oz = cz * g.cell;
            const double rx = wrap(xi - ox, g.box, g.half), ry = wrap(yi - oy, g.box, g.half), rz = wrap(zi - oz, g.box, g.half);
            // gap from the row to the neighbour cell's box [d*cell, (d+1)*cell) along each axis
            const double gx = fmax(fmax(dx * g.cell - rx, rx - (dx + 1) * g.cell), 0.0);
            const double gy = fmax(fmax(dy * g.cell - ry, ry - (dy + 1) * g.cell), 0.0);
            const double gz = fmax(fmax(dz * g.cell - rz, rz - (dz + 1) * g.cell), 0.0);
            double reach = hrow;
            if (SYM) reach = fmax(reach, g.chmax ? g.chmax[g.cell_off + c] : g.hall);
            const double rr = (reach + g.margin) * (1.0 + 1e-9) + 1e-12 * g.box;
            if (gx * gx + gy * gy + gz * gz > rr * rr) keep = false;
        }
        if (keep) code = c;
    }
    stencil_finish(rs, nc, code, st, en);
}

// (v < the total; the range k with pref[k] <= v < pref[k+1], the last such k when empty ranges
// share a prefix value: binary search over the at most 27 prefixes)
__device__ __forceinline__ int row_candidate(const RowStencil &rs, int v)
{
    int lo = 0, hi = rs.nst - 1;  // invariant: pref[lo] <= v, and the answer is at most hi
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (rs.pref[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return rs.start[lo] + (v - rs.pref[lo]);
}

// the same for totals up to kMarked, as RangeMarks::range_of
__device__ __forceinline__ int row_candidate_marked(const RowStencil &rs, int v) { return v + rs.shift[rs.marks.range_of(v)]; }

// ---------------------------------------------------------------------------------------
// search over many grid levels (WideGrid)
// ---------------------------------------------------------------------------------------

// the finest level (at most lmax) whose cells are no smaller than reach
__device__ __forceinline__ int wide_level(double box, int lmax, double reach)
{
    int L = 0;
    double side = 0.5 * box;  // of level L + 1 (halving is exact)
    while (L < lmax && side >= reach * (1.0 + 1e-6)) {
        L++;
        side *= 0.5;
    }
    return L;
}

// the range [a, b) of the cell with code c (key >> s) from table entry e, if the entry is
// exactly a maximal run of that code among positions [lo, hi) (key: of each position); otherwise
// the cell is empty
__device__ __forceinline__ bool wide_range(const int *__restrict__ start, const int *__restrict__ end, long long e,
                                           const uint32_t *__restrict__ key, int lo, int hi, int s,
                                           uint32_t c, int &a, int &b)
{
    a = start[e];
    b = end[e];
    if (!(a >= lo && a < b && b <= hi)) return false;
    // (all four at once: one wait)
    const uint32_t first = key[a] >> s, last = key[b - 1] >> s, before = key[max(a - 1, lo)] >> s, after = key[min(b, hi - 1)] >> s;
    return first == c && last == c && !(a > lo && before == c) && !(b < hi && after == c);
}

// The 27-cell stencil at level L around the row (home = the row's key >> s), from the tables
// of all particles (LIST false: ranges of the order) or of the particles of level L (LIST
// true: ranges of positions in lidx).  Cells beyond reach + margin are dropped when reach > 0.
template <bool LIST>
__device__ __forceinline__ void row_stencil_wide(const GridView &g, const WideGrid &W, int L, uint32_t home, double xi, double yi,
                                                 double zi, double reach, RowStencil &rs)
{
    const int lane = threadIdx.x;
    const int nc = 1 << L;
    const int s = 3 * (kFineLevel - L);
    const double cell = ldexp(g.box, -L);
    const int cx = compact10(home >> 2), cy = compact10(home >> 1), cz = compact10(home);
    int code = 0x7fffffff, st = 0, en = 0;
    if (lane < 27) {
        const int dx = lane / 9 - 1, dy = (lane / 3) % 3 - 1, dz = lane % 3 - 1;
        const int a = (cx + dx) & (nc - 1), b = (cy + dy) & (nc - 1), d = (cz + dz) & (nc - 1);
        const uint32_t c = (spread10(a) << 2) | (spread10(b) << 1) | spread10(d);
        const long long e = W.loff[L] + c;
        bool keep = LIST ? wide_range(W.lstart, W.lend, e, W.lkey, W.lofs[L], W.lofs[L + 1], s, c, st, en)
                         : wide_range(W.start, W.end, e, W.key, 0, W.n, s, c, st, en);
        if (keep && nc >= 4 && reach > 0) {
            const double ox = cx * cell, oy = cy * cell, oz = cz * cell;
            const double rx = wrap(xi - ox, g.box, g.half), ry = wrap(yi - oy, g.box, g.half), rz = wrap(zi - oz, g.box, g.half);
            const double gx = fmax(fmax(dx * cell - rx, rx - (dx + 1) * cell), 0.0);
            const double gy = fmax(fmax(dy * cell - ry, ry - (dy + 1) * cell), 0.0);
            const double gz = fmax(fmax(dz * cell - rz, rz - (dz + 1) * cell), 0.0);
            const double rr = (reach + g.margin) * (1.0 + 1e-9) + 1e-12 * g.box;
            if (gx * gx + gy * gy + gz * gz > rr * rr) keep = false;
        }
        if (!keep) { st = 0; en = 0; }
        if (keep) code = (int)c;
    }
    stencil_finish(rs, nc, code, st, en);
}

// ---------------------------------------------------------------------------------------
// Long walks over many levels.  The cells of a coarse level next to a clump hold up to a tenth of all
// particles (1M lognormal particles: 100K candidates for the rows of one cell), and one
// wavefront walks them.  The bounding box and the largest radius of every 64 consecutive particles
// let a lane drop 64 candidates at once.  Mean density round of 1M lognormal rows FP64 2.5 -> 1.9 ms, of
// 4M rows FP32 5.7 -> 4.3 ms (before the rounds collected their partners first, below).
// ---------------------------------------------------------------------------------------
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(256) k_block_boxes(int n, const double *__restrict__ X, const double *__restrict__ Y,
                                                     const double *__restrict__ Z, const double *__restrict__ H, double inv_box,
                                                     float4 *__restrict__ boxes)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = j < n;
    // in units of the box, whose squares FP32 holds whatever the caller's units are; rounded outwards by
    // the caller's slack (2^-23 of the box)
    const float x = on ? (float)(X[j] * inv_box) : 0.0f, y = on ? (float)(Y[j] * inv_box) : 0.0f, z = on ? (float)(Z[j] * inv_box) : 0.0f,
                h = on ? (float)(H[j] * inv_box) : 0.0f;
    const float lx = wave_minf(on ? x : 1e30f), ly = wave_minf(on ? y : 1e30f), lz = wave_minf(on ? z : 1e30f);
    const float mx = -wave_minf(on ? -x : 1e30f), my = -wave_minf(on ? -y : 1e30f), mz = -wave_minf(on ? -z : 1e30f), hm = -wave_minf(-h);
    if (on && (j & 63) == 0) {
        boxes[2 * (j >> 6)] = make_float4(lx, ly, lz, hm);
        boxes[2 * (j >> 6) + 1] = make_float4(mx, my, mz, 0.0f);
    }
}
#endif

// what a block's particles are tested against: the rows' bounding box (centre, half extents) and radius,
// in units of the box
struct BlockReach {
    float cx, cy, cz, ex, ey, ez, h;
    // whether a pair of a row and a particle of block b may lie within the larger radius (SYM) or the
    // row's; the slack covers the FP32 rounding of the positions and the boxes
    template <bool SYM> __device__ __forceinline__ bool hits(const float4 &lo, const float4 &hi) const
    {
        auto gap = [&](float c, float e, float l, float m) {
            float d = fabsf(c - 0.5f * (l + m));
            d = d > 0.5f ? 1.0f - d : d;
            return fmaxf(d - e - 0.5f * (m - l) - 2e-6f, 0.0f);
        };
        const float gx = gap(cx, ex, lo.x, hi.x), gy = gap(cy, ey, lo.y, hi.y), gz = gap(cz, ez, lo.z, hi.z);
        const float r = (SYM ? fmaxf(h, lo.w) : h) * (1.0f + 1e-5f);
        return gx * gx + gy * gy + gz * gz <= r * r;
    }
};

// Of 64 runs of RUN candidates from v0 on (at(v): candidate v's particle, negative: not from the
// order), the ones that may hold a partner, as a bit per run.  hit(lowest corner and largest
// radius, highest corner) tells whether a block may hold one; all lanes call it together.  A run
// whose particles are consecutive covers few blocks; any other run is kept.
template <int RUN, typename At, typename Hit>
__device__ __forceinline__ unsigned long long live_runs(const float4 *__restrict__ boxes, int v0, int total, At at, Hit hit)
{
    const int a = v0 + RUN * (int)(threadIdx.x & 63);
    bool live = false;
    int b = 1, e = 0;  // the blocks still to look at
    if (a < total) {
        const int last = min(a + RUN, total) - 1, j0 = at(a), j1 = at(last);
        live = j0 < 0 || j1 - j0 != last - a;
        if (!live) {
            b = j0 >> 6;
            e = j1 >> 6;
        }
    }
    while (wave_any(b <= e)) {
        const bool look = b <= e;
        const float4 lo = boxes[look ? 2 * b : 0], hi = boxes[look ? 2 * b + 1 : 0];
        if (hit(lo, hi) && look) {
            live = true;
            e = -1;
        }
        b++;
    }
    return __ballot(live);
}

// The place of this thread's entry among the flagged entries of its workgroup, in thread order
// (total: the flagged entries of the workgroup).  One barrier for several wavefronts, none for one.
// The masks are read behind it, so a call that takes the same smask[TPB / 64] must lie behind another
// barrier: one of the caller's own, or that of a call in between which took another buffer (two
// buffers that turn at every call and at nothing else).
template <int TPB>
__device__ __forceinline__ int flagged_rank(bool flag, unsigned long long *smask, int &total)
{
    const unsigned long long mask = __ballot(flag);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (TPB == 64) {
        total = __popcll(mask);
        return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
    }
    if (lane == 0) smask[w] = mask;
    __syncthreads();
    int before = 0;
    total = 0;
    for (int k = 0; k < TPB / 64; k++) {
        const int c = __popcll(smask[k]);
        if (k < w) before += c;
        total += c;
    }
    return before + __popcll(mask & ((1ull << lane) - 1ull));
}

// acc + s[0] + s[1] + ... + s[n-1] (or minus each, neg), added one after another in that order;
// the loads run ahead of the chain of additions (the terms of a round sit contiguously in LDS)
template <typename R>
__device__ __forceinline__ R ordered_sum(R acc, const R *s, int n, bool neg)
{
    int k = 0;
    for (; k + 4 <= n; k += 4) {
        R a = s[k], b = s[k + 1], c = s[k + 2], d = s[k + 3];
        if (neg) { a = -a; b = -b; c = -c; d = -d; }
        acc = acc + a;
        acc = acc + b;
        acc = acc + c;
        acc = acc + d;
    }
    for (; k < n; k++) acc = acc + (neg ? -s[k] : s[k]);
    return acc;
}

// density sums of the rows still iterating (DensitySpec::pair_kernel,
// src/hydro/density_loop.h:1141-1385), the terms in k_density_cells' order.
// Two phases: the candidates' distances find the partners (one in five to twenty), which a ring in LDS
// collects in order; whenever it holds a workgroup's worth, each thread computes one partner's terms
// and one thread per sum adds them in order.  The terms (about 150 instructions) thus run once per row
// on full wavefronts where they ran for every candidate chunk that held a partner.  Bound by
// latencies (the stencil, the candidates' gathers) and the 450 instructions of the stencil.
// 1M lognormal rows FP64 1.90 -> 1.35 ms (mean of a pass's rounds), 4M FP32 4.3 -> 3.0 ms; 4 wavefronts per row for a few
// hundred rows 19.2 -> 10.0 us.
template <int KERN, typename R, int TPB>
__global__ void __launch_bounds__(TPB) k_density_rows(DevParams P, GridView g, int nrows, const int *__restrict__ act,
                                                     const uint8_t *__restrict__ need, const uint32_t *__restrict__ key,
                                                     const double *__restrict__ X, const double *__restrict__ Y,
                                                     const double *__restrict__ Z, const double *__restrict__ VX,
                                                     const double *__restrict__ VY, const double *__restrict__ VZ,
                                                     const double *__restrict__ M, const double *__restrict__ hcur,
                                                     double *__restrict__ accout, BoxTable bt, int *__restrict__ npairs,
                                                     const int *__restrict__ rows, int nlist)
{
    __shared__ RowStencil rs;
    __shared__ R sc[kDensSumsFD][TPB + 1];  // the partners' terms, in candidate order (padded: no bank conflicts)
    __shared__ int list[2 * TPB];           // a ring of partners found
    __shared__ unsigned long long smask[2][TPB / 64];
    // workgroup b takes row b, or the b-th row of the list of rows still iterating; the pair
    // count goes to npairs[b]
    const long b = xcd_block();
    if (b >= (rows ? nlist : nrows)) return;
    const long r = rows ? rows[b] : b;
    if (!need[r]) {
        if (npairs && threadIdx.x == 0) npairs[b] = 0;
        return;
    }
    const int tid = threadIdx.x;
    const int i = act[r];
    resolve_box(bt, i, P, g);
    const double xi = X[i], yi = Y[i], zi = Z[i];
    const R vxi = (R)VX[i], vyi = (R)VY[i], vzi = (R)VZ[i];
    const double h = hcur[r];
    const R hR = (R)h;
    const R h2 = hR * hR;
    R hinv, hinv3, hinv4;
    kernel_hinv(hR, hinv, hinv3, hinv4);
    if (g.wide) {
        // the row's own level: cells no smaller than its radius plus twice the displacement bound
        const WideGrid &W = *g.wide;
        const int L = wide_level(g.box, W.lmax, h + 2.0 * g.margin);
        row_stencil_wide<false>(g, W, L, key[i] >> (3 * (kFineLevel - L)), xi, yi, zi, h, rs);
    } else {
        row_stencil<false>(g, key[i] >> g.shift, xi, yi, zi, h, rs);
    }
    // FP32 form on one grid of at least 8 cells a side: differences of positions relative to the
    // home cell's origin, the cell walk's arithmetic (the two walks give the same bits)
    const bool rel = std::is_same<R, float>::value && !g.wide && (1 << g.level) >= 8;
    double ox = 0, oy = 0, oz = 0;
    if (rel) {
        const uint32_t home = key[i] >> g.shift;
        ox = compact10(home >> 2) * g.cell; oy = compact10(home >> 1) * g.cell; oz = compact10(home) * g.cell;
    }
    const R rxi = (R)wrap(xi - ox, g.box, g.half), ryi = (R)wrap(yi - oy, g.box, g.half), rzi = (R)wrap(zi - oz, g.box, g.half);
    const int total = rs.pref[rs.nst];
    const bool fd = P.fd4alpha > 0;
    const int nsum = fd ? kDensSumsFD : kDensSums;
    const double inv_box = 1.0 / P.box;
    R acc = 0;  // thread q < nsum keeps sum q
    int accepted = 0;  // this wavefront's share of the row's pairs (the pass's work, counted when npairs is given)
    // the separation from particle j; both uses below compute the same bits
    auto separation = [&](int j, R &dp0, R &dp1, R &dp2) {
        if (rel) {
            dp0 = rxi - (R)wrap_near(X[j] - ox, P.box, inv_box);
            dp1 = ryi - (R)wrap_near(Y[j] - oy, P.box, inv_box);
            dp2 = rzi - (R)wrap_near(Z[j] - oz, P.box, inv_box);
        } else {
            dp0 = (R)wrap_near(xi - X[j], P.box, inv_box);
            dp1 = (R)wrap_near(yi - Y[j], P.box, inv_box);
            dp2 = (R)wrap_near(zi - Z[j], P.box, inv_box);
        }
    };
    // the terms of the first nt partners of the list, side by side in LDS, and the sums over them
    auto add_partners = [&](int first, int nt) {
        __syncthreads();  // the list is whole
        bool counted = false;
        if (tid < nt) {
            const int j = list[(first + tid) & (2 * TPB - 1)];
            const double mj = M[j];
            const R vxj = (R)VX[j], vyj = (R)VY[j], vzj = (R)VZ[j];
            R dp0, dp1, dp2;
            separation(j, dp0, dp1, dp2);
            R t[kDensSumsFD];
            // a retired particle adds zeros, and so does the particle itself (rr = 0) to all but the
            // first three sums: sums that start at +0 stay the same bit for bit
            for (int q = 0; q < kDensSumsFD; q++) t[q] = 0;
            counted = mj > 0;
            if (counted) {
                const R r2 = dp0 * dp0 + dp1 * dp1 + dp2 * dp2;
                const R rr = sqrt(r2);
                const R u = rr * hinv;
                R wk = 0, dwk = 0;
                kernel_main<KERN, 0>(u, hinv3, hinv4, wk, dwk);
                t[0] = wk;
                t[1] = (R)mj * wk;
                t[2] = -(R(3.0) * hinv * wk + u * dwk);
                if (rr > 0) {
                    t[4] = wk * (dp0 * dp0);
                    t[5] = wk * (dp1 * dp1);
                    t[6] = wk * (dp2 * dp2);
                    t[7] = wk * (dp0 * dp1);
                    t[8] = wk * (dp1 * dp2);
                    t[9] = wk * (dp0 * dp2);
                    t[10] = wk * dp0;
                    t[11] = wk * dp1;
                    t[12] = wk * dp2;
                    const R dv0 = vxi - vxj, dv1 = vyi - vyj, dv2 = vzi - vzj;
                    t[3] = dwk * (dp0 * dv0 + dp1 * dv1 + dp2 * dv2) / rr;
                    if (fd) {  // GradH_numer, GradH_denom (src/hydro/density_loop.h:1281-1286)
                        t[13] = (dwk / rr) * dp0;
                        t[14] = (dwk / rr) * dp1;
                        t[15] = (dwk / rr) * dp2;
                        t[16] = u * dwk;
                    }
                }
            }
            // static bounds: the terms stay in registers
            for (int q = 0; q < kDensSums; q++) sc[q][tid] = t[q];
            if (fd)
                for (int q = kDensSums; q < kDensSumsFD; q++) sc[q][tid] = t[q];
        }
        accepted += __popcll(__ballot(counted));
        __syncthreads();
        if (tid < nsum) acc = ordered_sum(acc, sc[tid], nt, tid == 3);
    };
    const bool long_walk = g.wide && total > kLongWalk;
    const bool marked = total <= kMarked;
    const BlockReach reach{(float)(xi * inv_box), (float)(yi * inv_box), (float)(zi * inv_box), 0.0f, 0.0f, 0.0f, (float)(h * inv_box)};
    unsigned long long live = ~0ull;
    int head = 0, fill = 0;  // the partners found and not yet added: list places head .. head + fill - 1
    int turn = 0;  // the rank buffer of the next walked run (a skipped run has no barrier: it must not turn)
    for (int base = 0, run = 0; base < total || fill > 0; base += TPB, run++) {
        bool walk = base < total;
        if (walk && long_walk) {
            // (every wavefront of the workgroup finds the same bits)
            if ((run & 63) == 0)
                live = live_runs<TPB>(g.wide->boxes, base, total, [&](int v) { return row_candidate(rs, v); },
                                      [&](const float4 &lo, const float4 &hi) { return reach.hits<false>(lo, hi); });
            walk = (live >> (run & 63)) & 1ull;
        }
        if (walk) {
            const int v = base + tid;
            bool ok = false;
            int j = 0;
            if (v < total) {
                j = marked ? row_candidate_marked(rs, v) : row_candidate(rs, v);
                R dp0, dp1, dp2;
                separation(j, dp0, dp1, dp2);
                ok = dp0 * dp0 + dp1 * dp1 + dp2 * dp2 < h2;
            }
            int nok;
            const int pos = flagged_rank<TPB>(ok, smask[turn], nok);
            turn ^= 1;
            if (ok) list[(head + fill + pos) & (2 * TPB - 1)] = j;
            fill += nok;
        }
        if (fill >= TPB || (base + TPB >= total && fill > 0)) {
            const int nt = min(fill, TPB);
            add_partners(head, nt);
            head += nt;
            fill -= nt;
        }
    }
    if (tid < nsum) accout[(size_t)tid * nrows + r] = (double)acc;
    if (npairs) {
        __syncthreads();
        if ((tid & 63) == 0) smask[0][tid >> 6] = (unsigned long long)accepted;
        __syncthreads();
        if (tid == 0) {
            int all = 0;
            for (int w = 0; w < TPB / 64; w++) all += (int)smask[0][w];
            npairs[b] = all;
        }
    }
}

// the symmetric list of few rows (the same entries, in the same order, as k_build_sym_cells)
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(kRowThreads) k_build_sym_rows(GridView g, int nrows, const int *__restrict__ act, const uint32_t *__restrict__ key,
                                                       const double *__restrict__ X, const double *__restrict__ Y,
                                                       const double *__restrict__ Z, const double *__restrict__ H, int *__restrict__ ell,
                                                       long ld, int cap, int *__restrict__ cnt, int *__restrict__ overflow,
                                                       BoxTable bt)
{
    __shared__ RowStencil rs;
    __shared__ int scount[2][kRowThreads / 64];
    const long r = xcd_block();
    if (r >= nrows) return;
    const int tid = threadIdx.x, w = tid >> 6;
    const int i = act[r];
    {
        DevParams P{};
        resolve_box(bt, i, P, g);
    }
    const double xi = X[i], yi = Y[i], zi = Z[i], hi = H[i];
    row_stencil<true>(g, key[i] >> g.shift, xi, yi, zi, hi, rs);
    const int total = rs.pref[rs.nst];
    int n = 0;
    for (int base = 0, it = 0; base < total; base += kRowThreads, it ^= 1) {
        const int v = base + tid;
        bool acc = false;
        int j = -1;
        if (v < total) {
            j = row_candidate(rs, v);
            acc = (j != i) && accept_pair<true>(xi, yi, zi, X[j], Y[j], Z[j], hi, H[j], g.box, g.half);
        }
        // place among the accepted candidates: the wavefronts before this one, then the lanes
        int cntk;
        const int pos = kept_rank(acc, cntk);
        if ((tid & 63) == 0) scount[it][w] = cntk;
        __syncthreads();  // (the two count buffers alternate: one barrier per round suffices)
        int off = 0, all = 0;
        for (int q = 0; q < kRowThreads / 64; q++) {
            const int cq = scount[it][q];
            if (q < w) off += cq;
            all += cq;
        }
        if (acc && n + off + pos < cap) ell[ell_at(ld, r, n + off + pos)] = j;
        n += all;
    }
    if (tid == 0) {
        cnt[r] = min(n, cap);  // readers stay inside the list; the overflow carries the full length
        if (n > cap) atomicMax(overflow, n);
    }
}

// ---------------------------------------------------------------------------------------
// search over many grid levels: tables, particle levels, symmetric rows
// ---------------------------------------------------------------------------------------

// the range of every cell of every level 0..lmax that holds particles (one lane per position)
__global__ void __launch_bounds__(256) k_wide_bounds(WideGrid W)
{
    const long p = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (p >= W.n) return;
    const uint32_t k = W.key[p];
    const uint32_t kp = p > 0 ? W.key[p - 1] : 0, kn = p + 1 < W.n ? W.key[p + 1] : 0;
    for (int L = 0; L <= W.lmax; L++) {
        const int s = 3 * (kFineLevel - L);
        const uint32_t c = k >> s;
        if (p == 0 || (kp >> s) != c) W.start[W.loff[L] + c] = (int)p;
        if (p + 1 == W.n || (kn >> s) != c) W.end[W.loff[L] + c] = (int)(p + 1);
    }
}

// each particle's own level (the finest, at most lmax, whose cells hold its radius plus twice
// the displacement bound), and the number of particles per level
__global__ void __launch_bounds__(256) k_particle_level(int n, const double *__restrict__ H, double box, double margin, int lmax,
                                                         int *__restrict__ plev, int *__restrict__ level_count)
{
    __shared__ int hist[kFineLevel + 1];
    if (threadIdx.x <= kFineLevel) hist[threadIdx.x] = 0;
    __syncthreads();
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) {
        const int L = wide_level(box, lmax, H[p] + 2.0 * margin);
        plev[p] = L;
        atomicAdd(&hist[L], 1);
    }
    __syncthreads();
    if (threadIdx.x <= kFineLevel && hist[threadIdx.x]) atomicAdd(&level_count[threadIdx.x], hist[threadIdx.x]);
}

// the range of every cell of level L among the particles of level L (positions in lidx)
__global__ void __launch_bounds__(256) k_wide_list_bounds(WideGrid W, const int *__restrict__ plev, const double *__restrict__ X,
                                                          const double *__restrict__ Y, const double *__restrict__ Z,
                                                          const double *__restrict__ H, double inv_box)
{
    const long p = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (p >= W.n) return;
    const int j = W.lidx[p];
    const int L = plev[j];
    const int s = 3 * (kFineLevel - L);
    const uint32_t c = W.key[j] >> s;
    const int lo = W.lofs[L], hi = W.lofs[L + 1];
    if (p == lo || (W.key[W.lidx[p - 1]] >> s) != c) W.lstart[W.loff[L] + c] = (int)p;
    if (p + 1 == hi || (W.key[W.lidx[p + 1]] >> s) != c) W.lend[W.loff[L] + c] = (int)(p + 1);
    W.lkey[p] = W.key[j];
    W.lpos[p] = make_float4((float)(X[j] * inv_box), (float)(Y[j] * inv_box), (float)(Z[j] * inv_box), (float)(H[j] * inv_box));
}

__device__ __forceinline__ bool periodic_adjacent(int a, int b, int nc)
{
    const int d = (a - b + 1) & (nc - 1);  // (nc is a power of two)
    return d <= 2 || nc < 3;
}

// Symmetric rows r2 < max(h_i,h_j)^2 (src/mesh/sfc_tiles_functions.h:83-102) over many levels.
// Part A: every particle in the 27 cells of the row's own level L_i (it holds every partner of
// level L_i or finer, and every partner within h_i).  Part B: for each coarser level L, the
// particles of level L in the 27 cells of level L around the row (a partner j of level L with
// r < h_j lies there) that Part A did not cover.  The row is then put in ascending order.
__global__ void __launch_bounds__(64) k_build_sym_wide(GridView g, int nrows, const int *__restrict__ act, const double *__restrict__ X,
                                                       const double *__restrict__ Y, const double *__restrict__ Z,
                                                       const double *__restrict__ H, int *__restrict__ ell, long ld, int cap,
                                                       int *__restrict__ cnt, int *__restrict__ overflow)
{
    __shared__ RowStencil rs;
    __shared__ int srt[1024];
    const long r = xcd_block();
    if (r >= nrows) return;
    const int lane = threadIdx.x;
    const int i = act[r];
    const WideGrid &W = *g.wide;
    const double xi = X[i], yi = Y[i], zi = Z[i], hi = H[i];
    const int Li = wide_level(g.box, W.lmax, hi + 2.0 * g.margin);
    const int si = 3 * (kFineLevel - Li);
    const uint32_t homei = W.key[i] >> si;
    row_stencil_wide<false>(g, W, Li, homei, xi, yi, zi, -1.0, rs);
    int total = rs.pref[rs.nst];
    int n = 0;
    for (int base = 0; base < total; base += 64) {
        const int v = base + lane;
        bool acc = false;
        int j = -1;
        if (v < total) {
            j = row_candidate(rs, v);
            acc = (j != i) && accept_pair<true>(xi, yi, zi, X[j], Y[j], Z[j], hi, H[j], g.box, g.half);
        }
        int cntk;
        const int pos = kept_rank(acc, cntk);
        if (acc && n + pos < cap) ell[ell_at(ld, r, n + pos)] = j;
        n += cntk;
    }
    const int nA = n;
    const int nci = 1 << Li;
    const int hx = compact10(homei >> 2), hy = compact10(homei >> 1), hz = compact10(homei);
    for (int L = 0; L < Li; L++) {
        if (W.lofs[L + 1] == W.lofs[L]) continue;  // no particle of this level
        __syncthreads();  // every lane is done with rs before it is built again
        const int s = 3 * (kFineLevel - L);
        row_stencil_wide<true>(g, W, L, W.key[i] >> s, xi, yi, zi, -1.0, rs);
        total = rs.pref[rs.nst];
        for (int base = 0; base < total; base += 64) {
            const int v = base + lane;
            bool acc = false;
            int j = -1;
            if (v < total) {
                j = W.lidx[row_candidate(rs, v)];
                const uint32_t cj = W.key[j] >> si;
                const bool in_a = periodic_adjacent((int)compact10(cj >> 2), hx, nci) && periodic_adjacent((int)compact10(cj >> 1), hy, nci) &&
                                  periodic_adjacent((int)compact10(cj), hz, nci);
                acc = !in_a && (j != i) && accept_pair<true>(xi, yi, zi, X[j], Y[j], Z[j], hi, H[j], g.box, g.half);
            }
            int cntk;
            const int pos = kept_rank(acc, cntk);
            if (acc && n + pos < cap) ell[ell_at(ld, r, n + pos)] = j;
            n += cntk;
        }
    }
    __syncthreads();  // the row's entries written by every lane are visible to all
    if (n > nA && n <= cap) {
        // ascending order: each entry's rank among the row's distinct entries
        if (n <= 1024) {
            for (int q = lane; q < n; q += 64) srt[q] = ell[ell_at(ld, r, q)];
            __syncthreads();
            for (int q = lane; q < n; q += 64) {
                const int e = srt[q];
                int rank = 0;
                for (int t = 0; t < n; t++) rank += srt[t] < e;
                ell[ell_at(ld, r, rank)] = e;
            }
        } else if (lane == 0) {
            for (int q = 1; q < n; q++) {
                const int e = ell[ell_at(ld, r, q)];
                int t = q - 1;
                while (t >= 0 && ell[ell_at(ld, r, t)] > e) { ell[ell_at(ld, r, t + 1)] = ell[ell_at(ld, r, t)]; t--; }
                ell[ell_at(ld, r, t + 1)] = e;
            }
        }
    }
    if (lane == 0) {
        cnt[r] = min(n, cap);  // readers stay inside the list; the overflow carries the full length
        if (n > cap) atomicMax(overflow, n);
    }
}
#endif

// ---------------------------------------------------------------------------------------
// symmetric list as a cell walk (one wavefront per occupied cell): rows r2 < max(h_i,h_j)^2, self
// excluded, ascending (src/mesh/sfc_tiles_functions.h:83-102); with row groups (CellRows.gsten) a
// group is one cell of one grid level or of one box.  Two kernels with the same lists:
// k_build_sym_cells, a row per lane, where the cells hold rows enough to fill a wavefront, and
// k_build_sym_groups, a candidate per lane, where they do not (kSymFewRows) and for the search
// over many levels.
// Before, one kernel with the exact FP64 test behind every staged candidate and a lane per row
// for both.  2M rows, 64 to a cell: 1.47 -> 1.00 ms (of cells, a row per lane); 128K rows, 4 to a
// cell: 700 -> 218 us; search over many levels (a dozen rows to a cell) 1M rows 6.3 -> 5.0 ms, 4M
// rows 23.1 -> 9.1 ms.  Candidates laid end to end (as the groups' ranges are) made the walk of
// full cells slower (1.00 -> 1.25 ms: the search for a lane's range).
// ---------------------------------------------------------------------------------------
#ifdef GZ_DEFINE_COMMON_KERNELS
// Candidates are culled against the rows' bounding box and staged 64 at a time; each lane masks the
// tile with the FP32 test of the candidate window (k_density_cells), against the larger of the two
// radii, and takes its own candidates through the exact test.
__global__ void __launch_bounds__(64) k_build_sym_cells(GridView g, CellRows cr, const int *__restrict__ act,
                                                        const double *__restrict__ X, const double *__restrict__ Y,
                                                        const double *__restrict__ Z, const double *__restrict__ H,
                                                        int *__restrict__ ell, long ld, int cap, int *__restrict__ cnt,
                                                        int *__restrict__ overflow)
{
    __shared__ double sx[kWinRing], sy[kWinRing], sz[kWinRing], sh[kWinRing];
    __shared__ int sj[kWinRing];
    __shared__ float4 st[64];
    __shared__ float sth[64];
    const long cb = xcd_block();
    if (cb >= (cr.ncells_dev ? *cr.ncells_dev : cr.ncells)) return;
    int c, a0, a1, nst;
    const int4 *sten;
    if (cr.gsten) {
        c = cr.gcode[cb]; a0 = cr.gstart[cb]; a1 = cr.gstart[cb + 1]; nst = cr.gnst[cb]; sten = cr.gsten + (size_t)27 * cb;
        DevParams P{};
        resolve_box(cr.bt, act[cr.grow ? cr.grow[a0] : a0], P, g);
    } else {
        c = cr.cells[cb]; a0 = cr.ca0[c]; a1 = cr.ca1[c]; nst = g.nsten[c]; sten = g.sten + (size_t)c * 27;
    }
    const int t = threadIdx.x;
    // a cell's rows in equal parts of at most 64, dealt to the workgroups along y
    const int parts = (a1 - a0 + 63) / 64, part_rows = (a1 - a0 + parts - 1) / parts;
    for (int part = blockIdx.y; part < parts; part += gridDim.y) {
        const int base = a0 + part * part_rows;
        const bool on = t < part_rows && base + t < a1;
        const int r = on ? (cr.grow ? cr.grow[base + t] : base + t) : 0;
        int i = -1;
        double xi = 0, yi = 0, zi = 0, hi = 0;
        if (on) { i = act[r]; xi = X[i]; yi = Y[i]; zi = Z[i]; hi = H[i]; }
        const LeafBox lb = leaf_box(g, c, on, xi, yi, zi);
        const double hleaf = wave_max(on ? hi : 0.0);
        const bool small = (1 << g.level) >= 8;
        const double inv_cell = 1.0 / g.cell;
        const float ux = (float)(wrap(xi - lb.ox, g.box, g.half) * inv_cell - 0.5), uy = (float)(wrap(yi - lb.oy, g.box, g.half) * inv_cell - 0.5),
                    uz = (float)(wrap(zi - lb.oz, g.box, g.half) * inv_cell - 0.5), uh = (float)(hi * inv_cell);
        const float qx = -2.0f * ux, qy = -2.0f * uy, qz = -2.0f * uz, qh = uh * uh;
        const float lim = on ? (small ? kWinSlack - (ux * ux + uy * uy + uz * uz) : kWinSlack) : -1e30f;
        Window win;
        int head = 0, fill = 0, n = 0;
        int q = 0, ts = nst > 0 ? sten[0].x : 0, te = nst > 0 ? sten[0].y : 0;  // the next candidates
        bool more = nst > 0, left = false, keep = false;
        // the next 64 candidates, loaded while the last are tested and staged (with the walk in
        // parts along y: twelve boxes of 16^3 to 64^3 796 -> 704 us; 128^3 990 either way)
        double xn = 0, yn = 0, zn = 0, hn = 0;
        auto load_next = [&]() {
            if (ts + t < te) {
                xn = X[ts + t]; yn = Y[ts + t]; zn = Z[ts + t]; hn = H[ts + t];
            }
        };
        load_next();
        int pos = 0, j = 0;
        double xj = 0, yj = 0, zj = 0, hj = 0;
        auto stage = [&](int k) {
            const int s = head + k;
            sx[s] = xj; sy[s] = yj; sz[s] = zj; sh[s] = hj; sj[s] = j;
            const float fx = (float)(wrap(xj - lb.ox, g.box, g.half) * inv_cell - 0.5), fy = (float)(wrap(yj - lb.oy, g.box, g.half) * inv_cell - 0.5),
                        fz = (float)(wrap(zj - lb.oz, g.box, g.half) * inv_cell - 0.5), fh = (float)(hj * inv_cell);
            st[k] = make_float4(fx, fy, fz, fx * fx + fy * fy + fz * fz);
            sth[k] = fh * fh;
        };
        while (more || left) {
            __syncthreads();  // the lanes are done with the tile before the last and its test values
            if (keep) stage(pos);  // what the last tile had no room for
            keep = false;
            left = false;
            while (more && fill < 64) {
                const bool in_range = ts + t < te;
                j = ts + t;
                xj = xn; yj = yn; zj = zn; hj = hn;
                ts += 64;
                if (ts >= te) {
                    q++;
                    more = q < nst;
                    if (more) { ts = sten[q].x; te = sten[q].y; }
                }
                if (more) load_next();
                keep = in_range && leaf_reach(g, lb, xj, yj, zj, fmax(hleaf, hj));
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
            if (t >= nt) { st[t] = make_float4(0.0f, 0.0f, 0.0f, 1e30f); sth[t] = 0.0f; }  // no candidate
            __syncthreads();
            uint32_t mlo = 0, mhi = 0;
            if (small) {
#pragma unroll 4
                for (int k = 31; k >= 0; k--) {
                    const float4 u = st[k], v = st[k + 32];
                    mask_push(mlo, __builtin_fmaf(qx, u.x, __builtin_fmaf(qy, u.y, __builtin_fmaf(qz, u.z, u.w))) - fmaxf(qh, sth[k]), lim);
                    mask_push(mhi, __builtin_fmaf(qx, v.x, __builtin_fmaf(qy, v.y, __builtin_fmaf(qz, v.z, v.w))) - fmaxf(qh, sth[k + 32]), lim);
                }
            } else {
                // coarse grids: the nearest image of each difference
                const float nc = (float)(1 << g.level), inv_nc = 1.0f / nc;
                for (int k = 31; k >= 0; k--) {
                    mask_push(mlo, wrapped_r2(ux, uy, uz, st[k], nc, inv_nc) - fmaxf(qh, sth[k]), lim);
                    mask_push(mhi, wrapped_r2(ux, uy, uz, st[k + 32], nc, inv_nc) - fmaxf(qh, sth[k + 32]), lim);
                }
                const unsigned long long valid = nt == 64 ? ~0ull : (1ull << nt) - 1ull;
                mlo &= (uint32_t)valid;
                mhi &= (uint32_t)(valid >> 32);
            }
            win.push(((unsigned long long)mhi << 32) | mlo);
            head = head == kWinRing - 64 ? 0 : head + 64;
            const int room = more || left ? kWinWords - 2 : -1;
            do {
                if (win.ready()) {
                    const int k = win.next();
                    const int jj = sj[k];
                    if (jj != i && accept_pair<true>(xi, yi, zi, sx[k], sy[k], sz[k], hi, sh[k], g.box, g.half)) {
                        if (n < cap) ell[ell_at(ld, r, n)] = jj;
                        n++;
                    }
                }
            } while (wave_any(win.behind > room));
        }
        __syncthreads();  // before the next rows' candidates take the ring
        if (on) {
            cnt[r] = min(n, cap);  // readers stay inside the list; the overflow carries the full length
            if (n > cap) atomicMax(overflow, n);
        }
    }
}

// The candidates of a cell walk: up to kMaxRanges index ranges in ascending order, laid end to end, so
// that 64 candidates are taken at a time whatever the ranges' lengths (cells of a dozen particles
// would leave most lanes of a range-by-range walk idle).  Candidate v is start[k] + v - pref[k]
// of the last range k with pref[k] <= v.
constexpr int kMaxRanges = 56;
struct CellRanges {
    int shift[kMaxRanges];  // start - pref
    int pref[kMaxRanges];
    int n, total;
    RangeMarks marks;
    __device__ __forceinline__ int at(int v) const
    {
        int lo = 0, hi = n - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (pref[mid] <= v) lo = mid;
            else hi = mid - 1;
        }
        return v + shift[lo];
    }
    // 64 consecutive v from a multiple of 64
    __device__ __forceinline__ int at_lanes(int v) const { return total <= kMarked ? v + shift[marks.range_of(v)] : at(v); }
    // laid out by one wavefront: lane k < 28 brings range 2 k (starting at a0, of len0 candidates) and
    // range 2 k + 1; empty ones are dropped
    __device__ __forceinline__ void lay(int a0, int len0, int a1, int len1)
    {
        const int lane = threadIdx.x & 63;
        const int upto = scan32(len0 + len1), pref0 = upto - len0 - len1, pref1 = upto - len1;
        const unsigned long long some0 = __ballot(len0 > 0), some1 = __ballot(len1 > 0), below = (1ull << lane) - 1;
        const int k = __popcll(some0 & below) + __popcll(some1 & below);
        marks.clear(lane);
        __syncthreads();
        if (len0 > 0) {
            pref[k] = pref0;
            shift[k] = a0 - pref0;
            marks.mark(pref0);
        }
        if (len1 > 0) {
            const int k1 = k + (len0 > 0);
            pref[k1] = pref1;
            shift[k1] = a1 - pref1;
            marks.mark(pref1);
        }
        if (lane == 31) {
            n = __popcll(some0) + __popcll(some1);
            total = upto;
        }
        __syncthreads();
        marks.count(lane);
        __syncthreads();
    }
};

// the ranges of a stencil (one wavefront; nst <= 27 entries, one lane each)
__device__ __forceinline__ void stencil_ranges(CellRanges &cr, const int4 *__restrict__ sten, int nst)
{
    const int lane = threadIdx.x & 63;
    const int4 e = lane < nst ? sten[lane] : make_int4(0, 0, 0, 0);
    cr.lay(0, 0, e.x, e.y - e.x);
}

// One candidate per lane and the rows of the group in turn: no lane is idle however few rows a cell
// holds (a dozen in the search over many levels, whose cells are sized by the rows' own radii),
// and a ballot gives each accepted candidate its place.  The test is FP32 in units of the cell
// side (|x_i|^2 + |x_j|^2 - 2 x_i.x_j against the larger radius squared) with a bound on its
// rounding error; only a pair within that bound of the radius takes the exact test.
//
// The search over many levels adds the particles of each coarser level L in the 27 cells of
// level L around the group's cell that lie outside the 27 cells of the group's level (part B, as
// k_build_sym_wide).  They are collected first, sorted, and laid between the group's own ranges,
// so that the walk meets every candidate in ascending order; more than kMaxCoarse of them are
// inserted into the finished rows one by one.
//
// Bound by its VALU instructions (4M lognormal rows: 63% of the issue rate) and the latency of part B's
// stencils (3 to 6 levels of dependent table reads).  1M lognormal rows 5.0 -> 1.53 ms, 4M 9.1 -> 6.1: at 8
// cells a side every pair took the exact test and no block was skipped (217 groups of 37,000
// candidates took 3 to 6 ms each; 1.93 ms without them), part B's candidates came by four gathers and a
// key each, not by one packed record loaded a step ahead (1.53 and 6.1, with the row loop's
// masks in scalar registers 1.86 -> 1.68 of that).
constexpr int kMaxCoarse = 768;
// bound on the FP32 test's rounding error, per unit of |x_j|^2 + h_j^2 + 13 (|x_i|^2 <= 12 in cells):
// a dozen roundings of 2^-24 each of at most twice that
constexpr float kSymSlack = 2e-6f;
constexpr int kCoarseRange = 1 << 30;
__global__ void __launch_bounds__(64, 4) k_build_sym_groups(GridView g, CellRows cr, const int *__restrict__ act,
                                                         const double *__restrict__ X, const double *__restrict__ Y,
                                                         const double *__restrict__ Z, const double *__restrict__ H,
                                                         int *__restrict__ ell, long ld, int cap, int *__restrict__ cnt,
                                                         int *__restrict__ overflow)
{
    __shared__ RowStencil rs;
    __shared__ CellRanges cells;
    __shared__ int coarse[kMaxCoarse], sorted[kMaxCoarse], runs[kFineLevel + 2];
    __shared__ float4 st[64];  // a tile of candidates: position in cells, radius squared
    __shared__ int sj[64];
    // (the groups of the search over many levels come level by level, at very different costs)
    const long cb = xcd_block_dealt();
    if (cb >= (cr.ncells_dev ? *cr.ncells_dev : cr.ncells)) return;
    int c, a0, a1, nst;
    const int4 *sten;
    if (cr.gsten) {
        c = cr.gcode[cb]; a0 = cr.gstart[cb]; a1 = cr.gstart[cb + 1]; nst = cr.gnst[cb]; sten = cr.gsten + (size_t)27 * cb;
        if (cr.bt.b) {
            DevParams P{};
            resolve_box(cr.bt, act[cr.grow ? cr.grow[a0] : a0], P, g);
        } else {
            g.level = cr.glev[cb];
            g.cell = g.box / (double)(1 << g.level);
        }
    } else {
        c = cr.cells[cb]; a0 = cr.ca0[c]; a1 = cr.ca1[c]; nst = g.nsten[c]; sten = g.sten + (size_t)c * 27;
    }
    // the search over many levels adds part B (its groups are cells of the rows' own levels)
    const bool wide = cr.gsten && !cr.bt.b && g.wide;
    const int t = threadIdx.x;
    const int nci = 1 << g.level;
    const int hx = compact10((uint32_t)c >> 2), hy = compact10((uint32_t)c >> 1), hz = compact10((uint32_t)c);
    const int si = 3 * (kFineLevel - g.level);
    // the FP32 tests relative to the cell: grids of at least 8 cells a side, where a partner lies
    // within half a box of the cell's centre; 16 where particles of levels 0 and 1 may be partners,
    // up to box / 2.6 from the row (those of level 2 reach a quarter)
    const bool small = nci >= 16 || (nci == 8 && !(wide && g.wide->lofs[2] > 0));
    const double inv_cell = 1.0 / g.cell, inv_box = 1.0 / g.box;
    // a coordinate relative to the centre of the group's cell (index h along its axis), in cells
    auto rel = [&](double x, int h) { return (float)(wrap_near(x - h * g.cell, g.box, inv_box) * inv_cell - 0.5); };
    // a particle of a coarser level that the group's own cells do not hold
    auto outside = [&](uint32_t key) {
        const uint32_t cj = key >> si;
        return !(periodic_adjacent((int)compact10(cj >> 2), hx, nci) && periodic_adjacent((int)compact10(cj >> 1), hy, nci) &&
                 periodic_adjacent((int)compact10(cj), hz, nci));
    };
    if (!wide) stencil_ranges(cells, sten, nst);
    // a group's rows in equal parts of at most 64, dealt to the workgroups along y: where those are several,
    // parts of 16 rows or more (group_parts)
    const int parts = max((a1 - a0 + 63) / 64, min((int)gridDim.y, (a1 - a0 + 15) / 16)), part_rows = (a1 - a0 + parts - 1) / parts;
    for (int part = blockIdx.y; part < parts; part += gridDim.y) {
        const int base = a0 + part * part_rows;
        const bool on = t < part_rows && base + t < a1;
        const int r = on ? (cr.grow ? cr.grow[base + t] : base + t) : 0;
        int i = -1;
        double xi = 0, yi = 0, zi = 0, hi = 0;
        if (on) { i = act[r]; xi = X[i]; yi = Y[i]; zi = Z[i]; hi = H[i]; }
        // the rows in units of the cell side around the cell's centre, and their bounding box
        const float ux = rel(xi, hx), uy = rel(yi, hy), uz = rel(zi, hz), uh = (float)(hi * inv_cell);
        const float qx = -2.0f * ux, qy = -2.0f * uy, qz = -2.0f * uz, qn = ux * ux + uy * uy + uz * uz, qh = uh * uh;
        const float lx = wave_minf(on ? ux : 1e30f), ly = wave_minf(on ? uy : 1e30f), lz = wave_minf(on ? uz : 1e30f);
        const float mx = -wave_minf(on ? -ux : 1e30f), my = -wave_minf(on ? -uy : 1e30f), mz = -wave_minf(on ? -uz : 1e30f);
        const float hleaf = -wave_minf(on ? -uh : 0.0f);
        // a candidate that no row can reach (conservative: the slack covers the rounding)
        auto culled = [&](float fx, float fy, float fz, float fh, float sl) {
            const float ex = fmaxf(fmaxf(lx - fx, fx - mx) - sl, 0.0f), ey = fmaxf(fmaxf(ly - fy, fy - my) - sl, 0.0f),
                        ez = fmaxf(fmaxf(lz - fz, fz - mz) - sl, 0.0f), hm = fmaxf(fh, hleaf);
            return small && ex * ex + ey * ey + ez * ez > hm * hm + kSymSlack * (fx * fx + fy * fy + fz * fz + hm * hm + 12.0f);
        };
        int ncoarse = 0;  // part B's particles (above kMaxCoarse: not collected)
        if (wide) {
            const WideGrid &W = *g.wide;
            // the group's centre in units of the box, and the slack for positions rounded to 32 bits, in cells
            const float ic = (float)nci, inv_c = 1.0f / ic, sl = 4e-7f * ic;
            const float gx = ((float)hx + 0.5f) * inv_c, gy = ((float)hy + 0.5f) * inv_c, gz = ((float)hz + 0.5f) * inv_c;
            auto near = [&](float d) { return (d - __builtin_rintf(d)) * ic; };
            for (int L = 0; L < g.level && ncoarse <= kMaxCoarse; L++) {
                if (t == 0) runs[L] = ncoarse;
                if (W.lofs[L + 1] == W.lofs[L]) continue;  // no particle of this level
                __syncthreads();  // every lane is done with rs before it is built again
                row_stencil_wide<true>(g, W, L, (uint32_t)c >> (3 * (g.level - L)), 0.0, 0.0, 0.0, -1.0, rs);
                const int total = rs.pref[rs.nst];
                int pn = 0;
                float4 fn = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                auto load_next = [&](int v) {  // the next candidates, while the last are tested
                    if (v < total) {
                        pn = total <= kMarked ? row_candidate_marked(rs, v) : row_candidate(rs, v);
                        fn = W.lpos[pn];
                    }
                };
                load_next(t);
                for (int v0 = 0; v0 < total; v0 += 64) {
                    const int p = pn;
                    const float4 f = fn;
                    load_next(v0 + 64 + t);
                    bool keep = v0 + t < total && !culled(near(f.x - gx), near(f.y - gy), near(f.z - gz), f.w * ic, sl);
                    if (!wave_any(keep)) continue;
                    int j = 0;
                    if (keep) {
                        j = W.lidx[p];
                        keep = outside(W.lkey[p]);
                    }
                    int nt;
                    const int pos = ncoarse + kept_rank(keep, nt);
                    if (keep && pos < kMaxCoarse) coarse[pos] = j;
                    ncoarse += nt;
                }
            }
            __syncthreads();
            const int nb = ncoarse <= kMaxCoarse ? ncoarse : 0;
            if (t == 0 && nb) runs[g.level] = nb;
            __syncthreads();
            // merged: each level's particles ascend, so a particle's place is the sum of its places
            // among every level's
            for (int k = t; k < nb; k += 64) {
                const int e = coarse[k];
                int rank = 0;
                for (int L = 0; L < g.level; L++) {
                    const int first = runs[L];
                    int lo = first, hi2 = runs[L + 1];
                    while (lo < hi2) {
                        const int mid = (lo + hi2) >> 1;
                        if (coarse[mid] < e) lo = mid + 1;
                        else hi2 = mid;
                    }
                    rank += lo - first;
                }
                sorted[rank] = e;
            }
            __syncthreads();
            // ranges 2 q + 1: the stencil's cells, 2 q: the coarse particles before them (as their
            // places in `sorted`, less kCoarseRange), 2 nst: those after the last
            const int4 e = t < nst ? sten[t] : make_int4(0x7fffffff, 0x7fffffff, 0, 0);
            int before = 0, above = nb;  // coarse particles below e.x
            while (before < above) {
                const int mid = (before + above) >> 1;
                if (sorted[mid] < e.x) before = mid + 1;
                else above = mid;
            }
            const int prev = __shfl_up(before, 1, 64), bcount = before - (t ? prev : 0);
            cells.lay(before - bcount - kCoarseRange, t <= nst ? bcount : 0, e.x, t < nst ? e.y - e.x : 0);
        }
        const int rows = min(a1 - base, part_rows);
        int n = 0, fill = 0, v0 = 0, pos = 0, j = 0;
        bool more = cells.total > 0, left = false, keep = false;
        const bool long_walk = wide && cells.total > kLongWalk;
        const float ncf = (float)nci, inv_ncf = 1.0f / ncf;
        const float side = inv_ncf;  // the cell's, in units of the box
        const BlockReach reach{((float)hx + 0.5f * (lx + mx) + 0.5f) * side, ((float)hy + 0.5f * (ly + my) + 0.5f) * side,
                               ((float)hz + 0.5f * (lz + mz) + 0.5f) * side, 0.5f * (mx - lx) * side, 0.5f * (my - ly) * side,
                               0.5f * (mz - lz) * side, hleaf * side};
        // a block within reach of the rows' box and, for few rows, of one of them: a coarse cell's few
        // rows span a box that holds whole clumps which none of them reaches
        const float xf = (float)(xi * inv_box), yf = (float)(yi * inv_box), zf = (float)(zi * inv_box), hf = (float)(hi * inv_box);
        auto hit = [&](const float4 &lo, const float4 &hi) {
            bool any = reach.hits<true>(lo, hi);
            if (rows <= 16 && wave_any(any)) {
                bool one = false;
                for (int a = 0; a < rows; a++)
                    one |= BlockReach{lane_value(xf, a), lane_value(yf, a), lane_value(zf, a), 0.0f, 0.0f, 0.0f, lane_value(hf, a)}.hits<true>(lo, hi);
                any = any && one;
            }
            return any;
        };
        unsigned long long live = ~0ull;
        int run = 0;
        float fx = 0, fy = 0, fz = 0, fh = 0;
        auto stage = [&](int k) {
            st[k] = make_float4(fx, fy, fz, fh * fh);
            sj[k] = j;
        };
        while (more || left) {
            __syncthreads();  // the lanes have read the last tile
            if (keep) stage(pos);  // what the last tile had no room for
            keep = false;
            left = false;
            while (more && fill < 64) {
                if (long_walk) {
                    if ((run & 63) == 0)
                        live = live_runs<64>(g.wide->boxes, v0, cells.total, [&](int v) { return cells.at(v); }, hit);
                    const bool skip = !((live >> (run++ & 63)) & 1ull);
                    if (skip) {
                        v0 += 64;
                        more = v0 < cells.total;
                        continue;
                    }
                }
                if (v0 + t < cells.total) {
                    j = cells.at_lanes(v0 + t);
                    if (j < 0) j = sorted[j + kCoarseRange];
                    fx = rel(X[j], hx); fy = rel(Y[j], hy); fz = rel(Z[j], hz); fh = (float)(H[j] * inv_cell);
                    keep = !culled(fx, fy, fz, fh, 0.0f);
                }
                int nt;
                pos = fill + kept_rank(keep, nt);
                if (keep && pos < 64) {
                    stage(pos);
                    keep = false;
                }
                fill += nt;
                v0 += 64;
                more = v0 < cells.total;
            }
            const int nt = fill < 64 ? fill : 64;
            fill -= nt;
            left = fill > 0;
            pos -= 64;
            __syncthreads();
            const bool mine = t < nt;
            const float4 u = mine ? st[t] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const int cj = mine ? sj[t] : -1;
            const float w = u.x * u.x + u.y * u.y + u.z * u.z;
            const float slack = kSymSlack * (w + u.w + 13.0f);  // (a row's radius is at most the cell side)
            const unsigned long long tile = nt == 64 ? ~0ull : (1ull << nt) - 1ull;
            for (int a = 0; a < rows; a++) {
                const float r2 = small ? __builtin_fmaf(lane_value(qx, a), u.x, __builtin_fmaf(lane_value(qy, a), u.y, __builtin_fmaf(lane_value(qz, a), u.z, w))) + lane_value(qn, a)
                                       : wrapped_r2(lane_value(ux, a), lane_value(uy, a), lane_value(uz, a), u, ncf, inv_ncf);
                // (squares: the larger is the larger as an integer)
                const float d = r2 - __int_as_float(max(__float_as_int(u.w), lane_value(__float_as_int(qh), a)));
                const unsigned long long others = tile & ~__builtin_amdgcn_ballot_w64(cj == lane_value(i, a));
                const unsigned long long within = __builtin_amdgcn_ballot_w64(d < -slack);
                const unsigned long long close = others & (within ^ __builtin_amdgcn_ballot_w64(d <= slack));
                unsigned long long acc = others & within;
                if (close) {
                    bool in = false;
                    if ((close >> t) & 1ull)
                        in = accept_pair<true>(lane_value(xi, a), lane_value(yi, a), lane_value(zi, a), X[cj], Y[cj], Z[cj], lane_value(hi, a), H[cj],
                                               g.box, g.half);
                    acc |= __builtin_amdgcn_ballot_w64(in);
                }
                if (!acc) continue;
                const int held = lane_value(n, a);
                const int place = __builtin_amdgcn_mbcnt_hi((unsigned)(acc >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)acc, held));
                if (((acc >> t) & 1ull) && place < cap) ell[ell_at(ld, lane_value(r, a), place)] = cj;
                if (t == a) n += __popcll(acc);
            }
        }
        if (ncoarse > kMaxCoarse) {
            // too many to collect: each accepted one inserted in ascending place of its row
            const WideGrid &W = *g.wide;
            for (int L = 0; L < g.level; L++) {
                if (W.lofs[L + 1] == W.lofs[L]) continue;  // no particle of this level
                __syncthreads();  // every lane is done with rs before it is built again
                row_stencil_wide<true>(g, W, L, (uint32_t)c >> (3 * (g.level - L)), 0.0, 0.0, 0.0, -1.0, rs);
                const int total = rs.pref[rs.nst];
                for (v0 = 0; v0 < total; v0 += 64) {
                    keep = false;
                    double xj = 0, yj = 0, zj = 0, hj = 0;
                    if (v0 + t < total) {
                        j = W.lidx[row_candidate(rs, v0 + t)];
                        if (outside(W.key[j])) {
                            xj = X[j]; yj = Y[j]; zj = Z[j]; hj = H[j];
                            keep = !culled(rel(xj, hx), rel(yj, hy), rel(zj, hz), (float)(hj * inv_cell), 0.0f);
                        }
                    }
                    for (unsigned long long m = __ballot(keep); m; m &= m - 1) {
                        const int k = __ffsll((long long)m) - 1, jj = lane_value(j, k);
                        const double xk = lane_value(xj, k), yk = lane_value(yj, k), zk = lane_value(zj, k), hk = lane_value(hj, k);
                        if (!on || jj == i || !accept_pair<true>(xi, yi, zi, xk, yk, zk, hi, hk, g.box, g.half)) continue;
                        if (n < cap) {
                            int q = n;
                            while (q > 0 && ell[ell_at(ld, r, q - 1)] > jj) { ell[ell_at(ld, r, q)] = ell[ell_at(ld, r, q - 1)]; q--; }
                            ell[ell_at(ld, r, q)] = jj;
                        }
                        n++;
                    }
                }
            }
        }
        if (on) {
            cnt[r] = min(n, cap);  // readers stay inside the list; the overflow carries the full length
            if (n > cap) atomicMax(overflow, n);
        }
        __syncthreads();  // before the next rows' ranges
    }
}
#endif


// ---------------------------------------------------------------------------------------
// groups of rows sharing one cell of one grid, for the cell walks of the search over many
// levels (the cell of the level of each row's radius) and of batches (the cell of the row's
// box): key = the level's or the box's first table entry + the cell code
// ---------------------------------------------------------------------------------------
#ifdef GZ_DEFINE_COMMON_KERNELS
__global__ void __launch_bounds__(256) k_row_group_key(int nrows, const int *__restrict__ act, const uint8_t *__restrict__ need,
                                                        const uint32_t *__restrict__ key, const double *__restrict__ hslot,
                                                        const double *__restrict__ H, double box, double margin,
                                                        const WideGrid *__restrict__ W, BoxTable bt, uint32_t *__restrict__ gkey,
                                                        int *__restrict__ val)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    if (val) val[r] = r;
    if (need && !need[r]) { gkey[r] = 0xffffffffu; return; }  // not in this pass: after every group
    const int i = act[r];
    if (bt.b) {
        const BoxDev &B = bt.b[bt.BOX[i]];
        gkey[r] = (uint32_t)(B.cell_off + (key[i] >> B.shift));
    } else {
        const double h = hslot ? hslot[r] : H[i];
        const int L = wide_level(box, W->lmax, h + 2.0 * margin);
        gkey[r] = (uint32_t)(W->loff[L] + (key[i] >> (3 * (kFineLevel - L))));
    }
}

// group heads of the sorted keys (flag[nrows] = 0 for the scan)
__global__ void __launch_bounds__(256) k_group_heads(int nrows, const uint32_t *__restrict__ skey, int *__restrict__ flag)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > nrows) return;
    flag[p] = (p < nrows && skey[p] != 0xffffffffu && (p == 0 || skey[p - 1] != skey[p])) ? 1 : 0;
}

// group starts (positions in the sorted rows), keys and count; gstart[count] = the number of
// rows in groups
__global__ void __launch_bounds__(256) k_group_list(int nrows, const uint32_t *__restrict__ skey, const int *__restrict__ flag,
                                                     const int *__restrict__ scan, int *__restrict__ gstart, uint32_t *__restrict__ gkey,
                                                     int *__restrict__ ngroups)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nrows) return;
    if (flag[p]) { gstart[scan[p]] = p; gkey[scan[p]] = skey[p]; }
    const bool last = skey[p] != 0xffffffffu && (p + 1 == nrows || skey[p + 1] == 0xffffffffu);
    if (last) { gstart[scan[p] + flag[p]] = p + 1; *ngroups = scan[p] + flag[p]; }
    if (p == 0 && skey[0] == 0xffffffffu) { gstart[0] = 0; *ngroups = 0; }
}

// the stencil of every group (one wavefront each): the 27 cells around its cell at its level,
// duplicates dropped, ascending code (ascending start)
__global__ void __launch_bounds__(64) k_group_stencil(GridView g, int ngroups, const uint32_t *__restrict__ gkey,
                                                       const int *__restrict__ gstart, const int *__restrict__ grow,
                                                       const int *__restrict__ act, BoxTable bt, int *__restrict__ glev,
                                                       int *__restrict__ gcode, int *__restrict__ gnst, int4 *__restrict__ gsten)
{
    __shared__ RowStencil rs;
    const long gb = blockIdx.x;
    if (gb >= ngroups) return;
    const uint32_t k = gkey[gb];
    int L, c;
    if (bt.b) {
        DevParams P{};
        resolve_box(bt, act[grow ? grow[gstart[gb]] : gstart[gb]], P, g);
        L = g.level;
        c = (int)(k - g.cell_off);
        row_stencil<false>(g, (uint32_t)c, 0.0, 0.0, 0.0, 1e300, rs);
    } else {
        const WideGrid &W = *g.wide;
        L = 0;
        while (L < W.lmax && (long long)k >= W.loff[L + 1]) L++;
        c = (int)(k - W.loff[L]);
        row_stencil_wide<false>(g, W, L, (uint32_t)c, 0.0, 0.0, 0.0, -1.0, rs);
    }
    const int lane = threadIdx.x;
    if (lane < rs.nst) gsten[(size_t)27 * gb + lane] = make_int4(rs.start[lane], rs.start[lane] + rs.len[lane], 0, 0);
    if (lane == 0) { glev[gb] = L; gcode[gb] = c; gnst[gb] = rs.nst; }
}
#endif

// gradients of few rows: the terms of each list entry in LDS, accumulated in list order by lane 0
template <int KERN, typename R, int TPB>
__global__ void __launch_bounds__(TPB) k_gradients_rows(DevParams P, int nrows, const int *__restrict__ act, const double *__restrict__ X,
                                                       const double *__restrict__ Y, const double *__restrict__ Z,
                                                       const double *__restrict__ H, const GradRec<R> *__restrict__ rec, GradSrc src, const double *__restrict__ T,
                                                       const double *__restrict__ CN, long n, const int *__restrict__ ell, long ld,
                                                       const int *__restrict__ cnt, double *__restrict__ GR, double *__restrict__ GP,
                                                       double *__restrict__ GV, BoxTable bt, int *__restrict__ force_flags)
{
    // the accepted entries' values packed in list order (padded rows: no bank conflicts)
    __shared__ R sd[5][TPB + 1], sw[3][TPB + 1], srr[TPB + 1];
    __shared__ unsigned long long smask[TPB / 64];
    const long r = xcd_block();
    // the coming force pass's error and wake-up flags (its records are made in its own kernel)
    if (r == 0 && threadIdx.x == 0 && force_flags) force_flags_clear(force_flags);
    if (r >= nrows) return;
    const int lane = threadIdx.x;  // thread of the workgroup
    const int i = act[r];
    {
        GridView g{};
        resolve_box(bt, i, P, g);
    }
    R G[3][5];
    R mx[5], mn[5];
    R maxd = 0;
    R acc = 0;  // the running quantity this lane keeps
    // records packed by an earlier launch, or made here from the state (few rows among many
    // particles: no packing launch)
    const GradRec<R> I = src.H ? make_grad_rec<R>(i, src, X, Y, Z, bt) : rec[i];
    const bool enabled = (I.m > 0 && I.rho > 0);
    const R hi = I.h;
    if (enabled) {
        const double xi = X[i], yi = Y[i], zi = Z[i];
        // the row's radius in FP64 (the kernel's edge factor, pair_kernel)
        const double hid = std::is_same<R, double>::value ? (double)hi : H[i];
        const double h2i = hid * hid;
        const int c = cnt[r];
        for (int base = 0; base < c; base += TPB) {
            const int q = base + lane;
            bool ok = false;
            R w3[3] = {0, 0, 0}, d5[5], rr = 0;
            if (q < c) {
                const int j = ell[ell_at(ld, r, q)];
                const GradRec<R> J = src.H ? make_grad_rec<R>(j, src, X, Y, Z, bt) : rec[j];
                if ((J.m > 0) && (J.rho > 0) && (J.h > 0)) {
                    R dp[3];
                    record_dp<R>(P, I, J, xi, yi, zi, X, Y, Z, j, dp[0], dp[1], dp[2]);
                    const R r2 = dp[0] * dp[0] + dp[1] * dp[1] + dp[2] * dp[2];
                    const double r2d = pair_r2d<R>(dp[0], dp[1], dp[2], r2);
                    if ((r2 > 0) && !((r2d >= h2i) && (r2d >= (double)J.h * (double)J.h))) {
                        rr = sqrt(r2);
                        const double rd = std::is_same<R, double>::value ? 0.0 : sqrt(r2d);
                        R wk = 0, dwk = 0;
                        ok = true;
                        // an entry beyond the row's own radius (inside the neighbour's) takes part
                        // in the extrema only: its weights stay +0, and its products (+-0) leave
                        // the gradient sums, which start at +0 and never reach -0, unchanged
                        if (std::is_same<R, double>::value ? (rr < hi) : (rd < hid)) {
                            pair_kernel<KERN, -1, R>(rr, rd, hid, wk, dwk);
                            for (int kk = 0; kk < 3; kk++) w3[kk] = -wk * dp[kk];
                        }
                        d5[0] = (R)(J.rho - I.rho);
                        d5[1] = (R)(J.p - I.p);
                        d5[2] = (R)(J.v0 - I.v0);
                        d5[3] = (R)(J.v1 - I.v1);
                        d5[4] = (R)(J.v2 - I.v2);
                    }
                }
            }
            // the accepted entries packed in list order; threads 0-14 then keep G[kk][b]
            // (kk = lane/5, b = lane%5), 15-19 the minima, 20-24 the maxima, 25 the largest
            // distance (with mn <= 0 <= mx the reference's else-if is two ifs)
            int nok;
            const int pos = flagged_rank<TPB>(ok, smask, nok);
            if (ok) {
                for (int kk = 0; kk < 3; kk++) sw[kk][pos] = w3[kk];
                for (int b = 0; b < 5; b++) sd[b][pos] = d5[b];
                srr[pos] = rr;
            }
            __syncthreads();
            if (lane < 15) {
                const R *a = sw[lane / 5], *b = sd[lane % 5];
                int k = 0;
                for (; k + 4 <= nok; k += 4) {
                    const R p0 = rounded(a[k] * b[k]), p1 = rounded(a[k + 1] * b[k + 1]);
                    const R p2 = rounded(a[k + 2] * b[k + 2]), p3 = rounded(a[k + 3] * b[k + 3]);
                    acc = acc + p0;
                    acc = acc + p1;
                    acc = acc + p2;
                    acc = acc + p3;
                }
                for (; k < nok; k++) acc = acc + rounded(a[k] * b[k]);
            } else if (lane < 26) {
                // minima (15-19, as maxima of the negated values: exact), maxima, distance
                const R *a = lane < 25 ? sd[(lane - 15) % 5] : srr;
                const bool mn = lane < 20;
                R m = mn ? -acc : acc;
                for (int k = 0; k < nok; k++) {
                    const R d = mn ? -a[k] : a[k];
                    if (d > m) m = d;
                }
                acc = mn ? -m : m;
            }
            __syncthreads();
        }
    }
    __shared__ R res[26];
    if (lane < 26) res[lane] = acc;
    __syncthreads();
    if (lane == 0) {
        for (int kk = 0; kk < 3; kk++)
            for (int b = 0; b < 5; b++) G[kk][b] = res[kk * 5 + b];
        for (int b = 0; b < 5; b++) { mn[b] = res[15 + b]; mx[b] = res[20 + b]; }
        maxd = res[25];
        gradients_tail<R>(I, enabled, G, mx, mn, maxd, T, CN, n, i, GR, GP, GV);
    }
}

// force of few rows: each lane evaluates one list entry (hydro_accumulate_neighbor), lane 0
// accumulates in list order, then the writeback and final operations
template <int KERN, typename R, bool STATS, int TPB, bool MAKE>
__global__ void __launch_bounds__(TPB) k_force_rows(DevParams P, Gam<R> G, int nrows, const int *__restrict__ act, ForceView F,
                                                   const Cell<R> *__restrict__ rec, const int *__restrict__ ell, long ld,
                                                   const int *__restrict__ cnt, const uint8_t *__restrict__ active,
                                                   const int *__restrict__ timebin, const double *__restrict__ msv_in,
                                                   int *__restrict__ wakeup, double *__restrict__ ACC, double *__restrict__ DTU,
                                                   double *__restrict__ MSV, int *__restrict__ err, int *__restrict__ need_wakeup,
                                                   unsigned long long *__restrict__ pairs, BoxTable bt, const int *__restrict__ gate)
{
    __shared__ R sv[5][TPB + 1];  // the entries' fluxes packed in list order (padded: no bank conflicts)
    __shared__ unsigned long long smask[TPB / 64];
    const long r = xcd_block();
    if (r >= nrows) return;
    if (gate && *gate) return;  // the density round behind this launch did not stand (its gate word)
    const int lane = threadIdx.x;  // thread of the workgroup
    const int i = act[r];
    {
        GridView g{};
        resolve_box(bt, i, P, g);
    }
    const double mi = F.M[i], rhoi = F.RHO[i];
    constexpr bool make = MAKE;
    double A0 = 0, A1 = 0, A2 = 0, dE = 0, msv = 0;
    const double sound_i = (rhoi > 0) ? sqrt(P.gamma * F.PR[i] / rhoi) : sqrt(P.gamma * (P.gamma - 1.) * F.U[i]);
    const bool enabled = (mi > 0 && rhoi > 0);
    const int c = cnt[r];
    if (lane == 0 && wakeup) wakeup[i] = 0;  // hydro_force_initial_operations_preloop
    if (enabled) {
        const Cell<R> I = make ? force_rec_of<R>(i, P.gamma, F, P.box, bt) : rec[i];
        const double xi = F.X[i], yi = F.Y[i], zi = F.Z[i];
        const int tbi = timebin ? timebin[i] : 0;
        // lanes 0-3 keep the momentum and energy sums, lane 4 the signal speed: max(c_s, vsig)
        // over the entries (the reference raises it to c_s before each entry, a no-op after the first)
        R acc = 0;       // lane 4
        CSum<R> sum;     // lanes 0-3
        if (lane == 4 && c > 0) acc = (acc < I.cs) ? I.cs : acc;
        for (int base = 0; base < c; base += TPB) {
            const int q = base + lane;
            int rc = 0;
            R f0, f1, f2, fp, vts;
            if (q < c) {
                const int j = ell[ell_at(ld, r, q)];
                const Cell<R> J = make ? force_rec_of<R>(j, P.gamma, F, P.box, bt) : rec[j];
                R dp0, dp1, dp2;
                record_dp<R>(P, I, J, xi, yi, zi, F.X, F.Y, F.Z, j, dp0, dp1, dp2);
                const R r2 = dp0 * dp0 + dp1 * dp1 + dp2 * dp2;
                unsigned rung;
                rc = force_pair<KERN, R>(P, G, I, J, dp0, dp1, dp2, r2, f0, f1, f2, fp, vts, rung);
                if constexpr (STATS) count_rungs(F.rungs, rung);
                if (rc < 0) {
                    atomicMax(err, 1234);
                    if (atomicCAS(err + 10, -1, i) == -1) err[11] = j;
                }
                if (rc > 0) {
                    if (active && !active[j] && wakeup) {
                        if ((double)vts > kWakeup * msv_in[j]) {
                            atomicMax(&wakeup[j], tbi + 1);
                            if (bt.b) bt.b[bt.BOX[i]].need_wakeup = 1;
                            else *need_wakeup = 1;
                        }
                    }
                }
            }
            // the entries with a flux packed in list order; lanes 0-4 then take them in turn
            int nok;
            const int pos = flagged_rank<TPB>(rc > 0, smask, nok);
            if (rc > 0) {
                sv[0][pos] = f0; sv[1][pos] = f1; sv[2][pos] = f2; sv[3][pos] = fp; sv[4][pos] = vts;
            }
            __syncthreads();
            if (lane < 4) {
                const R *a = sv[lane];
                int k = 0;
                for (; k + 4 <= nok; k += 4) {
                    const R x0 = a[k], x1 = a[k + 1], x2 = a[k + 2], x3 = a[k + 3];
                    sum.add(x0);
                    sum.add(x1);
                    sum.add(x2);
                    sum.add(x3);
                }
                for (; k < nok; k++) sum.add(a[k]);
            } else if (lane == 4) {
                for (int k = 0; k < nok; k++)
                    if (sv[4][k] > acc) acc = sv[4][k];
            }
            __syncthreads();
        }
        __shared__ double res[5];
        if (lane < 4) res[lane] = sum.value();
        if (lane == 4) res[lane] = (double)acc;
        __syncthreads();
        A0 = res[0]; A1 = res[1]; A2 = res[2]; dE = res[3]; msv = res[4];
    }
    if (lane == 0) {
        force_tail(P, F, i, enabled, sound_i, A0, A1, A2, dE, msv, ACC, DTU, MSV);
        // the pairs of the row last: no load of the row waits behind the atomic
        if (c && pairs) atomicAdd(pairs, (unsigned long long)c);
    }
}

}  // namespace gz
