// search_kernels.hip -- searchNeighbors (reference src/simulator.cu:60-178).
//
//   k_s_cells   : wrap positions into the box on periodic axes, cell id of
//                 every bubble, cell counts (reference wrapOverPeriodicBoundaries
//                 src/kernels.cu:992-1011, cellByPosition :598-607)
//   k_s_scan1   : per-block cell-count sums
//   k_s_scan2   : cell offsets (exclusive scan), cursors, counts reset
//                 (reference: cub::DeviceScan::InclusiveSum, simulator.cu:90-91)
//   k_s_bin     : bubbles into unsorted cell segments (reference indexByCell
//                 src/kernels.cu:609-615)
//   k_s_reorder : each bubble ranks itself among its cell's members by old
//                 index (a stable counting sort, where the reference's
//                 atomic order is arbitrary) and scatters its whole state to
//                 its new slot in the alternate buffers; saved <- current
//                 (reference reorganizeByIndex :721-770)
//   k_s_search  : full neighbour list of every bubble, ascending, over the
//                 de-duplicated 3^D cell neighbourhood: 32 x 32 pairs per
//                 matrix instruction, decided as in FP64 (reference neighborSearch / comparePair
//                 src/kernels.cu:617-701 with getNeighborCellIndex
//                 :1116-1189); the reference's half list is the subset j > i.
//                 Counts beyond the list capacity are reported, never written
//                 out of bounds.
//   k_s_fin     : one block per foam makes the reordered buffers current
//                 (the pointer rotation of simulator.cu:96-147) and totals the
//                 pair count
#include <type_traits>

#include "dev_util.hpp"
#include "launch.hpp"

namespace cubble_amd {

// Runs of equal keys among the wave's valid lanes (bubbles are in the cell
// order of the previous search, so neighbouring lanes mostly share a cell):
// `heads` has a bit for the first lane of each run; a head's run ends at the
// next head or at the last valid lane.  One atomic per run instead of one per
// bubble.
struct WaveRuns {
    unsigned long long heads;
    int len;   // run length (valid on head lanes)
    int head;  // lane of this lane's run head
};

__device__ __forceinline__ WaveRuns wave_runs(int key, bool valid) {
    const int lane = (int)(threadIdx.x & 63);
    const int prev = __shfl_up(key, 1);
    const bool is_head = valid && (0 == lane || prev != key);
    const unsigned long long heads = __builtin_amdgcn_ballot_w64(is_head);
    const unsigned long long vmask = __builtin_amdgcn_ballot_w64(valid);
    // valid lanes are a prefix of the wave (consecutive bubbles below n)
    const int nvalid = __popcll(vmask);
    const unsigned long long above = lane < 63 ? heads & (~0ull << (lane + 1)) : 0ull;
    const int end = above ? __builtin_ctzll(above) : nvalid;
    const unsigned long long upto = heads & (lane < 63 ? (2ull << lane) - 1ull : ~0ull);
    WaveRuns r;
    r.heads = heads;
    r.len = end - lane;
    r.head = upto ? 63 - __builtin_clzll(upto) : 0;
    return r;
}

template <int D>
__device__ __forceinline__ double cells_range(const Consts &c, const Roles &R, const Scratch &S,
                                              const int cd[3], int base, int ipt, int n) {
    double rmax = 0.0;
    for (int k = 0; k < ipt; ++k) {
        if (base + k * kBlock >= n) break;  // uniform per block
        const int i = base + k * kBlock + (int)threadIdx.x;
        const bool valid = i < n;
        int cid = -1;
        if (valid) {
            double p[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < D; ++q) {
                double xv = R.x[q][i];
                if (!c.wall[q]) {
                    const int mult = xv < c.lbb[q] ? 1 : (xv > c.tfr[q] ? -1 : 0);
                    xv = xv + (c.tfr[q] - c.lbb[q]) * (double)mult;
                    R.x[q][i] = xv;
                    if (mult) R.wc[q][i] -= mult;
                }
                p[q] = xv;
            }
            int id[3] = {0, 0, 0};
#pragma unroll
            for (int q = 0; q < D; ++q) {
                const double f = floor(cd[q] * (p[q] - c.lbb[q]) / c.interval[q]);
                id[q] = f < 0.0 ? 0 : (f >= (double)cd[q] ? cd[q] - 1 : (int)f);
            }
            cid = id[2] * cd[0] * cd[1] + id[1] * cd[0] + id[0];
            S.cell_of[i] = cid;
            rmax = fmax(rmax, R.x[3][i]);
        }
        const WaveRuns wr = wave_runs(cid, valid);
        if (valid && (int)(threadIdx.x & 63) == wr.head) atomicAdd(&S.cell_count[cid], wr.len);
    }
    return rmax;
}

__global__ __launch_bounds__(kBlock) void k_s_cells(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_search) return;
    const Consts c = F->c;
    const Roles R = F->r;
    const Scratch S = F->s;
    const int n = F->d.count, ipt = F->ipt;
    int cd[3];
    cell_dims(c, F->d.max_r_cell, F->cell_cap, cd);
    const int base = cx.lb * kBlock * ipt;
    double rmax = 3 == c.dim ? cells_range<3>(c, R, S, cd, base, ipt, n)
                             : cells_range<2>(c, R, S, cd, base, ipt, n);
    // largest radius of the foam, for the search's reach bound: radii are
    // positive, so their bit patterns order like the values
    rmax = block_max(rmax);
    if (0 == threadIdx.x && rmax > 0.0)
        atomicMax(reinterpret_cast<unsigned long long *>(&F->d.search_max_r),
                  (unsigned long long)__double_as_longlong(rmax));
    // every block computed the same grid; no block of this kernel reads it back
    if (0 == cx.lb && 0 == threadIdx.x) {
        F->d.cell_dim[0] = cd[0];
        F->d.cell_dim[1] = cd[1];
        F->d.cell_dim[2] = cd[2];
        F->d.num_cells = cd[0] * cd[1] * cd[2];
    }
}

__global__ __launch_bounds__(kBlock) void k_s_scan1(Foam *foams, const int2 *bt) {
    const Ctx cx = cell_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_search) return;
    const Scratch S = F->s;
    const int ncell = F->d.num_cells, cipt = F->cipt;
    const int base = cx.lb * kBlock * cipt;
    int s = 0;
    for (int k = 0; k < cipt; ++k) {
        const int q = base + k * kBlock + (int)threadIdx.x;
        if (q < ncell) s += S.cell_count[q];
    }
    s = block_sum_i(s);
    if (threadIdx.x == 0) S.cpart[cx.lb] = s;
}

// Cell offsets: each block sums the block totals before it (at most a few
// hundred ints), then scans its own cells.  The block holding the last cell
// also writes start[num_cells].
__global__ __launch_bounds__(kBlock) void k_s_scan2(Foam *foams, const int2 *bt) {
    const Ctx cx = cell_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_search) return;
    const Scratch S = F->s;
    const int ncell = F->d.num_cells, cipt = F->cipt;
    const int base = cx.lb * kBlock * cipt;
    if (base >= ncell) return;  // uniform per block
    int acc = 0;
    for (int b = threadIdx.x; b < cx.lb; b += kBlock) acc += S.cpart[b];
    int off = block_sum_i(acc);
    for (int k = 0; k < cipt; ++k) {
        const int q = base + k * kBlock + (int)threadIdx.x;
        const int v = q < ncell ? S.cell_count[q] : 0;
        int tot = 0;
        const int pre = block_excl_scan(v, tot);
        if (q < ncell) {
            S.cell_start[q] = off + pre;
            S.cell_cursor[q] = off + pre;
            S.cell_count[q] = 0;
        }
        off += tot;
    }
    if (ncell - 1 < base + kBlock * cipt && threadIdx.x == 0) S.cell_start[ncell] = off;
}

__global__ __launch_bounds__(kBlock) void k_s_bin(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_search) return;
    const Scratch S = F->s;
    const int n = F->d.count, ipt = F->ipt;
    const int base = cx.lb * kBlock * ipt;
    for (int k = 0; k < ipt; ++k) {
        if (base + k * kBlock >= n) break;  // uniform per block
        const int i = base + k * kBlock + (int)threadIdx.x;
        const bool valid = i < n;
        const int cid = valid ? S.cell_of[i] : -1;
        // one atomic per run of equal cells; the run's lanes take consecutive
        // slots (the order inside a cell segment does not matter: the reorder
        // ranks by old index)
        const WaveRuns wr = wave_runs(cid, valid);
        const int lane = (int)(threadIdx.x & 63);
        int slot = 0;
        if (valid && lane == wr.head) slot = atomicAdd(&S.cell_cursor[cid], wr.len);
        slot = __shfl(slot, wr.head) + (lane - wr.head);
        if (valid) S.members[slot] = i;
    }
}

template <int D, typename V>
__device__ __forceinline__ void reorder_range(const Roles &R, const Scratch &S, int base, int ipt,
                                              int n) {
    for (int k = 0; k < ipt; ++k) {
        const int i = base + k * kBlock + (int)threadIdx.x;
        if (i >= n) break;
        const int c = S.cell_of[i];
        const int s0 = S.cell_start[c], s1 = S.cell_start[c + 1];
        // rank among the cell's members by old index; the members are loaded
        // eight at a time (independent loads: crowded cells hold a hundred
        // bubbles and more)
        int rank = 0;
        for (int s = s0; s < s1; s += 8) {
            int mb[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) mb[u] = s + u < s1 ? S.members[s + u] : i;
#pragma unroll
            for (int u = 0; u < 8; ++u) rank += mb[u] < i ? 1 : 0;
        }
        const int np = s0 + rank;
        double xs[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (2 == q && 2 == D) continue;
            const double xv = R.x[q][i];
            xs[q] = xv;
            R.xp[q][np] = xv;
            field<V>(R.saved[q])[np] = (V)xv;
            field<V>(R.vp[q])[np] = field<V>(R.v[q])[i];
            field<V>(R.vs[q])[np] = field<V>(R.vo[q])[i];
        }
        S.x4[np] = D4{xs[0], xs[1], xs[2], xs[3]};
        R.path_new[np] = R.path[i];
        field<V>(R.err_alt)[np] = field<V>(R.err)[i];
#pragma unroll
        for (int q = 0; q < D; ++q) R.wc_alt[q][np] = R.wc[q][i];
        R.idx_alt[np] = R.idx[i];
    }
}

__global__ __launch_bounds__(kBlock) void k_s_reorder(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_search) return;
    const Roles R = F->r;
    const Scratch S = F->s;
    const int n = F->d.count, ipt = F->ipt;
    const int base = cx.lb * kBlock * ipt;
    const bool fvel = CUBBLE_PREC_MIXED == F->precision;  // FP32 velocities
    if (3 == F->c.dim) {
        if (fvel) reorder_range<3, float>(R, S, base, ipt, n);
        else reorder_range<3, double>(R, S, base, ipt, n);
    } else {
        if (fvel) reorder_range<2, float>(R, S, base, ipt, n);
        else reorder_range<2, double>(R, S, base, ipt, n);
    }
}

// After the reorder the new state sits in the alternate buffers; k_s_fin
// makes them current.
__device__ void swap_reordered_roles(Roles &W) {
    for (int q = 0; q < 4; ++q) {
        double *t = W.x[q];
        W.x[q] = W.xp[q];
        W.xp[q] = t;
        void *u = W.v[q];
        W.v[q] = W.vp[q];
        W.vp[q] = u;
        u = W.vo[q];
        W.vo[q] = W.vs[q];
        W.vs[q] = u;
    }
    double *t = W.path;
    W.path = W.path_new;
    W.path_new = t;
    void *e = W.err;
    W.err = W.err_alt;
    W.err_alt = e;
    for (int q = 0; q < 3; ++q) {
        int *u = W.wc[q];
        W.wc[q] = W.wc_alt[q];
        W.wc_alt[q] = u;
    }
    int *u = W.idx;
    W.idx = W.idx_alt;
    W.idx_alt = u;
}

// Sorted, de-duplicated neighbour coordinates of cell coordinate `x` along
// one axis: periodic axes wrap, wall axes drop out-of-range cells.  With
// fewer than 3 cells the wrapped offsets coincide and appear once.  Held in
// three named values, not an array, so no kernel indexes private memory.
struct AxisCells {
    int v0, v1, v2, n;
    __device__ __forceinline__ int at(int k) const { return 0 == k ? v0 : 1 == k ? v1 : v2; }
};

__device__ __forceinline__ AxisCells axis_cells(int x, int n, bool wall) {
    AxisCells r;
    if (wall) {
        const bool lo = x - 1 >= 0, hi = x + 1 < n;
        r.v0 = lo ? x - 1 : x;
        r.v1 = lo ? x : x + 1;
        r.v2 = x + 1;
        r.n = 1 + (lo ? 1 : 0) + (hi ? 1 : 0);
        return r;
    }
    int v0 = (x - 1 + n) % n, v1 = x, v2 = (x + 1) % n, t;
    if (v0 > v1) { t = v0; v0 = v1; v1 = t; }
    if (v1 > v2) { t = v1; v1 = v2; v2 = t; }
    if (v0 > v1) { t = v0; v0 = v1; v1 = t; }
    // drop duplicates, keeping order
    const bool d1 = v1 == v0, d2 = v2 == v1;
    r.v0 = v0;
    r.v1 = d1 ? v2 : v1;
    r.v2 = v2;
    r.n = 3 - (d1 ? 1 : 0) - (d2 ? 1 : 0);
    return r;
}

// The x-cells of one row as at most two runs of consecutive cells,
// [a0, b0] and (if two) [a1, b1], in ascending order.
struct XRuns {
    int a0, b0, a1, b1;
    bool two;
};

__device__ __forceinline__ XRuns x_runs(const AxisCells &X) {
    int f0 = 0;
    if (X.n > 1 && X.v1 == X.v0 + 1) f0 = 1;
    if (1 == f0 && X.n > 2 && X.v2 == X.v1 + 1) f0 = 2;
    XRuns r;
    r.a0 = X.v0;
    r.b0 = X.at(f0);
    r.two = f0 + 1 < X.n;
    r.a1 = r.two ? X.at(f0 + 1) : 0;
    r.b1 = r.two ? X.at(X.n - 1) : -1;
    return r;
}

// The x-cells [x0 - 1, x0 + k] around k consecutive own cells x0 .. x0 + k - 1
// of one row, as at most two runs in ascending order, each with its image
// code as `side` gives it for a neighbour cell (0; 1: the run lies past the
// high end, its candidates take d - L; 2: past the low end, d + L).  On a
// periodic axis k + 4 <= n, so the window wraps at one end at most and a
// cell appears once.  A pair of cells more than one apart in the window is
// at least a cell width apart under either image, so it never holds a pair
// within reach.
struct XWindow {
    int a0, b0, f0, a1, b1, f1;
    bool two;
};

__device__ __forceinline__ XWindow x_window(int x0, int k, int n, bool wall) {
    XWindow r{x0 - 1, x0 + k, 0, 0, -1, 0, false};
    if (wall) {
        r.a0 = max(r.a0, 0);
        r.b0 = min(r.b0, n - 1);
    } else if (x0 - 1 < 0) {  // [0, x0 + k], then cell n - 1 past the low end
        r = XWindow{0, x0 + k, 0, n - 1, n - 1, 2, true};
    } else if (x0 + k >= n) {  // cells past the high end first, then [x0 - 1, n - 1]
        r = XWindow{0, x0 + k - n, 1, x0 - 1, n - 1, 0, true};
    }
    return r;
}

// Wave-uniform append of the ballot `m` (non-zero) of candidates j to own
// bubble i's list.  Lane `ii` of the group (ii is wave-uniform) keeps the
// count: it is read with readlane and updated on the scalar unit.  A hit
// lane's slot is the count plus the hits in the lanes below it (mbcnt); the
// hit itself is re-derived from `m`, so the comparison result need not stay
// live across the branch.
__device__ __forceinline__ void append_hits(unsigned long long m, int ii, int i, int j,
                                            int *__restrict__ nbr_, unsigned cap, int nbr_cap,
                                            int &cnt) {
    const int base = __builtin_amdgcn_readlane(cnt, ii);
    const int upd = base + __popcll(m);  // scalar
    // the hit lanes become the exec mask directly (no per-lane bit test)
    if (__builtin_amdgcn_inverse_ballot_w64(m)) {
        const int below = (int)__builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        const int pos = base + below;
        auto nbr = (__attribute__((address_space(1))) int *)(nbr_ + i);
        // slots past the capacity are counted, not written; when all fit (a
        // scalar test) the bound is one no slot reaches
        const int lim = upd <= nbr_cap ? 0x7fffffff : nbr_cap;
        if (pos < lim) nbr[(uint64_t)(unsigned)pos * cap] = j;
    }
    cnt = (int)(threadIdx.x & 63) == ii ? upd : cnt;  // lane ii keeps the count
}

// The list length goes to nn and, as the degree the imposed flow divides by,
// to deg (which a removal moves but does not reduce).
__device__ __forceinline__ void finish_group(int cb, int nb, int cnt, int nbr_cap,
                                             int *__restrict__ nn, int *__restrict__ deg,
                                             int &sum_nn, int &max_nn, int &ovf) {
    if ((int)(threadIdx.x & 63) < nb) {
        const int v = cnt < nbr_cap ? cnt : nbr_cap;
        nn[cb + (int)(threadIdx.x & 63)] = v;
        deg[cb + (int)(threadIdx.x & 63)] = v;
        sum_nn += cnt;
        max_nn = max(max_nn, cnt);
        if (cnt > nbr_cap) ovf = 1;
    }
}

// Neighbour lists, one wavefront per cell, any box (the general path).
// The linear cell id z*cx*cy + y*cx + x grows lexicographically in
// (z, y, x), so walking the sorted per-axis cell lists in that nesting
// visits cells -- and, since bubbles are stored in cell order, candidates --
// in ascending index order; consecutive x-cells of one row form one
// contiguous run of bubbles.  The 64 lanes take 64 consecutive candidates of
// a run (one coalesced 32-byte record each); the cell's own bubbles are
// wave-uniform scalar loads; hits are found with a wave ballot and appended
// to that bubble's list in lane order, which keeps every list ascending.
// Lists longer than the capacity are counted, never written out of bounds.
// `cell` must be wave-uniform.  A function of its own: its loops would raise
// the register use of the common path.
struct ListTotals {
    int sum_nn, max_nn, ovf;
};

template <int D>
__device__ __forceinline__ ListTotals search_cell_general(const Foam *F, int cell,
                                                                    int i0, int i1) {
    const Consts &c = F->c;
    const auto x4 = gmem(F->s.x4);
    const auto x4s = cmem(F->s.x4);
    const auto start = cmem(F->s.cell_start);
    int *const nbr = F->s.nbr;
    const int cd[3] = {F->d.cell_dim[0], F->d.cell_dim[1], F->d.cell_dim[2]};
    const size_t cap = (size_t)F->cap;
    const int nbr_cap = F->nbr_cap;
    ListTotals sum{0, 0, 0};
    const int lane = (int)(threadIdx.x & 63);
    cell = uniform_i(cell);
    i0 = uniform_i(i0);
    i1 = uniform_i(i1);
    if (i0 >= i1) return sum;
    const int ccx = cell % cd[0];
    const int ccy = (cell / cd[0]) % cd[1];
    const int ccz = cell / (cd[0] * cd[1]);
    const AxisCells X = axis_cells(ccx, cd[0], c.wall[0] != 0);
    const AxisCells Y = axis_cells(ccy, cd[1], c.wall[1] != 0);
    const AxisCells Z = 3 == D ? axis_cells(ccz, cd[2], c.wall[2] != 0) : AxisCells{0, 0, 0, 1};
    const XRuns xr = x_runs(X);
    const double skin = c.skin;
    for (int cb = i0; cb < i1; cb += 64) {
        const int nb = uniform_i(min(64, i1 - cb));
        int cnt = 0;
#pragma unroll 1
        for (int a = 0; a < 3; ++a) {
#pragma unroll 1
            for (int b = 0; b < 3; ++b) {
#pragma unroll 1
                for (int part = 0; part < 2; ++part) {
                    if (a >= Z.n || b >= Y.n || (1 == part && !xr.two)) continue;
                    const int row = Z.at(a) * cd[0] * cd[1] + Y.at(b) * cd[0];
                    const int j0 = start[row + (0 == part ? xr.a0 : xr.a1)];
                    const int j1 = start[row + (0 == part ? xr.b0 : xr.b1) + 1];
                    for (int jb = j0; jb < j1; jb += 64) {
                        const int j = jb + lane;
                        const bool valid = j < j1;
                        const unsigned long long vmask = __builtin_amdgcn_ballot_w64(valid);
                        const int jl = valid ? j : j0;
                        const D4 pj = D4{x4[jl].x, x4[jl].y, 3 == D ? x4[jl].z : 0.0, x4[jl].r};
                        for (int ii = 0; ii < nb; ++ii) {
                            const int i = cb + ii;
                            const double px = x4s[i].x, py = x4s[i].y, pr = x4s[i].r;
                            const double pz = 3 == D ? x4s[i].z : 0.0;
                            const double maxd = pr + pj.r + skin;
                            double d[3];
                            wrapped_diff<D>(c, px, py, pz, pj.x, pj.y, pj.z, d);
                            // one ballot per comparison: each is the comparison's own
                            // lane mask, with no boolean materialised in a register
                            const unsigned long long m =
                                vmask & __builtin_amdgcn_ballot_w64(j != i) &
                                __builtin_amdgcn_ballot_w64(sq_len(d) < maxd * maxd);
                            if (m) append_hits(m, ii, i, j, nbr, (unsigned)cap, nbr_cap, cnt);
                        }
                    }
                }
            }
        }
        finish_group(cb, nb, cnt, nbr_cap, F->s.nn, F->s.deg, sum.sum_nn, sum.max_nn, sum.ovf);
    }
    return sum;
}

constexpr int kMaxRuns = 18;    // 3 z-rows x 3 y-rows x 2 x-runs
constexpr int kOwnUnit = 32;    // own bubbles per work unit of the general path
constexpr int kSub = 32;        // own bubbles per matrix tile
constexpr int kWindow = 10;     // most own cells of one row in a tile
constexpr int kSegment = 512;   // candidate places per pass of a tile
// Error bound of the matrix product's |d|^2 - (r_i + r_j + skin)^2 for a pair
// within reach, or nearly so, relative to Q, which bounds |u|^2 + r^2 of own
// bubbles and candidates (u relative to the window's centre).  In units of
// 2^-22 Q: rounding the coordinates and radii to FP32 1, their split into two
// FP16 values (2^-22 each, both sides) 4, the products of the two low parts
// left out 2, the FP32 norms and their split 4, sixteen products added with
// partial sums of at most 2 Q 8.  Pairs farther apart have a larger value by
// more than their error grows.
constexpr float kBand = 0x1.6p-18f;  // 22 2^-22
constexpr float kFar = 3e4f;         // norm of an empty place: never a hit

typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

union Operand {  // eight FP16 values of a lane: half the K range of its row
    uint32_t u[4];
    v8h h;
};

// a, b rounded to FP16, and what that leaves of them.
__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2h));
}
__device__ __forceinline__ uint32_t pack_lo(float a, float b, uint32_t hi) {
    const v2h h = __builtin_bit_cast(v2h, hi);
    return pack_hi(a - (float)h.x, b - (float)h.y);
}

// Sixteen candidate places of one run: bubbles j0 .. j0 + n - 1, and the
// run's image code.
struct Piece {
    int j0;
    int n_code;  // n | code << 8
};

// LDS of one wave: the hit masks of its two tiles over a segment of
// candidates (word w of own bubble o: places 32 w .. 32 w + 31), and the
// segment's pieces.
struct SearchLds {
    uint32_t mask[2][kSegment / 32][kSub];
    Piece piece[2][kSegment / 16];
};

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave-uniform value of vector arithmetic, into scalar registers.
__device__ __forceinline__ double uniform_d(double v) { return readlane_d(v, 0); }
__device__ __forceinline__ float uniform_f(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// One tile: own bubbles [i0, i0 + n), n <= kSub, in at most kWindow
// consecutive cells of one row, and its candidates: the bubbles of the rows
// around, from one cell before the own cells to one after.
struct Tile {
    int i0, n;
    int total;                          // candidate places, 16 per piece
    int run_piece, run_j, run_len, run_code;  // lane s: run s (first piece, ...)
    double o[3];                        // window centre
    float q_max, scale;                 // norm bound; power of two: cells of about 1
    Operand own;
    bool force;                         // an own bubble outside the bound
};

// Lane l's own bubble, position i0 + l of the span, and its cell.  (Its record
// is loaded again for each tile: eight registers over the loops otherwise.)
struct Own {
    int i, cx, cy, cz;
};

template <int D>
__device__ __forceinline__ Own load_own(const Consts &c, const D4 *__restrict__ x4, const int cd[3],
                                        int i) {
#pragma clang fp contract(off)
    Own w;
    w.i = i;
    const D4 r = load_rec(gmem(x4) + i);
    const double p[3] = {r.x, r.y, r.z};
    // the cell as k_s_cells forms it
    int id[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < D; ++q) {
        const double f = floor(cd[q] * (p[q] - c.lbb[q]) / c.interval[q]);
        id[q] = f < 0.0 ? 0 : (f >= (double)cd[q] ? cd[q] - 1 : (int)f);
    }
    w.cx = id[0];
    w.cy = id[1];
    w.cz = id[2];
    return w;
}

// The three cells around x of an axis of n >= 5 cells (or any number between
// walls) in ascending order; wrapped cells first or last.
__device__ __forceinline__ AxisCells near_cells(int x, int n, bool wall) {
    const bool lo = x > 0, hi = x + 1 < n;
    AxisCells r;
    if (wall) {
        r.n = 1 + (lo ? 1 : 0) + (hi ? 1 : 0);
        r.v0 = lo ? x - 1 : x;
        r.v1 = r.v0 + 1;
        r.v2 = r.v0 + 2;
        return r;
    }
    r.n = 3;
    r.v0 = !lo || !hi ? 0 : x - 1;
    r.v1 = !lo ? 1 : !hi ? n - 2 : x;
    r.v2 = !lo || !hi ? n - 1 : x + 1;
    return r;
}

// Inclusive prefix sum over lanes 0-31 (DPP row shifts; the second row of 16
// adds the first one's total).
__device__ __forceinline__ int prefix_32(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    const int row = __builtin_amdgcn_readlane(v, 15);
    return (int)(threadIdx.x & 63) >= 16 ? v + row : v;
}

// The tile of the own bubbles from lane q0 of the span on, `left` of them at
// most.  e: the cell edges.
template <int D>
__device__ __forceinline__ void tile_setup(Tile &t, const Consts &c, const Own &w,
                                           const D4 *__restrict__ x4, const int *__restrict__ start_, const int cd[3],
                                           const double e[3], double rmax, int span0, int q0,
                                           int left) {
    const auto start = gmem(start_);
    const int lane = (int)(threadIdx.x & 63);
    t.i0 = span0 + q0;
    t.n = 0;
    t.total = 0;
    if (left <= 0) return;
    const int ccx = __builtin_amdgcn_readlane(w.cx, q0);
    const int ccy = __builtin_amdgcn_readlane(w.cy, q0);
    const int ccz = 3 == D ? __builtin_amdgcn_readlane(w.cz, q0) : 0;
    const int kmax = min(kWindow, c.wall[0] ? cd[0] : cd[0] - 4);
    // positions are in cell order: those of the row's next kmax cells come first
    const bool in = lane >= q0 && lane < q0 + min(left, kSub) && w.cy == ccy &&
                    (2 == D || w.cz == ccz) && w.cx < ccx + kmax;
    t.n = __popcll(__builtin_amdgcn_ballot_w64(in));
    const int kx = __builtin_amdgcn_readlane(w.cx, q0 + t.n - 1) - ccx + 1;
    const AxisCells Y = near_cells(ccy, cd[1], c.wall[1] != 0);
    const AxisCells Z = 3 == D ? near_cells(ccz, cd[2], c.wall[2] != 0) : AxisCells{0, 0, 0, 1};
    const XWindow xw = x_window(ccx, kx, cd[0], c.wall[0] != 0);
    // 0: neighbour cell a of own cell b does not cross the boundary; 1: its
    // bubbles' image lies at x + L; 2: at x - L
    auto side = [](int a, int b) { return b - a > 1 ? 1 : (a - b > 1 ? 2 : 0); };
    {
        const int r = lane >> 1, part = lane & 1;
        const int a = r / 3, b = r % 3;
        const bool ok = lane < kMaxRuns && a < Z.n && b < Y.n && (0 == part || xw.two);
        const int zc = Z.at(a), yc = Y.at(b);
        const int row = (zc * cd[1] + yc) * cd[0];
        const int js = ok ? start[row + (0 == part ? xw.a0 : xw.a1)] : 0;
        const int je = ok ? start[row + (0 == part ? xw.b0 : xw.b1) + 1] : 0;
        t.run_j = js;
        t.run_len = je - js;
        t.run_code = (side(yc, ccy) << 2) | (side(zc, ccz) << 4) | (0 == part ? xw.f0 : xw.f1);
        // a run starts a piece of its own
        const int np = (t.run_len + 15) >> 4;
        const int incl = prefix_32(np);
        t.run_piece = incl - np;
        t.total = 16 * __builtin_amdgcn_readlane(incl, kMaxRuns - 1);
    }
    const D4 wp = load_rec(gmem(x4) + w.i);
    t.o[0] = uniform_d(c.lbb[0] + (ccx + 0.5 * kx) * e[0]);
    t.o[1] = uniform_d(c.lbb[1] + (ccy + 0.5) * e[1]);
    t.o[2] = 3 == D ? uniform_d(c.lbb[2] + (ccz + 0.5) * e[2]) : 0.0;
    const double hx = (0.5 * kx + 1.0) * e[0], hy = 1.5 * e[1], hz = 1.5 * e[2],
                 hr = rmax + c.skin;
    t.q_max = uniform_f((float)(1.001 * (hx * hx + hy * hy + hz * hz + hr * hr)));
    const float ux = (float)(wp.x - t.o[0]), uy = (float)(wp.y - t.o[1]);
    const float uz = 3 == D ? (float)(wp.z - t.o[2]) : 0.f;
    const float ur = (float)(wp.r + c.skin);
    const float d2 = fmaf(ux, ux, fmaf(uy, uy, uz * uz));
    t.force = __builtin_amdgcn_ballot_w64(in && !(fmaf(ur, ur, d2) <= t.q_max)) != 0ull;
    // the own operand of the own bubble that lane q0 + (lane mod 32) holds:
    // lanes 0-31 (x y z r) high twice, lanes 32-63 (x y z r) low, 1, 1 and
    // the norm's two parts
    const float sc = t.scale, nr = fmaf(-ur, ur, d2) * (sc * sc);
    const uint32_t h0 = pack_hi(ux * sc, uy * sc), h1 = pack_hi(uz * sc, ur * sc);
    const uint32_t l0 = pack_lo(ux * sc, uy * sc, h0), l1 = pack_lo(uz * sc, ur * sc, h1);
    const float nh = (float)(_Float16)nr;
    const uint32_t n2 = pack_hi(nh, nr - nh);
    const int ow = lane & (kSub - 1), from = (q0 + ow) & 63;
    const bool have = ow < t.n, half = lane >= kSub;
    const uint32_t s0 = __shfl((int)(h0), from), s1 = __shfl((int)(h1), from);
    const uint32_t s2 = __shfl((int)(l0), from), s3 = __shfl((int)(l1), from);
    const uint32_t s4 = __shfl((int)(n2), from);
    const uint32_t one = pack_hi(1.f, 1.f), far = pack_hi(kFar, 0.f);
    t.own.u[0] = have ? (half ? s2 : s0) : 0u;
    t.own.u[1] = have ? (half ? s3 : s1) : 0u;
    t.own.u[2] = half ? one : (have ? s0 : 0u);
    t.own.u[3] = half ? (have ? s4 : far) : (have ? s1 : 0u);
}

// Tiles the FP32 values do not settle (bit 2 k + q of `marks`: candidates
// 64 k + 32 q .. of the segment), decided in FP64: each lane its own bubble i
// against its 16 candidates of the tile, into its half of the mask word.
// Rare, and apart from the loop over the candidates, whose registers it would
// share.
template <int D>
__device__ __forceinline__ void exact_tiles(const Foam *F, const Piece *piece, uint32_t *mask,
                                            unsigned marks, int i, int n) {
#pragma clang fp contract(off)
    const auto x4 = gmem(F->s.x4);
    const auto c = cmem(&F->c);  // scalar loads where they are used
    const int lane = (int)(threadIdx.x & 63), ow = lane & (kSub - 1), half = lane >> 5;
    const D4 pi = load_rec(x4 + (ow < n ? i : i - ow));
    for (; marks; marks &= marks - 1u) {
        const int tile = __builtin_ctz(marks);
        const Piece pc = piece[2 * tile + half];
        const int cnt = pc.n_code & 0xff;
        uint32_t w = 0;
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            const D4 pj = load_rec(x4 + (r < cnt ? pc.j0 + r : i - ow));
            // wrapped_diff, sq_len
            const double d1[3] = {pi.x - pj.x, pi.y - pj.y, pi.z - pj.z};
            double m = 0;
#pragma unroll
            for (int k = 0; k < D; ++k) {
                const double a = d1[k] < 0 ? -d1[k] : d1[k];
                const double t = c->interval[k] - a;
                const double image = d1[k] < 0 ? t : -t;
                const double d = !c->wall[k] && t * t < d1[k] * d1[k] ? image : d1[k];
                m += d * d;
            }
            const double maxd = pi.r + pj.r + c->skin;
            if (r < cnt && ow < n && m < maxd * maxd) w |= 1u << r;
        }
        reinterpret_cast<uint16_t *>(mask)[2 * (tile * kSub + ow) + half] = (uint16_t)w;
    }
}

// A chunk of 64 candidates, one per lane: bubble (-1: none), image code and
// record.
struct Chunk {
    int j, f;
    D4 p;
};

// The hit masks of candidates [seg, seg + kSegment) of a tile, decided as the
// FP64 test decides them.
//
// |d|^2 - (r_i + r_j + skin)^2 with both points relative to the window's
// centre is N_i + N_j - 2 (u_i . u_j + r_i' r_j), N = |u|^2 - r^2: a product
// of the own operand (u, r', 1, N_i) with the candidate's (-2u, -2r, N_j, 1).
// With every factor split into two FP16 values, a = a_h + a_l, and a_l b_l
// left out, that is a product over K = 16 -- a_h b_h and a_l b_h in lanes
// 0-31's half, a_h b_l and the norms in lanes 32-63's --, so 32 candidates
// against 32 own bubbles are one 32x32x16 matrix instruction (32 cycles of
// the matrix cores for 1024 pairs; three FP32 ones take 192, and as FP64
// vector instructions the same tests took 13 each).  A lane ends with one own
// bubble and 16 candidates; their sign bits are its part of the mask.  Where
// a value lies within the rounding bound of zero, or a bubble outside the
// bound's window, the tile's pairs are decided again in FP64.
template <int D>
__device__ __forceinline__ void tile_masks(const Tile &t, const Consts &c,
                                           const Foam *F, int seg, int h, SearchLds &lds) {
    const auto x4 = gmem(F->s.x4);
    const int lane = (int)(threadIdx.x & 63), ow = lane & (kSub - 1);
    // the row of a candidate is placed so that a lane's 16 rows are 16
    // consecutive candidates
    const int m = lane & 31;
    const int slot = (lane & 32) | (((m >> 2) & 1) << 4) | ((m >> 3) << 2) | (m & 3);
    const int p_end = min(seg + kSegment, t.total);
    const float eps = kBand * t.q_max * (t.scale * t.scale);
    Piece *const piece = lds.piece[h];
    // the segment's pieces, each run's by its lane; the places after the last
    // run hold none
    if (lane < 4) piece[min((p_end - seg) / 16 + lane, kSegment / 16 - 1)] = Piece{0, 0};
    wave_sync();
    for (int k = 0; __builtin_amdgcn_ballot_w64(16 * k < t.run_len) != 0ull; ++k) {
        const int g = t.run_piece + k - (seg >> 4);
        if (16 * k < t.run_len && g >= 0 && g < kSegment / 16)
            piece[g] = Piece{t.run_j + 16 * k, min(16, t.run_len - 16 * k) | t.run_code << 8};
    }
    wave_sync();
    auto fetch = [&](int p0) {
        const int g = min(p0 - seg + slot, kSegment - 1);
        const Piece pc = piece[g >> 4];
        const bool valid = (slot & 15) < (pc.n_code & 0xff) && p0 < p_end;
        Chunk k;
        k.j = valid ? pc.j0 + (slot & 15) : -1;
        k.f = valid ? pc.n_code >> 8 : 0;
        k.p = load_rec(x4 + (unsigned)(valid ? k.j : t.i0));
        return k;
    };
    unsigned marks = 0;  // tiles to decide in FP64
    Chunk k = fetch(seg);
#pragma unroll 1
    for (int p0 = seg; p0 < p_end; p0 += 64) {
        const bool valid = k.j >= 0;
        double ox = t.o[0], oy = t.o[1], oz = t.o[2];
        if (__builtin_amdgcn_ballot_w64(k.f != 0) != 0ull) {
            // the candidate's image at x + L or x - L
            auto shift = [&](int a) {
                const int fk = (k.f >> (2 * a)) & 3;
                const double up = 1 == fk ? c.interval[a] : 0.0;
                return 2 == fk ? -c.interval[a] : up;
            };
            ox -= shift(0);
            oy -= shift(1);
            if (3 == D) oz -= shift(2);
        }
        const float ux = (float)(k.p.x - ox), uy = (float)(k.p.y - oy);
        const float uz = 3 == D ? (float)(k.p.z - oz) : 0.f;
        const float ur = (float)k.p.r;
        const float d2 = fmaf(ux, ux, fmaf(uy, uy, uz * uz));
        const bool exact =
            t.force || __builtin_amdgcn_ballot_w64(valid && !(fmaf(ur, ur, d2) <= t.q_max)) != 0ull;
        const float m2 = -2.f * t.scale;
        const uint32_t h0 = pack_hi(ux * m2, uy * m2), h1 = pack_hi(uz * m2, ur * m2);
        const uint32_t l0 = pack_lo(ux * m2, uy * m2, h0), l1 = pack_lo(uz * m2, ur * m2, h1);
        // a place without a candidate: any operand with the norm of one far away
        const float nr = valid ? fmaf(-ur, ur, d2) * (t.scale * t.scale) : kFar;
        const float nh = (float)(_Float16)nr;
        const uint32_t n2 = pack_hi(nh, nr - nh), one = pack_hi(1.f, 1.f);
        // the K halves of candidates 0-31 and of 32-63
        Operand op[2];
        auto halves = [&](int d, uint32_t a, uint32_t b) {
            const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
            op[0].u[d] = r[0];
            op[1].u[d] = r[1];
        };
        halves(0, h0, h0);
        halves(1, h1, h1);
        halves(2, l0, n2);
        halves(3, l1, one);
        // the next chunk's records are in flight while this one is tested
        // (past the end too: a branch around the loads would wait for them)
        k = fetch(p0 + 64);
        uint32_t w16[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const v16f acc =
                __builtin_amdgcn_mfma_f32_32x32x16_f16(op[q].h, t.own.h, v16f{}, 0, 0, 0);
            uint32_t w = 0;
            float near = kFar;
#pragma unroll
            for (int r = 15; r >= 0; --r) {
                w = __builtin_amdgcn_alignbit(w, __float_as_uint(acc[r]), 31);
                near = fminf(near, fabsf(acc[r]));
            }
            // (no branch: it would hold the products of both halves in registers)
            const unsigned mark =
                (exact | (__builtin_amdgcn_ballot_w64(near <= eps) != 0ull)) ? 1u : 0u;
            marks |= mark << (((p0 - seg) >> 5) + q);
            w16[q] = w;
        }
        // words of candidates p0 .. p0 + 31 (lanes 0-31) and p0 + 32 .. (lanes
        // 32-63) of own bubble ow, from the halves of both
        const uint32_t w = w16[0] | (w16[1] << 16);
        const auto x = __builtin_amdgcn_permlane32_swap(w, w, false, false);
        const uint32_t word = lane < 32 ? (x[0] & 0xffffu) | (x[1] << 16)
                                        : (x[0] >> 16) | (x[1] & 0xffff0000u);
        lds.mask[h][((p0 - seg) >> 5) + (lane >> 5)][ow] = word;
    }
    if (marks) {
        wave_sync();
        exact_tiles<D>(F, piece, &lds.mask[h][0][0], marks, t.i0 + ow, t.n);
    }
}

// Neighbour lists of the own bubbles [span0, end) of one wave, end - span0 <=
// 64, when every periodic axis has at least 5 cells and no bubble reaches
// beyond the neighbouring cells (the common case).  The own bubbles form two
// tiles (more when a row ends among them).  A tile's candidates -- the runs
// of its window, at most two per row (the x-cells of a row split only where
// the row wraps), in ascending bubble order -- are walked 64 at a time into
// hit masks (tile_masks); then each lane takes one own bubble and appends its
// hits, ascending, one per iteration: consecutive own bubbles are consecutive
// in the list columns, so the lanes' stores share cache lines.
//
// With 5 or more cells per axis the minimum image is decided by the cells
// alone: a candidate in a neighbouring cell that does not cross the boundary
// is within 2/5 of the box and needs no wrap (|d| < L - |d|), one across the
// boundary is at least 3/5 away and always takes the image.  Cells of the
// window more than one apart hold no pair within reach.
//
// Before, a wave tested 64 candidates against one own bubble at a time with
// 13 FP64 operations each and appended the hits of each ballot: bound by
// instruction issue (VALU 69%, SALU 62% of the cycles).  List kernel, same
// foams: 3D 1e6 0.49 -> 0.24 ms, 3D 1e5 (mixed, 45 bubbles a cell) 0.20 ->
// 0.10 ms, batch of 256 foams 2.09 -> 1.21 ms, 2D 1e4 0.017 ms both.  Its
// bound now is latency at five waves per SIMD (a wave waits in two thirds of
// its cycles); four, with ten registers more and no spills, are 4% slower.
template <int D>
__device__ __forceinline__ void search_span(const Foam *F, const Consts &c, const Scratch &S,
                                            const int cd[3], size_t cap, int nbr_cap, double rmax,
                                            int span0, int end, SearchLds &lds, int &sum_nn,
                                            int &max_nn, int &ovf) {
    const int lane = (int)(threadIdx.x & 63), ow = lane & (kSub - 1), h = lane >> 5;
    span0 = uniform_i(span0);
    const int all = uniform_i(end) - span0;
    const Own own = load_own<D>(c, S.x4, cd, span0 + min(lane, all - 1));
    double e[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) e[k] = k < D ? uniform_d(c.interval[k] / cd[k]) : 0.0;
    int ex;
    (void)frexp(fmax(e[0], fmax(e[1], e[2])), &ex);
    const float scale = uniform_f(ldexpf(1.f, -ex));
    int q0 = 0;
    while (q0 < all) {
        int cnt = 0, i = 0, next = q0, most = 0;
        bool have = false;
        auto out = (__attribute__((address_space(1))) int *)S.nbr;
        int seg = 0;
        do {
            int words = 0;
            next = q0;
            // the two tiles in turn (one copy of the code)
#pragma unroll 1
            for (int g = 0; g < 2; ++g) {
                Tile t;
                t.scale = scale;
                tile_setup<D>(t, c, own, S.x4, S.cell_start, cd, e, rmax, span0, next, all - next);
                next += t.n;
                most = max(most, t.total);
                if (seg < t.total) tile_masks<D>(t, c, F, seg, g, lds);
                if (h == g) {
                    have = ow < t.n;
                    i = t.i0 + ow;
                    words = have ? (min(t.total - seg, kSegment) + 31) >> 5 : 0;
                }
            }
            if (0 == seg) out += i;
            wave_sync();
            int w = 0;
            bool live = words > 0;
            uint32_t bits = live ? lds.mask[h][0][ow] : 0u;
            while (live) {
                if (bits) {
                    const int b = __builtin_ctz(bits);
                    bits &= bits - 1u;
                    const int j = lds.piece[h][2 * w + (b >> 4)].j0 + (b & 15);
                    if (j != i) {
                        // entries past the capacity are counted, not written
                        if (cnt < nbr_cap) *out = j;
                        out += cap;
                        ++cnt;
                    }
                }
                if (!bits) {
                    ++w;
                    live = w < words;
                    if (live) bits = lds.mask[h][w][ow];
                }
            }
            wave_sync();
            seg += kSegment;
        } while (seg < most);
        q0 = next;
        if (have) {
            // the list length goes to nn and, as the degree the imposed flow
            // divides by, to deg (which a removal moves but does not reduce)
            const int v = cnt < nbr_cap ? cnt : nbr_cap;
            S.nn[i] = v;
            S.deg[i] = v;
            sum_nn += cnt;
            max_nn = max(max_nn, cnt);
            if (cnt > nbr_cap) ovf = 1;
        }
    }
}

// Search grid: tile t of a foam searches for the own bubbles [t B, t B + B),
// B = stile bubbles, whatever cells they lie in, so the grid stays
// proportional to the bubbles of a foam whatever its cell occupancy (2D
// cells hold a few bubbles, crowded 3D ones a hundred and more).  A wave
// takes 64 of them; the workgroup has as many waves as a tile has spans of
// 64, at most kWaves.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_s_search(
    Foam *foams, const int2 *bt) {
    const Ctx cx = cell_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_search) return;
    extern __shared__ SearchLds s_lds[];  // one per wave
    __shared__ int s_red[3][kWaves];
    const Consts c = F->c;
    const Scratch S = F->s;
    const int cd[3] = {F->d.cell_dim[0], F->d.cell_dim[1], F->d.cell_dim[2]};
    const double rmax = F->d.search_max_r > 0.0 ? F->d.search_max_r : F->d.list_max_r;
    const int b0 = cx.lb * F->stile;
    const int b1 = min(b0 + F->stile, F->d.count);
    const size_t cap = (size_t)F->cap;
    const int nbr_cap = F->nbr_cap;
    int sum_nn = 0, max_nn = 0, ovf = 0;
    // the fast path needs 5 or more cells along every periodic axis, and
    // cells no pair within reach can skip
    bool fast = rmax > 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k < c.dim) {
            if (!c.wall[k] && cd[k] < 5) fast = false;
            if (!((2.0 * rmax + c.skin) * 1.000001 <= c.interval[k] / cd[k])) fast = false;
        }
    const int w = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
    if (fast) {
        for (int i0 = b0 + 64 * w; i0 < b1; i0 += 64 * nw) {
            const int end = min(i0 + 64, b1);
            if (3 == c.dim)
                search_span<3>(F, c, S, cd, cap, nbr_cap, rmax, i0, end, s_lds[w], sum_nn, max_nn,
                               ovf);
            else
                search_span<2>(F, c, S, cd, cap, nbr_cap, rmax, i0, end, s_lds[w], sum_nn, max_nn,
                               ovf);
        }
    } else if (b0 < b1) {
        // the cells holding the own bubbles; units of up to kOwnUnit own
        // bubbles of one cell, dealt round-robin to the waves
        const auto mem = cmem(S.members);
        const auto cof = cmem(S.cell_of);
        const auto cstart = cmem(S.cell_start);
        const int base = cof[mem[b0]], end = cof[mem[b1 - 1]] + 1;
        int uid = 0;
        for (int cell = base; cell < end; ++cell) {
            const int s0 = max(cstart[cell], b0), s1 = min(cstart[cell + 1], b1);
            for (int o0 = s0; o0 < s1; o0 += kOwnUnit, ++uid) {
                if (uid % nw != w) continue;
                const int o1 = min(o0 + kOwnUnit, s1);
                const ListTotals t = 3 == c.dim ? search_cell_general<3>(F, cell, o0, o1)
                                                : search_cell_general<2>(F, cell, o0, o1);
                sum_nn += t.sum_nn;
                max_nn = max(max_nn, t.max_nn);
                ovf = max(ovf, t.ovf);
            }
        }
    }
    sum_nn = wave_sum_i(sum_nn);
    max_nn = wave_max_i(max_nn);
    ovf = wave_max_i(ovf);
    if (0 == (threadIdx.x & 63)) {
        s_red[0][w] = sum_nn;
        s_red[1][w] = max_nn;
        s_red[2][w] = ovf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < nw; ++k) {
            sum_nn += s_red[0][k];
            max_nn = max(max_nn, s_red[1][k]);
            ovf = max(ovf, s_red[2][k]);
        }
        S.cpart_i[cx.lb * kPartI + 1] = sum_nn;
        S.cpart_i[cx.lb * kPartI + 2] = max_nn;
        S.cpart_i[cx.lb * kPartI + 3] = ovf;
    }
}

// One block per foam: make the reordered buffers current (swap = 1), pair
// count, list-capacity check, counters.
__global__ __launch_bounds__(kBlock) void k_s_fin(Foam *foams, int swap) {
    Foam *F = foams + blockIdx.x;
    if (!F->d.need_search) return;
    const Scratch S = F->s;
    const int nb = F->sblk;
    int s = 0, mx = 0, of = 0;
    for (int b = threadIdx.x; b < nb; b += kBlock) {
        s += S.cpart_i[b * kPartI + 1];
        mx = max(mx, S.cpart_i[b * kPartI + 2]);
        of = max(of, S.cpart_i[b * kPartI + 3]);
    }
    const int tot = block_sum_i(s);
    mx = block_max_i(mx);
    of = block_max_i(of);
    if (threadIdx.x == 0) {
        if (swap) swap_reordered_roles(F->r);
        F->d.num_pairs = tot / 2;
        F->d.max_nn = mx;
        F->d.searches += 1;
        if (of) {
            F->d.overflow = 1;
            F->d.halt = 1;
        }
        F->d.need_search = 0;
        if (F->d.search_max_r > 0.0) F->d.list_max_r = F->d.search_max_r;
        F->d.search_max_r = 0.0;  // the next search recomputes it
    }
}

__global__ void k_set_flags(Foam *foams, int nf, int ns, int nr, int clear_halt) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    if (ns >= 0) foams[f].d.need_search = ns;
    if (nr >= 0) foams[f].d.need_remove = nr;
    if (clear_halt) {
        foams[f].d.halt = 0;
        foams[f].d.overflow = 0;
    }
}

// add > 0: every foam halts after `add` more accepted steps; add == 0:
// no limit.  Clears halt / overflow.
__global__ void k_set_limits(Foam *foams, int nf, long long add) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    Dyn &d = foams[f].d;
    d.step_limit = add > 0 ? d.steps + add : 0;
    d.halt = 0;
    d.overflow = 0;
}

void launch_set_limits(const Grid &g, long long add) {
    const int nb = (g.nfoams + 63) / 64;
    hipLaunchKernelGGL(k_set_limits, dim3(nb), dim3(64), 0, g.stream, g.foams, g.nfoams, add);
}

static void launch_lists(const Grid &g) {
    hipLaunchKernelGGL(k_s_search, dim3(g.nb_scell), dim3(g.search_threads),
                       g.search_threads / 64 * sizeof(SearchLds), g.stream, g.foams, g.bt_scell);
}

void launch_search(const Grid &g) {
    hipLaunchKernelGGL(k_s_cells, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    hipLaunchKernelGGL(k_s_scan1, dim3(g.nb_cell), dim3(kBlock), 0, g.stream, g.foams, g.bt_cell);
    hipLaunchKernelGGL(k_s_scan2, dim3(g.nb_cell), dim3(kBlock), 0, g.stream, g.foams, g.bt_cell);
    hipLaunchKernelGGL(k_s_bin, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    hipLaunchKernelGGL(k_s_reorder, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    launch_lists(g);
    hipLaunchKernelGGL(k_s_fin, dim3(g.nfoams), dim3(kBlock), 0, g.stream, g.foams, 1);
}

void launch_search_lists(const Grid &g) {
    launch_lists(g);
    hipLaunchKernelGGL(k_s_fin, dim3(g.nfoams), dim3(kBlock), 0, g.stream, g.foams, 0);
}

void launch_search_part(const Grid &g, int part) {
    if (kPartReorder == part)
        hipLaunchKernelGGL(k_s_reorder, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams,
                           g.bt_bub);
    else  // the list build is the list kernel alone
        launch_lists(g);
}

void launch_set_flags(const Grid &g, int need_search, int need_remove, int clear_halt) {
    const int nb = (g.nfoams + 63) / 64;
    hipLaunchKernelGGL(k_set_flags, dim3(nb), dim3(64), 0, g.stream, g.foams, g.nfoams, need_search,
                       need_remove, clear_halt);
}

}  // namespace cubble_amd
