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
#include "tiles.hpp"

namespace cubble_amd {

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
            // (all loads before a store, which they would not pass)
            double p[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int q = 0; q < D; ++q) p[q] = R.x[q][i];
            rmax = fmax(rmax, R.x[3][i]);
#pragma unroll
            for (int q = 0; q < D; ++q) {
                const double xv = p[q];
                const int mult = c.wall[q] || (xv >= c.lbb[q] && xv <= c.tfr[q]) ? 0
                                 : xv < c.lbb[q] ? 1 : (xv > c.tfr[q] ? -1 : 0);
                if (mult) {
                    p[q] = xv + (c.tfr[q] - c.lbb[q]) * (double)mult;
                    R.x[q][i] = p[q];
                    R.wc[q][i] -= mult;
                    // more than a period outside: it stays in an edge cell, far
                    // from where the matrix tiles take its pairs to be
                    if (!(p[q] >= c.lbb[q] && p[q] <= c.tfr[q])) rmax = __builtin_inf();
                }
            }
            int id[3] = {0, 0, 0};
#pragma unroll
            for (int q = 0; q < D; ++q) {
                const double f = floor(cd[q] * (p[q] - c.lbb[q]) / c.interval[q]);
                id[q] = f < 0.0 ? 0 : (f >= (double)cd[q] ? cd[q] - 1 : (int)f);
            }
            cid = id[2] * cd[0] * cd[1] + id[1] * cd[0] + id[0];
            S.cell_of[i] = cid;
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
        // the whole state before any store (which the loads would not pass),
        // and before the chain to the new slot
        double xs[4] = {0.0, 0.0, 0.0, 0.0};
        V v[4], vo[4];
        int wc[3];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (2 == q && 2 == D) continue;
            xs[q] = R.x[q][i];
            v[q] = field<V>(R.v[q])[i];
            vo[q] = field<V>(R.vo[q])[i];
        }
        const double path = R.path[i];
        const V err = field<V>(R.err)[i];
#pragma unroll
        for (int q = 0; q < D; ++q) wc[q] = R.wc[q][i];
        const int idx = R.idx[i];
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
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (2 == q && 2 == D) continue;
            R.xp[q][np] = xs[q];
            field<V>(R.saved[q])[np] = (V)xs[q];
            field<V>(R.vp[q])[np] = v[q];
            field<V>(R.vs[q])[np] = vo[q];
        }
        S.x4[np] = D4{xs[0], xs[1], xs[2], xs[3]};
        R.path_new[np] = path;
        field<V>(R.err_alt)[np] = err;
#pragma unroll
        for (int q = 0; q < D; ++q) R.wc_alt[q][np] = wc[q];
        R.idx_alt[np] = idx;
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
// `cell` must be wave-uniform.
struct ListTotals {
    int sum_nn, max_nn, ovf;
};

template <int D>
__device__ __forceinline__ ListTotals search_cell_general(const Foam *F, int cell, int i0,
                                                          int i1) {
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

constexpr int kOwnUnit = 32;    // own bubbles per work unit of the general path

// LDS of one wave: the hit masks of its two tiles over a segment of
// candidates (word w of own bubble o: places 32 w .. 32 w + 31), and the
// segment's pieces.
struct SearchLds {
    uint32_t mask[2][kSegment / 32][kSub];
    Piece piece[2][kSegment / 16];
};

template <int D>
__device__ __forceinline__ Own load_own(const Consts &c, const D4 *__restrict__ x4, const int cd[3],
                                        int i) {
#pragma clang fp contract(off)
    const D4 r = load_rec(gmem(x4) + i);
    const double p[3] = {r.x, r.y, r.z};
    // the cell as k_s_cells forms it
    int id[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < D; ++q) {
        const double f = floor(cd[q] * (p[q] - c.lbb[q]) / c.interval[q]);
        id[q] = f < 0.0 ? 0 : (f >= (double)cd[q] ? cd[q] - 1 : (int)f);
    }
    return Own{i, id[0], id[1], id[2]};
}

// The tile of the own bubbles from lane q0 of the span on, `left` of them at
// most, and the centre o of its window.  e: the cell edges.
template <int D>
__device__ __forceinline__ void tile_setup(Tile &t, double o[3], const Consts &c, const Own &w,
                                           const D4 *__restrict__ x4,
                                           const int *__restrict__ start, const int cd[3],
                                           const double e[3], double rmax, int span0, int q0,
                                           int left) {
    t.i0 = span0 + q0;
    t.n = 0;
    t.total = 0;
    if (left <= 0) return;
    const bool wall[3] = {c.wall[0] != 0, c.wall[1] != 0, c.wall[2] != 0};
    const bool in = tile_runs<D>(t, w, start, cd, wall, span0, q0, left);
    o[0] = uniform_d(c.lbb[0] + (t.cx + 0.5 * t.kx) * e[0]);
    o[1] = uniform_d(c.lbb[1] + (t.cy + 0.5) * e[1]);
    o[2] = 3 == D ? uniform_d(c.lbb[2] + (t.cz + 0.5) * e[2]) : 0.0;
    const double hx = (0.5 * t.kx + 1.0) * e[0], hy = 1.5 * e[1], hz = 1.5 * e[2],
                 hr = rmax + c.skin;
    t.q_max = uniform_f((float)(1.001 * (hx * hx + hy * hy + hz * hz + hr * hr)));
    // (the record is loaded again: eight registers over the loops otherwise)
    const D4 p = load_rec(gmem(x4) + w.i);
    own_operand(t, in, q0, (float)(p.x - o[0]), (float)(p.y - o[1]),
                3 == D ? (float)(p.z - o[2]) : 0.f, (float)(p.r + c.skin));
}

// Pair (i, j) as the FP64 test decides it.
template <int D>
__device__ __forceinline__ bool pair_hit(const Foam *F, const D4 &pi, const D4 &pj) {
#pragma clang fp contract(off)
    const auto c = cmem(&F->c);  // scalar loads where they are used
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
    return m < maxd * maxd;
}

// A chunk of 64 candidates, one per lane: bubble (-1: none), image code and
// record.
struct Chunk {
    int j, f;
    D4 p;
};

// The hit masks of candidates [seg, seg + kSegment) of a tile with window
// centre o, decided as the FP64 test decides them.
template <int D>
__device__ __forceinline__ void tile_masks(const Tile &t, const double o[3], const Consts &c,
                                           const Foam *F, int seg, int h, SearchLds &lds) {
    const auto x4 = gmem(F->s.x4);
    const int lane = (int)(threadIdx.x & 63), ow = lane & (kSub - 1), slot = candidate_slot();
    const int p_end = min(seg + kSegment, t.total);
    const float eps = kBand * t.q_max * (t.scale * t.scale);
    Piece *const piece = lds.piece[h];
    tile_pieces(t, seg, piece);
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
    auto operand = [&](const Chunk &k) {
        double ox = o[0], oy = o[1], oz = o[2];
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
        return chunk_operand(t, k.j >= 0, (float)(k.p.x - ox), (float)(k.p.y - oy),
                             3 == D ? (float)(k.p.z - oz) : 0.f, (float)k.p.r);
    };
    unsigned marks = 0;  // halves of chunks to settle in FP64
    Chunk k = fetch(seg);
#pragma unroll 1
    for (int p0 = seg; p0 < p_end; p0 += 64) {
        const ChunkOperand op = operand(k);
        // the next chunk's records are in flight while this one is tested
        // (past the end too: a branch around the loads would wait for them)
        k = fetch(p0 + 64);
        unsigned mk;
        lds.mask[h][((p0 - seg) >> 5) + (lane >> 5)][ow] = chunk_words(t, op, eps, mk);
        marks |= mk << ((p0 - seg) >> 5);
    }
    if (!marks) return;
    wave_sync();
    const D4 pi = load_rec(x4 + t.i0 + (ow < t.n ? ow : 0));
    uint16_t *const half = reinterpret_cast<uint16_t *>(&lds.mask[h][0][ow]) + (lane >> 5);
#pragma unroll 1
    for (; marks; marks &= marks - 1u) {
        const int tile = __builtin_ctz(marks);
        const ChunkOperand op = operand(fetch(seg + 32 * (tile & ~1)));
        const Piece pc = piece[2 * tile + (lane >> 5)];
        const int cnt = ow < t.n ? pc.n_code & 0xff : 0;
        // (places without a candidate too: an own bubble far outside has no
        // sign to go by)
        const uint32_t places = (1u << cnt) - 1u;
        uint32_t open = chunk_open(t, op, tile & 1, eps) & places;
        uint32_t w = half[2 * kSub * tile] & places;
        while (open) {
            const int r = __builtin_ctz(open);
            open &= open - 1u;
            const bool hit = pair_hit<D>(F, pi, load_rec(x4 + pc.j0 + r));
            w = hit ? w | 1u << r : w & ~(1u << r);
        }
        half[2 * kSub * tile] = (uint16_t)w;
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
// 0.094 ms, batch of 256 foams 2.09 -> 1.23 ms, 2D 1e4 17 -> 11 us.  Its
// bound now is VALU issue (64% of the cycles) at four waves per SIMD, of which
// each waits 41% of its cycles; five, with 25 registers spilled, are 15% slower.
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
                double o[3];
                t.scale = scale;
                tile_setup<D>(t, o, c, own, S.x4, S.cell_start, cd, e, rmax, span0, next,
                              all - next);
                next += t.n;
                most = max(most, t.total);
                if (seg < t.total) tile_masks<D>(t, o, c, F, seg, g, lds);
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
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_s_search(
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
    // cells no pair within reach can skip (rmax: none is known to be such when
    // a bubble lies more than a period outside)
    bool fast = rmax > 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (k < c.dim) {
            if (!c.wall[k] && cd[k] < 5) fast = false;
            const double e = c.interval[k] / cd[k];
            if (!((2.0 * rmax + c.skin) * 1.000001 <= e)) fast = false;
            if (!(e > 1e-12 && e < 1e12)) fast = false;  // within FP32's squares
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
        int32_t *const p = S.cpart_i + (cx.lb & (kSearchParts - 1)) * kPartI;
        atomicAdd(p + 1, sum_nn);
        atomicMax(p + 2, max_nn);
        if (ovf) atomicMax(p + 3, ovf);
    }
}

// (The workgroups' totals are integers, added with atomics to kSearchParts
// records of the foam; one record per workgroup took a workgroup per foam 157
// us to reduce at 4e6 bubbles.)
//
// One block per foam: make the reordered buffers current (swap = 1), pair
// count, list-capacity check, counters.
__global__ __launch_bounds__(kSearchParts) void k_s_fin(Foam *foams, int swap) {
    Foam *F = touch_header(foams + blockIdx.x);
    // a removal was carried out before the search
    if (0 == threadIdx.x) F->d.need_remove = 0;
    if (!F->d.need_search) return;
    const Scratch S = F->s;
    int s = 0, mx = 0, of = 0;
    if ((int)threadIdx.x < min(F->sblk, kSearchParts)) {
        int32_t *const p = S.cpart_i + (int)threadIdx.x * kPartI;
        s = p[1];
        mx = p[2];
        of = p[3];
        p[1] = p[2] = p[3] = 0;  // for the next search
    }
    const int tot = wave_sum_i(s);
    mx = wave_max_i(mx);
    of = wave_max_i(of);
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
    d.need_remove = 0;  // carried out
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
    hipLaunchKernelGGL(k_s_fin, dim3(g.nfoams), dim3(kSearchParts), 0, g.stream, g.foams, 1);
}

void launch_search_lists(const Grid &g) {
    launch_lists(g);
    hipLaunchKernelGGL(k_s_fin, dim3(g.nfoams), dim3(kSearchParts), 0, g.stream, g.foams, 0);
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
