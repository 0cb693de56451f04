// pairs.hip -- the reference's searchNeighbors output (src/simulator.cu:60-178)
// as a function of caller-owned device arrays: cubble_find_pairs.
//
// The reference fills Pairs {i, j} (src/data_definitions.h:157-178) with every
// pair i < j whose minimum-image distance is below r_i + r_j + skin
// (comparePair, src/kernels.cu:617-634), grouped by first index (sortPairs,
// :703-711).  Here the caller hands over x, y, z, r (device, FP64) and gets
// pair_i / pair_j in that order, each group also ascending in j, plus the
// pair count in device memory: nothing is read back to the host and the
// host never waits.  The bubbles are not moved: positions are wrapped into the box on the fly (the
// reference wraps them in place first, wrapOverPeriodicBoundaries :992-1011).
//
//   k_p_maxr  : largest radius per block, for the cell size 2 (max r + skin)
//               (simulator.cu:69-75); cell counts zeroed (no memset: the calls
//               may be captured)
//   k_p_cells : cell grid (every block derives the same one), cell of every
//               bubble and its place there (cellByPosition :598-607)
//   k_p_scan* : exclusive scans (cell starts; per-bubble pair offsets)
//   k_p_bin   : bubbles into cell segments (indexByCell :609-615), with the
//               16-byte record the tests read
//   k_p_walk  : the pairs j > i of every bubble, over the de-duplicated 3^D
//               stencil: first counted, then sorted and written
//
// The tests are matrix products over 32 x 32 tiles (tiles.hpp), on positions
// in 32-bit fixed point over the box relative to the tile's window and FP32
// radii; what they leave open is decided on the caller's FP64 values.  The
// bubbles of a cell lie in the order in which atomics gave them their places;
// the pairs, sorted by index, do not depend on it.
//
// Scratch is sized from the bubble count alone, at 40 bytes a bubble: the cell
// grid is shrunk to at most count + 64 cells, which only makes cells larger.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>

#include "cubble_amd.h"
#include "dev_util.hpp"
#include "tiles.hpp"

namespace cubble_amd {

void set_global_error(const std::string &m);

namespace {

constexpr int kScanChunk = kBlock * 16;  // elements per scan block
constexpr int kMaxRBlocks = 256;         // blocks of the radius maximum
constexpr int kSortSlots = 32;           // pairs of a bubble sorted in LDS

struct PairScratch {
    double *max_r;         // largest radius of each k_p_maxr block
    Q4 *rec;               // slot order: fixed-point position, radius (NaN: outside the box)
    int32_t *cell_count, *cell_start, *cell_part, *off_part;
    int32_t *members;      // slot order: bubble
    int32_t *cell_s;       // slot order: cell
    int32_t *cnt, *off;    // per bubble: pairs, their offset; before the
                           // binning its cell and its place there
};

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

int cells_cap_of(int n) { return n + 64; }

int chunks(int m) { return (m + kScanChunk - 1) / kScanChunk; }

// Assigns the scratch arrays in one block at `base` (nullptr: size only).
size_t carve_pairs(PairScratch &P, char *base, int n) {
    size_t off = 0;
    auto take = [&](auto *&p, size_t count) {
        using T = std::remove_reference_t<decltype(*p)>;
        const size_t o = off;
        off = align256(off + std::max<size_t>(count, 1) * sizeof(T));
        p = base ? reinterpret_cast<T *>(base + o) : nullptr;
    };
    const int cc = cells_cap_of(n);
    take(P.max_r, (size_t)kMaxRBlocks);
    take(P.rec, (size_t)n);
    take(P.cell_count, (size_t)cc);
    take(P.cell_start, (size_t)cc + 1);
    take(P.cell_part, (size_t)chunks(cc) + 1);
    take(P.members, (size_t)n);
    take(P.cell_s, (size_t)n);
    take(P.cnt, (size_t)n);
    take(P.off, (size_t)n + 1);
    take(P.off_part, (size_t)chunks(n) + 1);
    return off;
}

// Coordinate wrapped into the box on a periodic axis (one period, as the
// reference's wrap).
__device__ __forceinline__ double wrap_in(const Consts &c, int k, double x) {
    if (c.wall[k]) return x;
    return x < c.lbb[k] ? x + c.interval[k] : (x > c.tfr[k] ? x - c.interval[k] : x);
}

__global__ __launch_bounds__(kBlock) void k_p_maxr(const double *r, int n, PairScratch P,
                                                   int cells_cap) {
    double m = 0.0;
    for (int i = blockIdx.x * kBlock + (int)threadIdx.x; i < n; i += gridDim.x * kBlock)
        m = fmax(m, r[i]);
    m = block_max(m);
    if (0 == threadIdx.x) P.max_r[blockIdx.x] = m;
    for (int q = blockIdx.x * kBlock + (int)threadIdx.x; q < cells_cap; q += gridDim.x * kBlock)
        P.cell_count[q] = 0;
}

// The cell grid, the same in every block (from the nmax block maxima, by the
// whole block), and whether the matrix tiles serve it: five or more cells on
// every periodic axis, edges within FP32's squares.
struct PairGrid {
    int cd[3], cells;
    double max_r;
    bool fast;
};

__device__ __forceinline__ PairGrid grid_of(const Consts &c, const PairScratch &P, int nmax,
                                            int cap) {
    PairGrid g;
    double m = 0.0;
    for (int b = (int)(threadIdx.x & 63); b < nmax; b += 64) m = fmax(m, P.max_r[b]);
    g.max_r = uniform_d(wave_max(m));
    cell_dims(c, g.max_r, cap, g.cd);
    g.cells = g.cd[0] * g.cd[1] * g.cd[2];
    g.fast = true;
    for (int k = 0; k < c.dim; ++k) {
        if (!c.wall[k] && g.cd[k] < 5) g.fast = false;
        const double e = c.interval[k] / g.cd[k];
        if (!((2.0 * g.max_r + c.skin) * 1.000001 <= e && e > 1e-12 && e < 1e12)) g.fast = false;
    }
    return g;
}

template <int D>
__device__ __forceinline__ void cell_of_pos(const Consts &c, const int cd[3], const double p[3],
                                            int id[3]) {
    id[0] = id[1] = id[2] = 0;
#pragma unroll
    for (int q = 0; q < D; ++q) {
        const double f = floor(cd[q] * (p[q] - c.lbb[q]) / c.interval[q]);
        id[q] = f < 0.0 ? 0 : (f >= (double)cd[q] ? cd[q] - 1 : (int)f);
    }
}

template <int D>
__global__ __launch_bounds__(kBlock) void k_p_cells(Consts c, const double *x, const double *y,
                                                    const double *z, int n, PairScratch P,
                                                    int nmax, int cells_cap) {
    const PairGrid g = grid_of(c, P, nmax, cells_cap);
    for (int i0 = blockIdx.x * kBlock; i0 < n; i0 += gridDim.x * kBlock) {
        const int i = i0 + (int)threadIdx.x;
        const bool valid = i < n;
        int cid = -1;
        if (valid) {
            const double p[3] = {wrap_in(c, 0, x[i]), wrap_in(c, 1, y[i]),
                                 3 == D ? wrap_in(c, 2, z[i]) : 0.0};
            int id[3];
            cell_of_pos<D>(c, g.cd, p, id);
            cid = (id[2] * g.cd[1] + id[1]) * g.cd[0] + id[0];
        }
        // one atomic per run of equal cells among the lanes (foams kept in
        // cell order have runs of a cell's bubbles)
        const WaveRuns wr = wave_runs(cid, valid);
        const int lane = (int)(threadIdx.x & 63);
        int place = 0;
        if (valid && lane == wr.head) place = atomicAdd(P.cell_count + cid, wr.len);
        place = __shfl(place, wr.head) + (lane - wr.head);
        if (valid) {
            P.cnt[i] = cid;
            P.off[i] = place;
        }
    }
}

// Exclusive scan of v[0, m) into out[0, m] (out[m] = total, also *total if
// set), in chunks of kScanChunk: pass 1 sums each chunk, pass 2 scans a chunk
// after the sums of the chunks before it (one chunk needs no pass 1).
__global__ __launch_bounds__(kBlock) void k_p_scan_part(const int32_t *v, int m, int32_t *part) {
    const int base = blockIdx.x * kScanChunk;
    int s = 0;
    for (int q = base + (int)threadIdx.x; q < min(base + kScanChunk, m); q += kBlock) s += v[q];
    s = block_sum_i(s);
    if (0 == threadIdx.x) part[blockIdx.x] = s;
}

// A thread scans 16 consecutive elements, so the chunk is one block scan.
__global__ __launch_bounds__(kBlock) void k_p_scan_out(const int32_t *v, int m,
                                                       const int32_t *part, int32_t *out,
                                                       int64_t *total) {
    constexpr int kPer = kScanChunk / kBlock;
    const int base = blockIdx.x * kScanChunk, q0 = base + (int)threadIdx.x * kPer;
    int acc = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += kBlock) acc += part[b];
    int val[kPer], sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        val[k] = q0 + k < m ? v[q0 + k] : 0;
        sum += val[k];
    }
    const int before = block_sum_i(acc);
    int tot = 0;
    int off = before + block_excl_scan(sum, tot);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (q0 + k < m) out[q0 + k] = off;
        off += val[k];
    }
    if (m - 1 < base + kScanChunk && 0 == threadIdx.x) {
        out[m] = before + tot;
        if (total) *total = (int64_t)(before + tot);
    }
}

template <int D>
__global__ __launch_bounds__(kBlock) void k_p_bin(Consts c, const double *x, const double *y,
                                                  const double *z, const double *r, int n,
                                                  PairScratch P) {
    for (int i = blockIdx.x * kBlock + (int)threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const double p[3] = {wrap_in(c, 0, x[i]), wrap_in(c, 1, y[i]),
                             3 == D ? wrap_in(c, 2, z[i]) : 0.0};
        const int cid = P.cnt[i], slot = P.cell_start[cid] + P.off[i];
        int q[3] = {0, 0, 0};
        bool inside = true;
#pragma unroll
        for (int k = 0; k < D; ++k) {
            inside = inside && p[k] >= c.lbb[k] && p[k] <= c.tfr[k];
            q[k] = fixed_code(p[k], c.lbb[k], c.interval[k], c.wall[k] != 0);
        }
        // outside the box (past a wall, or more than a period): no code, and
        // a radius that sends its tiles to the FP64 tests
        P.rec[slot] = Q4{q[0], q[1], q[2], inside ? (float)r[i] : __int_as_float(0x7fc00000)};
        P.members[slot] = i;
        P.cell_s[slot] = cid;
    }
}

// Sorted, de-duplicated cells of coordinate v along one axis (periodic axes
// wrap; wall axes drop cells outside the grid).
__device__ __forceinline__ int axis_neighbours(int v, int n, bool wall, int out[3]) {
    int k = 0;
    for (int o = -1; o <= 1; ++o) {
        int w = v + o;
        if (wall) {
            if (w < 0 || w >= n) continue;
        } else {
            w = (w + n) % n;
        }
        bool dup = false;
        for (int t = 0; t < k; ++t) dup = dup || out[t] == w;
        if (!dup) out[k++] = w;
    }
    return k;
}

// The caller's arrays.
struct PairInput {
    const double *x, *y, *z, *r;
};

// Bubble i's wrapped position and radius.
template <int D>
__device__ __forceinline__ D4 wrapped(const Consts &c, const PairInput &in, int i) {
    return D4{wrap_in(c, 0, in.x[i]), wrap_in(c, 1, in.y[i]),
              3 == D ? wrap_in(c, 2, in.z[i]) : 0.0, in.r[i]};
}

// Two bubbles within r_i + r_j + skin (comparePair).
template <int D>
__device__ __forceinline__ bool within(const Consts &c, const D4 &a, const D4 &b) {
#pragma clang fp contract(off)
    double d[3];
    wrapped_diff<D>(c, a.x, a.y, a.z, b.x, b.y, b.z, d);
    const double maxd = a.r + b.r + c.skin;
    return sq_len(d) < maxd * maxd;
}

// A bubble's group of k pairs written at o0 (within pair_cap): its entries
// ascending, from LDS when they fitted there, else as they were written to
// pair_j.
__device__ __forceinline__ void sort_group(int32_t *pair_j, long long o0, long long hi) {
    for (long long q = o0 + 1; q < hi; ++q) {
        const int v = pair_j[q];
        long long t = q - 1;
        while (t >= o0 && pair_j[t] > v) {
            pair_j[t + 1] = pair_j[t];
            --t;
        }
        pair_j[t + 1] = v;
    }
}

// Any grid: a thread per slot walks the stencil of its cell, four candidates at
// a time (independent loads).  Lanes of one cell read the same candidates, so
// their loads are one line each.  In the bubbles' order, which lets a wave skip
// candidates before all of its bubbles, 64 scattered lanes a load cost more:
// 2e5 bubbles in 27 cells 760 ms a call.
template <int D, bool FILL>
__device__ __forceinline__ void walk_slot(const Consts &c, const PairInput &in,
                                          const PairScratch &P, const PairGrid &g, int slot,
                                          int32_t *pair_i, int32_t *pair_j, long long pair_cap) {
    const int i = P.members[slot], cid = P.cell_s[slot];
    const D4 own = wrapped<D>(c, in, i);
    const int cc[3] = {cid % g.cd[0], (cid / g.cd[0]) % g.cd[1], cid / (g.cd[0] * g.cd[1])};
    int ax[3][3], na[3] = {1, 1, 1};
    ax[2][0] = 0;
    for (int q = 0; q < D; ++q) na[q] = axis_neighbours(cc[q], g.cd[q], c.wall[q] != 0, ax[q]);
    const long long o0 = FILL ? (long long)P.off[i] : 0;
    int k = 0;
    for (int a = 0; a < na[2]; ++a)
        for (int b = 0; b < na[1]; ++b)
            for (int e = 0; e < na[0]; ++e) {
                const int cell = (ax[2][a] * g.cd[1] + ax[1][b]) * g.cd[0] + ax[0][e];
                const int s1 = P.cell_start[cell + 1];
                for (int s = P.cell_start[cell]; s < s1; s += 4) {
                    int js[4];
                    bool later = false;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        js[u] = s + u < s1 ? P.members[s + u] : i;
                        later = later || js[u] > i;
                    }
                    if (!later) continue;
                    D4 other[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) other[u] = wrapped<D>(c, in, js[u]);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (js[u] <= i || !within<D>(c, own, other[u])) continue;
                        if (FILL && o0 + k < pair_cap) {
                            pair_i[o0 + k] = i;
                            pair_j[o0 + k] = js[u];
                        }
                        ++k;
                    }
                }
            }
    if (FILL) sort_group(pair_j, o0, min(o0 + k, pair_cap));
    else P.cnt[i] = k;
}

struct PairLds {
    uint32_t mask[kSegment / 32][kSub];
    Piece piece[kSegment / 16];
    int bubble[kSegment];          // the places' bubbles
    int sorted[kSortSlots][kSub];  // used by the fill alone
};

// The pairs of the own slots [span0, span0 + 32) of one wave, with matrix
// tiles.  FILL = false counts them into cnt[i]; FILL = true sorts each
// bubble's and writes them at off[i] (within pair_cap).
template <int D, bool FILL>
__device__ __forceinline__ void walk_tiles(const Consts &c, const PairInput &in,
                                           const PairScratch &P, const PairGrid &g, int span0,
                                           int n, int32_t *pair_i, int32_t *pair_j,
                                           long long pair_cap, PairLds &lds) {
    const int lane = (int)(threadIdx.x & 63), ow = lane & (kSub - 1), slot = candidate_slot();
    const auto rec = gmem(P.rec);
    const auto mem = gmem(P.members);
    const int all = min(kSub, n - span0);
    const bool wall[3] = {c.wall[0] != 0, c.wall[1] != 0, c.wall[2] != 0};
    Own own;
    own.i = span0 + min(lane, all - 1);
    {
        const int cid = P.cell_s[own.i], row = cid / g.cd[0];
        own.cx = cid - row * g.cd[0];
        own.cz = 3 == D ? row / g.cd[1] : 0;
        own.cy = row - own.cz * g.cd[1];
    }
    const Q4 mine = load_rec(rec + own.i);
    double e[3];
    float step[3], s_max = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        e[k] = k < D ? uniform_d(c.interval[k] / g.cd[k]) : 0.0;
        step[k] = k < D ? uniform_f(fixed_step(c.interval[k], wall[k])) : 0.f;
        s_max = fmaxf(s_max, step[k]);
    }
    int ex;
    (void)frexp(fmax(e[0], fmax(e[1], e[2])), &ex);
    Tile t;
    t.scale = uniform_f(ldexpf(1.f, -ex));
    const float skin = uniform_f((float)c.skin);
    for (int q0 = 0; q0 < all;) {
        const bool mine_in = tile_runs<D>(t, own, P.cell_start, g.cd, wall, span0, q0, all - q0);
        const double hx = (0.5 * t.kx + 1.0) * e[0], hy = 1.5 * e[1], hz = 1.5 * e[2],
                     hr = g.max_r + c.skin;
        t.q_max = uniform_f((float)(1.001 * (hx * hx + hy * hy + hz * hz + hr * hr)));
        const double o[3] = {c.lbb[0] + (t.cx + 0.5 * t.kx) * e[0], c.lbb[1] + (t.cy + 0.5) * e[1],
                             c.lbb[2] + (t.cz + 0.5) * e[2]};
        int oc[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            oc[k] = k < D ? uniform_i(fixed_code(o[k], c.lbb[k], c.interval[k], wall[k])) : 0;
        // relative coordinates: code differences, whose wrap-around is the
        // minimum image
        auto rel = [&](int code, int k) { return (float)fixed_diff(code, oc[k]) * step[k]; };
        own_operand(t, mine_in, q0, rel(mine.x, 0), rel(mine.y, 1), 3 == D ? rel(mine.z, 2) : 0.f,
                    mine.r + skin);
        // two more roundings of the coordinates (4 2^-22 Q), and the codes
        const float eps = (kBand * (26.f / 22.f) * t.q_max +
                           16.f * (float)(2.0 * g.max_r + c.skin) * s_max) *
                          (t.scale * t.scale);
        const bool have = lane < t.n;
        const int self = t.i0 + (ow < t.n ? ow : 0);
        const int i = mem[self];
        int k = 0;  // pairs so far
        const long long o0 = FILL && have ? (long long)P.off[i] : 0;
        for (int seg = 0; seg < t.total; seg += kSegment) {
            const int p_end = min(seg + kSegment, t.total);
            tile_pieces(t, seg, lds.piece);
            struct Place {
                bool valid;
                int j;
                Q4 q;
            };
            auto fetch = [&](int p0) {
                const Piece pc = lds.piece[min(p0 - seg + slot, kSegment - 1) >> 4];
                Place k;
                k.valid = (slot & 15) < (pc.n_code & 0xff) && p0 < p_end;
                const unsigned s = (unsigned)(k.valid ? pc.j0 + (slot & 15) : t.i0);
                k.q = load_rec(rec + s);
                k.j = mem[s];
                return k;
            };
            auto operand = [&](const Place &k) {
                return chunk_operand(t, k.valid, rel(k.q.x, 0), rel(k.q.y, 1),
                                     3 == D ? rel(k.q.z, 2) : 0.f, k.q.r);
            };
            unsigned marks = 0;  // halves of chunks to settle in FP64
            Place k0 = fetch(seg);
#pragma unroll 1
            for (int p0 = seg; p0 < p_end; p0 += 64) {
                const ChunkOperand op = operand(k0);
                lds.bubble[p0 - seg + slot] = k0.j;
                // the next chunk's records are in flight while this one is
                // tested (past the end too: a branch would wait for them)
                k0 = fetch(p0 + 64);
                unsigned mk;
                lds.mask[((p0 - seg) >> 5) + (lane >> 5)][ow] = chunk_words(t, op, eps, mk);
                marks |= mk << ((p0 - seg) >> 5);
            }
            wave_sync();
            // A bubble outside the box lies in an edge cell, so its window is
            // not its stencil: there the cells decide which pairs may meet.
            uint16_t *const half = reinterpret_cast<uint16_t *>(&lds.mask[0][ow]) + (lane >> 5);
#pragma unroll 1
            for (; marks; marks &= marks - 1u) {
                const int tile = __builtin_ctz(marks);
                const ChunkOperand op = operand(fetch(seg + 32 * (tile & ~1)));
                const Piece pc = lds.piece[2 * tile + (lane >> 5)];
                const int cnt = ow < t.n ? pc.n_code & 0xff : 0;
                // (places without a candidate too: an own bubble far outside has no
                // sign to go by)
                const uint32_t places = (1u << cnt) - 1u;
                uint32_t open = chunk_open(t, op, tile & 1, eps) & places;
                uint32_t w = half[2 * kSub * tile] & places;
                const int b = mem[self], cx = P.cell_s[self] % g.cd[0];
                while (open) {
                    const int r = __builtin_ctz(open);
                    open &= open - 1u;
                    const int dx = cx - P.cell_s[pc.j0 + r] % g.cd[0];
                    const bool near = (dx >= -1 && dx <= 1) ||
                                      (!wall[0] && (dx == g.cd[0] - 1 || dx == 1 - g.cd[0]));
                    const bool hit = near && within<D>(c, wrapped<D>(c, in, b),
                                                     wrapped<D>(c, in, mem[pc.j0 + r]));
                    w = hit ? w | 1u << r : w & ~(1u << r);
                }
                half[2 * kSub * tile] = (uint16_t)w;
            }
            wave_sync();
            const int words = (p_end - seg + 31) >> 5;
            int w = 0;
            bool live = have && words > 0;
            uint32_t bits = live ? lds.mask[0][ow] : 0u;
            while (live) {
                if (bits) {
                    const int b = __builtin_ctz(bits);
                    bits &= bits - 1u;
                    const int j = lds.bubble[32 * w + b];
                    if (j > i) {
                        if (FILL) {
                            if (k < kSortSlots) {  // insertion keeps them ascending
                                int q = k;
                                while (q > 0 && lds.sorted[q - 1][ow] > j) {
                                    lds.sorted[q][ow] = lds.sorted[q - 1][ow];
                                    --q;
                                }
                                lds.sorted[q][ow] = j;
                            } else if (o0 + k < pair_cap) {
                                pair_j[o0 + k] = j;
                            }
                        }
                        ++k;
                    }
                }
                if (!bits) {
                    ++w;
                    live = w < words;
                    if (live) bits = lds.mask[w][ow];
                }
            }
            wave_sync();
        }
        if (have) {
            if (FILL) {
                const long long hi = min(o0 + k, pair_cap);
                for (int q = 0; q < k && o0 + q < hi; ++q) {
                    pair_i[o0 + q] = i;
                    if (q < kSortSlots) pair_j[o0 + q] = lds.sorted[q][ow];
                }
                if (k > kSortSlots) sort_group(pair_j, o0, hi);
            } else {
                P.cnt[i] = k;
            }
        }
        q0 += t.n;
    }
}

// Pairs j > i of 64 slots per workgroup, a wave per 32 (matrix tiles), or of 128
// slots, one a thread (small and odd grids).  What bounds it is latency, as the
// list kernel of the simulation; two passes, because the pairs' places are
// known only after all are counted and the scratch holds no pairs.
template <int D, bool FILL>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_p_walk(
    Consts c, PairInput in, int n, PairScratch P, int nmax, int cells_cap, int32_t *pair_i,
    int32_t *pair_j, long long pair_cap) {
    __shared__ PairLds lds[2];
    const PairGrid g = grid_of(c, P, nmax, cells_cap);
    if (g.fast) {
        const int span0 = blockIdx.x * 64 + (int)(threadIdx.x >> 6) * kSub;
        if (span0 < n)
            walk_tiles<D, FILL>(c, in, P, g, span0, n, pair_i, pair_j, pair_cap,
                                lds[threadIdx.x >> 6]);
    } else {  // (128 slots a workgroup: half of them suffice)
        const unsigned slot = blockIdx.x * 128u + threadIdx.x;  // (up to 2^32)
        if (slot < (unsigned)n)
            walk_slot<D, FILL>(c, in, P, g, (int)slot, pair_i, pair_j, pair_cap);
    }
}

__global__ void k_p_none(int64_t *num_pairs) {
    if (0 == threadIdx.x) *num_pairs = 0;
}

int grid_blocks(int items) { return std::max(1, std::min((items + kBlock - 1) / kBlock, 8192)); }

// The whole search on `stream` with scratch P (carved for >= n bubbles).
int enqueue_pairs(const Consts &c, const double *x, const double *y, const double *z,
                  const double *r, int n, const PairScratch &P, int32_t *pair_i, int32_t *pair_j,
                  long long pair_cap, int64_t *num_pairs, hipStream_t st) {
    auto launched = [] {
        const hipError_t e = hipGetLastError();
        if (hipSuccess == e) return CUBBLE_OK;
        set_global_error(std::string("find_pairs launch: ") + hipGetErrorString(e));
        return CUBBLE_E_HIP;
    };
    if (0 == n) {  // no bubbles, no pairs (and no empty launches)
        hipLaunchKernelGGL(k_p_none, dim3(1), dim3(64), 0, st, num_pairs);
        return launched();
    }
    const int cc = cells_cap_of(n);
    const int gb = grid_blocks(n), nmax = std::min(gb, kMaxRBlocks);
    const dim3 walk((n + 63) / 64);
    const PairInput in{x, y, z, r};
    auto scan = [&](const int32_t *v, int m, int32_t *part, int32_t *out, int64_t *total) {
        if (chunks(m) > 1)
            hipLaunchKernelGGL(k_p_scan_part, dim3(chunks(m)), dim3(kBlock), 0, st, v, m, part);
        hipLaunchKernelGGL(k_p_scan_out, dim3(chunks(m)), dim3(kBlock), 0, st, v, m, part, out,
                           total);
    };
    auto run = [&](auto dim) {
        constexpr int D = decltype(dim)::value;
        hipLaunchKernelGGL(k_p_maxr, dim3(nmax), dim3(kBlock), 0, st, r, n, P, cc);
        hipLaunchKernelGGL(k_p_cells<D>, dim3(gb), dim3(kBlock), 0, st, c, x, y, z, n, P, nmax, cc);
        // cell starts (the counts above the grid's cells are zero)
        scan(P.cell_count, cc, P.cell_part, P.cell_start, nullptr);
        hipLaunchKernelGGL(k_p_bin<D>, dim3(gb), dim3(kBlock), 0, st, c, x, y, z, r, n, P);
        hipLaunchKernelGGL((k_p_walk<D, false>), walk, dim3(128), 0, st, c, in, n, P, nmax, cc,
                           pair_i, pair_j, pair_cap);
        scan(P.cnt, n, P.off_part, P.off, num_pairs);
        hipLaunchKernelGGL((k_p_walk<D, true>), walk, dim3(128), 0, st, c, in, n, P, nmax, cc,
                           pair_i, pair_j, pair_cap);
    };
    if (3 == c.dim) run(std::integral_constant<int, 3>{});
    else run(std::integral_constant<int, 2>{});
    return launched();
}

// Arguments checked on the host; the box becomes the kernels' constants.
int check_args(const double *x, const double *y, const double *z, const double *r, int32_t n,
               const cubble_box *box, double skin, const int32_t *pair_i, const int32_t *pair_j,
               int64_t pair_cap, const int64_t *num_pairs, Consts &c) {
    auto bad = [](const char *m) {
        set_global_error(std::string("find_pairs: ") + m);
        return CUBBLE_E_INVALID;
    };
    if (!box || (box->dim != 2 && box->dim != 3)) return bad("box.dim must be 2 or 3");
    if (n < 0 || pair_cap < 0 || !(skin >= 0.0)) return bad("negative count, capacity or skin");
    if (!num_pairs) return bad("num_pairs is null");
    if (n > 0 && (!x || !y || !r || (3 == box->dim && !z)))
        return bad("a position or radius array is null");
    if (pair_cap > 0 && (!pair_i || !pair_j)) return bad("pair arrays are null");
    std::memset(&c, 0, sizeof(c));
    c.dim = box->dim;
    for (int k = 0; k < 3; ++k) {
        const bool used = k < box->dim;
        c.wall[k] = used ? (box->wall[k] != 0) : 0;
        c.lbb[k] = used ? box->lbb[k] : 0.0;
        c.tfr[k] = used ? box->tfr[k] : 0.0;
        c.interval[k] = c.tfr[k] - c.lbb[k];
        if (used && !(c.interval[k] > 0.0)) return bad("box.tfr must exceed box.lbb");
    }
    c.skin = skin;
    return CUBBLE_OK;
}

}  // namespace

// Arguments checked, scratch taken (from `scratch`, `scratch_bytes` long, or
// when that is null with hipMallocAsync / hipFreeAsync on the stream), the
// search enqueued.
int find_pairs_run(const double *x, const double *y, const double *z, const double *r,
                   int32_t count, const cubble_box *box, double skin, int32_t *pair_i,
                   int32_t *pair_j, int64_t pair_cap, int64_t *num_pairs, void *scratch,
                   size_t scratch_bytes, hipStream_t st) {
    Consts c;
    int rc = check_args(x, y, z, r, count, box, skin, pair_i, pair_j, pair_cap, num_pairs, c);
    if (rc) return rc;
    PairScratch P;
    const size_t bytes = carve_pairs(P, nullptr, count);
    if (scratch) {
        if (bytes > scratch_bytes) {
            set_global_error("find_pairs: " + std::to_string(count) +
                             " bubbles need " + std::to_string(bytes) +
                             " bytes of scratch, more than the " +
                             std::to_string(scratch_bytes) + " available");
            return CUBBLE_E_CAPACITY;
        }
        carve_pairs(P, static_cast<char *>(scratch), count);
        return enqueue_pairs(c, x, y, z, r, count, P, pair_i, pair_j, pair_cap, num_pairs, st);
    }
    void *mem = nullptr;
    hipError_t e = hipMallocAsync(&mem, bytes, st);
    if (e != hipSuccess) {
        set_global_error(std::string("find_pairs: hipMallocAsync: ") + hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? CUBBLE_E_NOMEM : CUBBLE_E_HIP;
    }
    carve_pairs(P, static_cast<char *>(mem), count);
    rc = enqueue_pairs(c, x, y, z, r, count, P, pair_i, pair_j, pair_cap, num_pairs, st);
    e = hipFreeAsync(mem, st);
    if (!rc && e != hipSuccess) {
        set_global_error(std::string("find_pairs: hipFreeAsync: ") + hipGetErrorString(e));
        rc = CUBBLE_E_HIP;
    }
    return rc;
}

size_t find_pairs_scratch_bytes(int32_t count) {
    PairScratch P;
    return carve_pairs(P, nullptr, count < 0 ? 0 : count);
}

}  // namespace cubble_amd

using namespace cubble_amd;

extern "C" {

int cubble_find_pairs(const double *x, const double *y, const double *z, const double *r,
                      int32_t count, const cubble_box *box, double skin, int32_t *pair_i,
                      int32_t *pair_j, int64_t pair_cap, int64_t *num_pairs, void *stream) {
    return find_pairs_run(x, y, z, r, count, box, skin, pair_i, pair_j, pair_cap, num_pairs,
                          nullptr, 0, static_cast<hipStream_t>(stream));
}

}  // extern "C"
