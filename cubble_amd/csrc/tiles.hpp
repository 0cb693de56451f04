// tiles.hpp -- candidate tests of the neighbour searches on the matrix cores.
//
// Bubbles are in cell order.  A tile is up to 32 own bubbles in consecutive
// cells of one row and, as candidates, the bubbles of the rows around, from
// one cell before the own cells to one after.  |d|^2 - (r_i + r_j + skin)^2
// with both points relative to the window's centre is N_i + N_j - 2 (u_i .
// u_j + r_i' r_j), N = |u|^2 - r^2: a product of the own operand (u, r', 1,
// N_i) with the candidate's (-2u, -2r, N_j, 1).  With every factor split into
// two FP16 values, a = a_h + a_l, and a_l b_l left out, that is a product over
// K = 16 -- a_h b_h and a_l b_h in lanes 0-31's half, a_h b_l and the norms in
// lanes 32-63's --, so 32 candidates against 32 own bubbles are one 32x32x16
// matrix instruction (32 cycles of the matrix cores for 1024 pairs; three
// FP32 ones take 192, and as FP64 vector instructions the same tests took 13
// each).  A lane ends with one own bubble and 16 candidates; their sign bits
// are its part of the hit mask.  Where a value lies within the rounding bound
// of zero, or a bubble outside the bound's window, the caller decides the
// tile's pairs in FP64, so the result is that of the FP64 test.
#pragma once

#include "dev_util.hpp"

namespace cubble_amd {

constexpr int kMaxRuns = 18;    // 3 z-rows x 3 y-rows x 2 x-runs
constexpr int kSub = 32;        // own bubbles per matrix tile
constexpr int kWindow = 10;     // most own cells of one row in a tile
constexpr int kSegment = 512;   // candidate places per pass of a tile
// Error bound of the matrix product's |d|^2 - (r_i + r_j + skin)^2 for a pair
// within reach, or nearly so, relative to Q, which bounds |u|^2 + r^2 of own
// bubbles and candidates (u relative to the window's centre).  In units of
// 2^-22 Q:
//   1    coordinates and radii rounded to FP32 (0.6 near the cutoff, where |d|
//        is at most a cell and Q at least 4.5 cells squared)
//   4    their split into two FP16 values, 2^-22 each, both sides
//   1.5  low parts below FP16's normal range, which the instruction keeps: steps
//        of 2^-24 where the largest cell edge is 0.5 to 1
//   2    the products of the two low parts, left out
//   4    the FP32 norms and their split
//   8    the instruction.  It adds the eight products of a half of K at a time,
//        aligned to the largest, and drops what lies below 2^-24 of that (its
//        results for 1 +- 15 x 2^-24, x = 1/8 .. 3/2, with the 1 in any place):
//        7 2^-24 2 Q and, with the norms, 7 2^-24 Q, then the halves' sum
//        rounded, 6 in all; one after the other with partial sums of at most
//        2 Q, 8
// Pairs at the cutoff in windows of 1 to 10 cells measured 0.4 to 2.7 in all, 0.3
// to 1.9 of it from the instruction.  Pairs farther apart have a larger value by
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

// A wave-uniform value of vector arithmetic, into scalar registers.
__device__ __forceinline__ double uniform_d(double v) { return readlane_d(v, 0); }
__device__ __forceinline__ float uniform_f(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
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

// Own bubbles [i0, i0 + n), n <= kSub, in the kx <= kWindow cells from (cx, cy,
// cz) on, and their candidates.
struct Tile {
    int i0, n, cx, cy, cz, kx;
    int total;                                // candidate places, 16 per piece
    int run_piece, run_j, run_len, run_code;  // lane s: run s (first piece, ...)
    float q_max, scale;                       // norm bound; power of two: cells of about 1
    Operand own;
    bool force;                               // an own bubble outside the bound
};

// Lane l's own bubble, position span0 + l, and its cell.
struct Own {
    int i, cx, cy, cz;
};

// The tile of the own bubbles from lane q0 of the span on, `left` > 0 of them
// at most: its cells and candidate runs, at most two per row (the x-cells of a
// row split only where the row wraps), in ascending bubble order.  Returns
// whether this lane's own bubble is in it.  Needs 5 or more cells on every
// periodic axis.
template <int D>
__device__ __forceinline__ bool tile_runs(Tile &t, const Own &w, const int *__restrict__ start_,
                                          const int cd[3], const bool wall[3], int span0, int q0,
                                          int left) {
    const auto start = gmem(start_);
    const int lane = (int)(threadIdx.x & 63);
    t.i0 = span0 + q0;
    t.cx = __builtin_amdgcn_readlane(w.cx, q0);
    t.cy = __builtin_amdgcn_readlane(w.cy, q0);
    t.cz = 3 == D ? __builtin_amdgcn_readlane(w.cz, q0) : 0;
    const int kmax = min(kWindow, wall[0] ? cd[0] : cd[0] - 4);
    // positions are in cell order: those of the row's next kmax cells come first
    const bool in = lane >= q0 && lane < q0 + min(left, kSub) && w.cy == t.cy &&
                    (2 == D || w.cz == t.cz) && w.cx < t.cx + kmax;
    t.n = __popcll(__builtin_amdgcn_ballot_w64(in));
    t.kx = __builtin_amdgcn_readlane(w.cx, q0 + t.n - 1) - t.cx + 1;
    const AxisCells Y = near_cells(t.cy, cd[1], wall[1]);
    const AxisCells Z = 3 == D ? near_cells(t.cz, cd[2], wall[2]) : AxisCells{0, 0, 0, 1};
    const XWindow xw = x_window(t.cx, t.kx, cd[0], wall[0]);
    // 0: neighbour cell a of own cell b does not cross the boundary; 1: its
    // bubbles' image lies at x + L; 2: at x - L
    auto side = [](int a, int b) { return b - a > 1 ? 1 : (a - b > 1 ? 2 : 0); };
    const int r = lane >> 1, part = lane & 1;
    const int a = r / 3, b = r % 3;
    const bool ok = lane < kMaxRuns && a < Z.n && b < Y.n && (0 == part || xw.two);
    const int zc = Z.at(a), yc = Y.at(b);
    const int row = (zc * cd[1] + yc) * cd[0];
    const int js = ok ? start[row + (0 == part ? xw.a0 : xw.a1)] : 0;
    const int je = ok ? start[row + (0 == part ? xw.b0 : xw.b1) + 1] : 0;
    t.run_j = js;
    t.run_len = je - js;
    t.run_code = (side(yc, t.cy) << 2) | (side(zc, t.cz) << 4) | (0 == part ? xw.f0 : xw.f1);
    // a run starts a piece of its own
    const int np = (t.run_len + 15) >> 4;
    const int incl = prefix_32(np);
    t.run_piece = incl - np;
    t.total = 16 * __builtin_amdgcn_readlane(incl, kMaxRuns - 1);
    return in;
}

// The own operand: lane l holds own bubble q0 + (l mod 32)'s half -- lanes
// 0-31 (x y z r) high twice, lanes 32-63 (x y z r) low, 1, 1 and the norm's
// two parts -- from the lanes of the span.  ur: radius + skin.
__device__ __forceinline__ void own_operand(Tile &t, bool in, int q0, float ux, float uy, float uz,
                                            float ur) {
    const int lane = (int)(threadIdx.x & 63);
    const float d2 = fmaf(ux, ux, fmaf(uy, uy, uz * uz));
    t.force = __builtin_amdgcn_ballot_w64(in && !(fmaf(ur, ur, d2) <= t.q_max)) != 0ull;
    const float sc = t.scale, nr = fmaf(-ur, ur, d2) * (sc * sc);
    const uint32_t h0 = pack_hi(ux * sc, uy * sc), h1 = pack_hi(uz * sc, ur * sc);
    const uint32_t l0 = pack_lo(ux * sc, uy * sc, h0), l1 = pack_lo(uz * sc, ur * sc, h1);
    const float nh = (float)(_Float16)nr;
    const uint32_t n2 = pack_hi(nh, nr - nh);
    const int ow = lane & (kSub - 1), from = (q0 + ow) & 63;
    const bool have = ow < t.n, half = lane >= kSub;
    const uint32_t s0 = __shfl((int)h0, from), s1 = __shfl((int)h1, from);
    const uint32_t s2 = __shfl((int)l0, from), s3 = __shfl((int)l1, from);
    const uint32_t s4 = __shfl((int)n2, from);
    const uint32_t one = pack_hi(1.f, 1.f), far = pack_hi(kFar, 0.f);
    t.own.u[0] = have ? (half ? s2 : s0) : 0u;
    t.own.u[1] = have ? (half ? s3 : s1) : 0u;
    t.own.u[2] = half ? one : (have ? s0 : 0u);
    t.own.u[3] = half ? (have ? s4 : far) : (have ? s1 : 0u);
}

// The pieces of candidate places [seg, min(seg + kSegment, total)), each run's
// by its lane; the places after the last run hold none.
__device__ __forceinline__ void tile_pieces(const Tile &t, int seg, Piece *piece) {
    const int lane = (int)(threadIdx.x & 63);
    const int p_end = min(seg + kSegment, t.total);
    if (lane < 4) piece[min((p_end - seg) / 16 + lane, kSegment / 16 - 1)] = Piece{0, 0};
    wave_sync();
    for (int k = 0; __builtin_amdgcn_ballot_w64(16 * k < t.run_len) != 0ull; ++k) {
        const int g = t.run_piece + k - (seg >> 4);
        if (16 * k < t.run_len && g >= 0 && g < kSegment / 16)
            piece[g] = Piece{t.run_j + 16 * k, min(16, t.run_len - 16 * k) | t.run_code << 8};
    }
    wave_sync();
}

// The place within a chunk of 64 that this lane's candidate has: the row of a
// candidate is chosen so that a lane's 16 result rows are 16 consecutive
// places (one piece).
__device__ __forceinline__ int candidate_slot() {
    const int lane = (int)(threadIdx.x & 63), m = lane & 31;
    return (lane & 32) | (((m >> 2) & 1) << 4) | ((m >> 3) << 2) | (m & 3);
}

// The candidates of one chunk, as operands: K halves of places 0-31 and 32-63.
struct ChunkOperand {
    Operand op[2];
    bool exact;  // a candidate outside the bound, or an own bubble
};

__device__ __forceinline__ ChunkOperand chunk_operand(const Tile &t, bool valid, float ux, float uy,
                                                      float uz, float ur) {
    ChunkOperand k;
    const float d2 = fmaf(ux, ux, fmaf(uy, uy, uz * uz));
    k.exact =
        t.force || __builtin_amdgcn_ballot_w64(valid && !(fmaf(ur, ur, d2) <= t.q_max)) != 0ull;
    const float m2 = -2.f * t.scale;
    const uint32_t h0 = pack_hi(ux * m2, uy * m2), h1 = pack_hi(uz * m2, ur * m2);
    const uint32_t l0 = pack_lo(ux * m2, uy * m2, h0), l1 = pack_lo(uz * m2, ur * m2, h1);
    // a place without a candidate: any operand with the norm of one far away
    const float nr = valid ? fmaf(-ur, ur, d2) * (t.scale * t.scale) : kFar;
    const float nh = (float)(_Float16)nr;
    const uint32_t n2 = pack_hi(nh, nr - nh), one = pack_hi(1.f, 1.f);
    auto halves = [&](int d, uint32_t a, uint32_t b) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        k.op[0].u[d] = r[0];
        k.op[1].u[d] = r[1];
    };
    halves(0, h0, h0);
    halves(1, h1, h1);
    halves(2, l0, n2);
    halves(3, l1, one);
    return k;
}

// The chunk's hit words, of own bubble l mod 32: places 0-31 in lanes 0-31,
// 32-63 in lanes 32-63.  Bits 0 and 1 of `marks` are set for the halves to be
// decided in FP64.
__device__ __forceinline__ uint32_t chunk_words(const Tile &t, const ChunkOperand &k, float eps,
                                                unsigned &marks) {
    uint32_t w16[2];
    marks = 0;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const v16f acc =
            __builtin_amdgcn_mfma_f32_32x32x16_f16(k.op[q].h, t.own.h, v16f{}, 0, 0, 0);
        uint32_t w = 0;
        float near = kFar;
#pragma unroll
        for (int r = 15; r >= 0; --r) {
            w = __builtin_amdgcn_alignbit(w, __float_as_uint(acc[r]), 31);
            near = fminf(near, fabsf(acc[r]));
        }
        // (no branch: it would hold the products of both halves in registers)
        const unsigned mark =
            (k.exact | (__builtin_amdgcn_ballot_w64(near <= eps) != 0ull)) ? 1u : 0u;
        marks |= mark << q;
        w16[q] = w;
    }
    // the two halves of a word come from the lanes l and l + 32
    const uint32_t w = w16[0] | (w16[1] << 16);
    const auto x = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    return (threadIdx.x & 63) < 32 ? (x[0] & 0xffffu) | (x[1] << 16)
                                   : (x[0] >> 16) | (x[1] & 0xffff0000u);
}

// The places of half q (0, 1) of a chunk that the product does not settle, as
// this lane's 16 bits of them: for the halves chunk_words marked, formed again
// apart from the loop over the chunks, whose registers they would share.
__device__ __forceinline__ uint32_t chunk_open(const Tile &t, const ChunkOperand &k, int q,
                                               float eps) {
    if (k.exact) return 0xffffu;
    Operand op;
#pragma unroll
    for (int d = 0; d < 4; ++d) op.u[d] = q ? k.op[1].u[d] : k.op[0].u[d];
    const v16f acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(op.h, t.own.h, v16f{}, 0, 0, 0);
    uint32_t w = 0;
#pragma unroll
    for (int r = 15; r >= 0; --r) w |= fabsf(acc[r]) <= eps ? 1u << r : 0u;
    return w;
}

}  // namespace cubble_amd
