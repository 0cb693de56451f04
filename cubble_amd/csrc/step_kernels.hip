// step_kernels.hip -- the kernels of one step() attempt.
//
//   k_predict : (in a captured run the removal of the attempt before;) AB2
//               predictor + block partials of S_A, S_Ar; writes the 32-byte
//               FP64 neighbour record, or in mixed precision the 16-byte
//               fixed-point one (reference preIntegrate,
//               src/kernels.cu:40-170)
//   k_pair, k_pair_quad : pairwise Durian velocity, overlap area and gas flux,
//               gathered per bubble over its full neighbour list, by one lane
//               or (small launches) four; partials of S_OA, S_OAr
//               (reference pairwiseInteraction, src/kernels.cu:172-337)
//   k_sums    : S_A, S_Ar, S_OA, S_OAr of foams whose corrector does not form
//               them itself
//   k_correct : walls, liquid-mediated gas exchange, trapezoid corrector,
//               error / expansion / radius / volume partials, deletion marks,
//               path (reference postIntegrate, src/kernels.cu:339-495,
//               :546-593)
//   k_control : one workgroup per foam: the corrector's partials, the dt
//               controller and, when committing, the rotation of the role
//               pointers and the plan of a removal (reference
//               step()/integrate(), src/simulator.cu:192-314)
//
// The reference scatters every pair into both bubbles with FP64 atomics in
// unspecified order.  Here each bubble gathers its own neighbours in
// ascending index order, so results are deterministic, independent of the
// launch shape, and need no atomics.  All reductions are fixed-order trees.
#include <type_traits>

#include "dev_util.hpp"
#include "launch.hpp"
#include "remove_apply.hpp"
#include "remove_plan.hpp"

namespace cubble_amd {

// ---------------------------------------------------------------- predictor
// FP64: writes the 32-byte record the FP64 pair kernel gathers.  Mixed
// (FIXED, FP32 velocities): writes only the 16-byte fixed-point record.
template <int D, bool GAS, bool FIXED>
__device__ __forceinline__ void predict_range(const Consts &c, const Roles &R, D4 *__restrict__ p4,
                                              Q4 *__restrict__ q4, int base, int ipt, int n,
                                              double h, double &sa, double &sar) {
    for (int k = 0; k < ipt; ++k) {
        const int i = base + k * kBlock + (int)threadIdx.x;
        if (i >= n) break;
        const D4 pr = predicted<D, GAS, typename std::conditional<FIXED, float, double>::type>(
            R, h, i);
        if (GAS) {
            double apr = 2.0 * kPi;
            if (3 == D) apr *= 2.0 * pr.r;
            sa += apr * pr.r;
            sar += apr;
        }
        if (FIXED) {
            const double p[3] = {pr.x, pr.y, pr.z};
            int32_t qc[3] = {0, 0, 0};
#pragma unroll
            for (int q = 0; q < D; ++q) qc[q] = fixed_code(p[q], c.lbb[q], c.interval[q], c.wall[q] != 0);
            typedef int v4i __attribute__((ext_vector_type(4)));
            const v4i w = {qc[0], qc[1], qc[2], __float_as_int((float)pr.r)};
            stream_store(reinterpret_cast<v4i *>(q4 + i), w);
        } else {
            p4[i] = pr;
        }
    }
}

template <int D, bool GAS>
__device__ __forceinline__ void predict_dispatch(const Consts &c, const Roles &R,
                                                 D4 *__restrict__ p4, Q4 *__restrict__ q4,
                                                 int base, int ipt, int n, double h, double &sa,
                                                 double &sar) {
    if (q4) predict_range<D, GAS, true>(c, R, p4, q4, base, ipt, n, h, sa, sar);
    else predict_range<D, GAS, false>(c, R, p4, q4, base, ipt, n, h, sa, sar);
}

// APPLY: first the removal of the attempt before, if there was one, on the
// block's own slots (a variant of its own: it takes 84 registers, the plain
// predictor 41).
template <bool APPLY>
__global__ __launch_bounds__(kBlock) void k_predict(Foam *foams, const int2 *bt, uint32_t flags) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (standing(F->d)) return;
    if (APPLY && F->d.need_remove) {
        apply_removal(F, cx.lb);
        __syncthreads();  // its waves wrote this block's slots
    }
    const int n = F->d.count, ipt = F->ipt;
    const double h = 0.5 * F->d.dt;
    const Roles R = F->r;
    const int base = cx.lb * kBlock * ipt;
    double sa = 0.0, sar = 0.0;
    const bool gas = (flags & kGas) != 0;
    D4 *p4 = F->s.p4;
    Q4 *q4 = F->s.q4;
    const Consts c = F->c;
    if (3 == c.dim) {
        if (gas) predict_dispatch<3, true>(c, R, p4, q4, base, ipt, n, h, sa, sar);
        else predict_dispatch<3, false>(c, R, p4, q4, base, ipt, n, h, sa, sar);
    } else {
        if (gas) predict_dispatch<2, true>(c, R, p4, q4, base, ipt, n, h, sa, sar);
        else predict_dispatch<2, false>(c, R, p4, q4, base, ipt, n, h, sa, sar);
    }
    double sums[2] = {sa, sar};
    int none = 0;
    block_reduce_t0(sums, 0u, none);
    if (threadIdx.x == 0) {
        F->s.part[cx.lb * kPartD + 0] = sums[0];
        F->s.part[cx.lb * kPartD + 1] = sums[1];
    }
}

// ---------------------------------------------------------------- pair (FP64)
// FLOW: also the imposed-flow term.  The neighbour-velocity sum takes every
// listed neighbour with a smaller index and the overlapping ones with a
// larger index: the reference adds dxdt[idx1] into idx2 for every listed pair
// (idx1 < idx2) but dxdt[idx2] into idx1 only past its overlap test
// (src/kernels.cu:191-208 vs :281-307).
//
// Adds what pair (i, j) adds to bubble i: zeros unless it overlaps (or j < 0),
// which it returns.  d = x_i - x_j (minimum image); inv_ri = 1 / ri, risq =
// ri^2.  Without a branch, so that the chains of several pairs overlap.
template <int D, bool GAS>
__device__ __forceinline__ bool add_pair(double f0, int i, double ri, double risq, double inv_ri,
                                         int j, double rj, const double (&d)[3], double (&acc)[3],
                                         double &ovl, double &dr) {
    const double radii = ri + rj;
    const double m = sq_len(d);
    const bool on = j >= 0 && radii * radii >= m;
    const double rs = rsq_nr(m);
    const double s = rs - rcp_nr(radii);
#pragma unroll
    for (int a = 0; a < D; ++a) {
        const double t = d[a] * f0 * s;
        acc[a] += on ? t : 0.0;
    }
    if (GAS) {
        const double rjsq = rj * rj;
        const double r1sq = i < j ? risq : rjsq;  // of the smaller index
        const double r2sq = i < j ? rjsq : risq;
        double oa = 0.5 * (r2sq - r1sq + m);
        oa *= oa;
        oa *= rs * rs;  // / m
        oa = fabs(r2sq - oa);
        if (m < r1sq || m < r2sq) oa = r1sq < r2sq ? r1sq : r2sq;
        if (3 == D) {
            oa *= kPi;
        } else {
            oa = 2.0 * sqrt(oa);
        }
        const double t = oa * (rcp_nr(rj) - inv_ri);
        ovl += on ? oa : 0.0;
        dr += on ? t : 0.0;
    }
    return on;
}

template <int D, bool GAS, bool FLOW>
__device__ __forceinline__ void pair_range(const Consts &c, const Roles &R, const Scratch &S,
                                           size_t cap, int base, int ipt, int n, double &soa,
                                           double &soar) {
    const D4 *__restrict__ p4 = S.p4;
    const int *__restrict__ nnA = S.nn;
    const int *__restrict__ nbr = S.nbr;
    const double f0 = c.f0;
    // below it, a difference is its own minimum image
    double near[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) near[a] = c.wall[a] ? __builtin_inf() : 0.49 * c.interval[a];
    for (int k = 0; k < ipt; ++k) {
        const int i = base + k * kBlock + (int)threadIdx.x;
        if (i >= n) break;
        const D4 pi = p4[i];
        const double xi = pi.x, yi = pi.y, zi = pi.z, ri = pi.r;
        const double inv_ri = 1.0 / ri, risq = ri * ri;
        double acc[3] = {0.0, 0.0, 0.0};
        double fv[3] = {0.0, 0.0, 0.0};
        double ovl = 0.0, dr = 0.0;
        const int m_nn = nnA[i];
        for_neighbours(nbr, p4, cap, i, m_nn, [&](const int(&js)[kGather],
                                                  const D4(&ps)[kGather]) {
            double d[kGather][3];
            bool far = false;
#pragma unroll
            for (int u = 0; u < kGather; ++u) {
                d[u][0] = xi - ps[u].x;
                d[u][1] = yi - ps[u].y;
                d[u][2] = 3 == D ? zi - ps[u].z : 0.0;
#pragma unroll
                for (int a = 0; a < D; ++a) far = far || fabs(d[u][a]) > near[a];
            }
            // the minimum image, for waves with a pair across the boundary
            // (one in five at 35 cells an axis)
            if (__builtin_amdgcn_ballot_w64(far) != 0ull) {
#pragma unroll
                for (int u = 0; u < kGather; ++u)
                    wrapped_diff<D>(c, xi, yi, zi, ps[u].x, ps[u].y, ps[u].z, d[u]);
            }
#pragma unroll
            for (int u = 0; u < kGather; ++u) {
                const int j = js[u];
                const bool on = add_pair<D, GAS>(f0, i, ri, risq, inv_ri, j, ps[u].r, d[u], acc,
                                                 ovl, dr);
                if (FLOW && j >= 0 && (j < i || on)) {
#pragma unroll
                    for (int a = 0; a < D; ++a) fv[a] += field<double>(R.v[a])[j];
                }
            }
        });
        if (FLOW) add_flow<D>(c, pi, S.deg[i], fv, acc);
#pragma unroll
        for (int a = 0; a < D; ++a) field<double>(R.vp[a])[i] = acc[a];
        field<double>(R.vp[3])[i] = dr;
        field<double>(S.ov)[i] = ovl;
        soa += ovl;
        soar += ovl * inv_ri;
    }
}

// Block b's sums of S_A, S_Ar, S_OA, S_OAr; quad: the pair kernel's as
// k_pair_quad left them, four a block, added in the order of the block's waves.
__device__ __forceinline__ void block_sums(const double *part, const double *quad, int b,
                                           double (&v)[4]) {
#pragma unroll
    for (int k = 0; k < 2; ++k) v[k] = part[b * kPartD + k];
    if (quad) {
        v[2] = v[3] = 0.0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            v[2] += quad[8 * b + 2 * w];
            v[3] += quad[8 * b + 2 * w + 1];
        }
    } else {
        v[2] = part[b * kPartD + 2];
        v[3] = part[b * kPartD + 3];
    }
}

// One value quadruple per block, read(b, v), reduced in one pass (each thread
// takes blocks t, t + kBlock, ... in order), and the integer slot 0 of the int
// partials summed alongside, their non-zero ones given to found(b, count), if
// part_i.  Bit k of `dmax` makes value k a maximum
// (from 0), else a sum.  The results are defined in thread 0 only.
template <typename Read, typename Found>
__device__ __forceinline__ void reduce_parts4(Read &&read, const int32_t *part_i, Found &&found,
                                              int nb, unsigned dmax, double (&r)[4], int &ri) {
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    int ai = 0;
#pragma unroll 2
    for (int b = threadIdx.x; b < nb; b += kBlock) {
        double v[4];
        read(b, v);
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = (dmax >> k) & 1u ? fmax(a[k], v[k]) : a[k] + v[k];
        if (part_i) {
            const int c = part_i[b * kPartI];
            if (c > 0) found(b, c);
            ai += c;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = a[k];
    ri = ai;
    block_reduce_t0(r, dmax, ri);
}

// One kernel per FLOW value: the flow variant needs more registers, which
// would otherwise lower the occupancy of the plain one (96: five waves a SIMD).
//
// The body has no branch per neighbour: the four chains of a chunk overlap,
// where one after another each waited for its own square root and
// reciprocals (2D 1e4: 9.0 -> 7.5 us a launch), and terms that do not count
// are selected away (adding 0).  At 1e6 bubbles (65 to 78 us) it is bound by
// instruction issue: VALU work in 61% of the cycles, and waves wait to issue for
// 46% of theirs, on memory for 30%, with the address units busy for 37%.  Neither
// six waves (114 us, spilled) nor halves of records gathered by neighbouring
// lanes (110 us) help.
template <bool FLOW>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(FLOW ? 4 : 5, 8))) void
k_pair(Foam *foams, const int2 *bt, uint32_t flags) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (standing(F->d)) return;
    const int n = F->d.count, ipt = F->ipt;
    const Consts c = F->c;
    const Roles R = F->r;
    const Scratch S = F->s;
    const size_t cap = (size_t)F->cap;
    const int base = cx.lb * kBlock * ipt;
    double soa = 0.0, soar = 0.0;
    const bool gas = (flags & kGas) != 0;
    if (3 == c.dim) {
        if (gas) pair_range<3, true, FLOW>(c, R, S, cap, base, ipt, n, soa, soar);
        else pair_range<3, false, FLOW>(c, R, S, cap, base, ipt, n, soa, soar);
    } else {
        if (gas) pair_range<2, true, FLOW>(c, R, S, cap, base, ipt, n, soa, soar);
        else pair_range<2, false, FLOW>(c, R, S, cap, base, ipt, n, soa, soar);
    }
    double sums[2] = {soa, soar};
    int none = 0;
    block_reduce_t0(sums, 0u, none);
    if (threadIdx.x == 0) {
        S.part[cx.lb * kPartD + 2] = sums[0];
        S.part[cx.lb * kPartD + 3] = sums[1];
    }
}

// Bubble i's pairs by four lanes, lane u of them taking list entries u, u + 4,
// ..., two at a time; every lane adds all four's terms in list order, the
// order (and so the bits) of pair_range.  i >= n: nothing.
template <int D, bool GAS, bool FLOW>
__device__ __forceinline__ void pair_quad(const Consts &c, const Roles &R, const Scratch &S,
                                          size_t cap, int i, int n, double &soa, double &soar) {
    if (i >= n) return;
    const auto p4 = gmem(S.p4);
    const auto nbr = gmem(S.nbr);
    const int u = (int)(threadIdx.x & 3);
    const double f0 = c.f0;
    double near[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) near[a] = c.wall[a] ? __builtin_inf() : 0.49 * c.interval[a];
    const D4 pi = load_rec(p4 + i);
    const double inv_ri = 1.0 / pi.r, risq = pi.r * pi.r;
    double acc[3] = {0.0, 0.0, 0.0};
    double fv[3] = {0.0, 0.0, 0.0};
    double ovl = 0.0, dr = 0.0;
    const int m_nn = S.nn[i];
    for (int q0 = 0; q0 < m_nn; q0 += 8) {
        int js[2];
        D4 ps[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int q = q0 + 4 * w + u;
            const int j = nbr[(size_t)min(q, m_nn - 1) * cap + i];
            js[w] = q < m_nn ? j : -1;
        }
#pragma unroll
        for (int w = 0; w < 2; ++w) ps[w] = load_rec(p4 + (js[w] >= 0 ? js[w] : i));
        double d[2][3];
        bool far = false;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            d[w][0] = pi.x - ps[w].x;
            d[w][1] = pi.y - ps[w].y;
            d[w][2] = 3 == D ? pi.z - ps[w].z : 0.0;
#pragma unroll
            for (int a = 0; a < D; ++a) far = far || fabs(d[w][a]) > near[a];
        }
        if (__builtin_amdgcn_ballot_w64(far) != 0ull) {
#pragma unroll
            for (int w = 0; w < 2; ++w)
                wrapped_diff<D>(c, pi.x, pi.y, pi.z, ps[w].x, ps[w].y, ps[w].z, d[w]);
        }
        double t[2][3] = {}, to[2] = {}, tr[2] = {}, tv[2][3];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const bool on = add_pair<D, GAS>(f0, i, pi.r, risq, inv_ri, js[w], ps[w].r, d[w], t[w],
                                             to[w], tr[w]);
            if (FLOW) {
                const bool count = js[w] >= 0 && (js[w] < i || on);
#pragma unroll
                for (int a = 0; a < D; ++a) tv[w][a] = count ? field<double>(R.v[a])[js[w]] : 0.0;
            }
        }
#pragma unroll
        for (int w = 0; w < 2; ++w) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                acc[a] = quad_add(acc[a], t[w][a]);
                if (FLOW) fv[a] = quad_add(fv[a], tv[w][a]);
            }
            if (GAS) {
                ovl = quad_add(ovl, to[w]);
                dr = quad_add(dr, tr[w]);
            }
        }
    }
    if (FLOW) add_flow<D>(c, pi, S.deg[i], fv, acc);
    if (0 == u) {
#pragma unroll
        for (int a = 0; a < D; ++a) field<double>(R.vp[a])[i] = acc[a];
        field<double>(R.vp[3])[i] = dr;
        field<double>(S.ov)[i] = ovl;
    }
    soa = ovl;
    soar = ovl * inv_ri;
}

// The pair kernel of launches of up to kQuadBlocks blocks with one bubble a
// thread: a workgroup takes 64 bubbles, four lanes each.  k_pair is bound there
// by each wave's chain of loads and FP64 operations, list entry after list
// entry, with few waves to overlap it; here a lane evaluates a quarter of the
// pairs, and a wave waits for the longest of 16 lists instead of 64.  us a
// launch, k_pair / this: 2D 1e3 6.9 / 3.8, 3e4 7.5 / 5.1, 2e5 12.7 / 11.7; 3D
// 1e3 13.1 / 6.4, 3e4 15.3 / 7.8, 2e5 26.5 / 21.6; 8 foams of 1e4 17.4 / 10.9,
// 128 of 2e3 30.7 / 26.9.  Beyond, the additions of every term in four lanes
// cost more: 2D 5e5 23.5 / 27.4, 3D 42.8 / 46.5, 1e6 75.6 / 86.6.  The sums
// leave as those of k_pair's waves, two for each 64 bubbles, at quad_parts().
template <bool FLOW>
__global__ __launch_bounds__(kBlock) void k_pair_quad(Foam *foams, const int2 *bt,
                                                      uint32_t flags) {
    const int2 e = bt ? bt[blockIdx.x >> 2] : make_int2(0, 0);
    Foam *F = bt ? foams + e.x : touch_header(foams);
    if (standing(F->d)) return;
    const int part = bt ? 4 * xcd_remap(e.y, F->nblk) + (int)(blockIdx.x & 3)
                        : xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int n = F->d.count;
    const Consts c = F->c;
    const Roles R = F->r;
    const Scratch S = F->s;
    const size_t cap = (size_t)F->cap;
    const int i = part * 64 + (int)(threadIdx.x >> 2);
    double soa = 0.0, soar = 0.0;
    const bool gas = (flags & kGas) != 0;
    if (3 == c.dim) {
        if (gas) pair_quad<3, true, FLOW>(c, R, S, cap, i, n, soa, soar);
        else pair_quad<3, false, FLOW>(c, R, S, cap, i, n, soa, soar);
    } else {
        if (gas) pair_quad<2, true, FLOW>(c, R, S, cap, i, n, soa, soar);
        else pair_quad<2, false, FLOW>(c, R, S, cap, i, n, soa, soar);
    }
    quad_store(S, part, soa, soar);
}

// One block per foam: S_A, S_Ar, S_OA, S_OAr from the predictor and pair
// partials, in a fixed order.  (A separate launch: on MI355X the eight XCD
// L2 caches are not coherent, so an in-kernel last-block reduction would
// need an agent-scope release -- an L2 write-back -- in every block.)
__global__ __launch_bounds__(kBlock) void k_sums(Foam *foams, bool quad) {
    Foam *F = touch_header(foams + blockIdx.x);
    if (standing(F->d)) return;
    double r[4];
    int none;
    const double *const part = F->s.part, *const q = quad ? quad_parts(F->s) : nullptr;
    reduce_parts4([&](int b, double (&v)[4]) { block_sums(part, q, b, v); }, nullptr,
                  [](int, int) {}, F->nblk, 0u, r, none);
    if (threadIdx.x == 0) {
        F->d.s_a = r[0];
        F->d.s_ar = r[1];
        F->d.s_oa = r[2];
        F->d.s_oar = r[3];
    }
}

// S_A, S_Ar, S_OA, S_OAr of a foam, in every thread of the calling workgroup:
// the sums of k_sums in its order, so the same bits.  Reading the partials in
// every block of the corrector costs it under a microsecond up to kFuseBlocks;
// the launch of k_sums that it replaces costs 2.5 to 3.5.  In a batch the launch
// is the cheaper one: 256 foams' correctors took 36 us longer.
// Up to 64 blocks every wave sums for itself, without a barrier.
__device__ __forceinline__ void block_foam_sums(const double *__restrict__ part,
                                                const double *__restrict__ quad, int nb,
                                                double (&r)[4]) {
    __shared__ double s_sum[kWaves][4];
    const bool few = nb <= 64;
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = 0.0;
    for (int b = few ? threadIdx.x & 63 : threadIdx.x; b < nb; b += kBlock) {
        double v[4];
        block_sums(part, quad, b, v);
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] += v[k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = wave_sum(r[k]);
    if (few) return;
    if (0 == (threadIdx.x & 63)) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s_sum[threadIdx.x >> 6][k] = r[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        r[k] = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) r[k] += s_sum[w][k];
    }
}

// ---------------------------------------------------------------- corrector
// reference src/kernels.cu:546-593 (addWallVelocity)
template <int D>
__device__ __forceinline__ void add_wall_velocity(const Consts &c, double xp, double yp, double zp,
                                                  double rad, double &vx, double &vy, double &vz) {
    const double drag = 1.0 - c.wall_drag;
    double xDrag = 1.0, velocity = 0.0;
    auto touches = [&](double x, double low, double high) -> bool {
        double d1 = x - low;
        double d2 = x - high;
        d1 = d1 * d1 < d2 * d2 ? d1 : d2;
        if (rad * rad >= d1 * d1) {
            d2 = d1 < 0.0 ? -1.0 : 1.0;
            d1 *= d2;
            velocity = d2 * c.f0 * (1.0 - d1 / rad);
            return true;
        }
        return false;
    };
    double yDrag = 1.0;
    velocity = 0.0;
    if (c.wall[0] && touches(xp, c.lbb[0], c.tfr[0])) {
        vx += velocity;
        vy *= drag;
        if (3 == D) vz *= drag;
        xDrag = drag;
    }
    velocity = 0.0;
    if (c.wall[1] && touches(yp, c.lbb[1], c.tfr[1])) {
        vx *= drag;
        vy += velocity * xDrag;
        if (3 == D) vz *= drag;
        yDrag = drag;
    }
    velocity = 0.0;
    if (3 == D && c.wall[2] && touches(zp, c.lbb[2], c.tfr[2])) {
        vx *= drag;
        vy *= drag;
        vz += velocity * xDrag * yDrag;
    }
}

struct CorrAcc {
    double s_v, max_err, max_r, max_exp;
    int n_del;
};

// What the gas exchange takes from a foam's sums, the same for every bubble.
struct GasSums {
    double inv_rho, flux;
};

__device__ __forceinline__ GasSums gas_sums(const Consts &c, int n, double s_a, double s_ar,
                                            double s_oa, double s_oar) {
    return GasSums{(s_ar - s_oar) / (s_a - s_oa), c.kappa * c.avg_area_in * n / s_a};
}

// MIXED: no FP64 predicted record is stored (recompute it) and velocities
// are FP32.  WALLS false: no foam of the launch has a wall (the wall code,
// and its registers, compiled out).  sums() gives the foam's GasSums; it is
// called behind the loads of the first bubble.
template <int D, bool GAS, bool PATH, bool MIXED, bool WALLS, bool OWN, typename Sums>
__device__ __forceinline__ void correct_range(const Consts &c, const Roles &R, const Scratch &S,
                                              double dt, int base, int ipt, int n, Sums &&sums,
                                              CorrAcc &a) {
    typedef typename std::conditional<MIXED, float, double>::type V;
    const double h = 0.5 * dt;
    const bool walls = WALLS && (c.wall[0] || c.wall[1] || (3 == D && c.wall[2]));
    GasSums gs{0.0, 0.0};
    for (int k = 0; k < ipt; ++k) {
        const int i = base + k * kBlock + (int)threadIdx.x;
        const bool valid = i < n;
        if ((!OWN || k > 0) && !valid) break;  // (OWN: the whole workgroup calls sums())
        const int at = valid ? i : 0;
        const D4 pp = MIXED ? predicted<D, GAS, V>(R, h, at) : S.p4[at];
        const double pv[3] = {pp.x, pp.y, pp.z};
        double vp[3], xo[3], v[3], sv[4];
#pragma unroll
        for (int q = 0; q < D; ++q) {
            vp[q] = (double)field<V>(R.vp[q])[at];
            xo[q] = R.x[q][at];
            v[q] = (double)field<V>(R.v[q])[at];
            sv[q] = (double)field<V>(R.saved[q])[at];
        }
        double ov = 0.0, vpr = 0.0, ro = 0.0, vr0 = 0.0;
        if (GAS) {
            ov = (double)field<V>(S.ov)[at];
            vpr = (double)field<V>(R.vp[3])[at];
            ro = R.x[3][at];
            vr0 = (double)field<V>(R.v[3])[at];
            sv[3] = (double)field<V>(R.saved[3])[at];
        }
        const double path = PATH ? R.path[at] : 0.0;
        const double err = (double)field<V>(R.err)[at];
        if (0 == k) gs = sums();
        if (OWN && !valid) break;
        if (walls) {
            double vz = 3 == D ? vp[2] : 0.0;
            add_wall_velocity<D>(c, pp.x, pp.y, pp.z, pp.r, vp[0], vp[1], vz);
            if (3 == D) vp[2] = vz;
#pragma unroll
            for (int q = 0; q < D; ++q) {
                vp[q] = (double)(V)vp[q];  // the stored value drives the corrector
                stream_store(field<V>(R.vp[q]) + i, (V)vp[q]);
            }
        }
        double e = 0.0, dist = 0.0;
        double xc[3];
#pragma unroll
        for (int q = 0; q < D; ++q) {
            const double pred = pv[q];
            const double corr = xo[q] + h * (v[q] + vp[q]);
            xc[q] = corr;
            stream_store(R.xp[q] + i, corr);
            e = fmax(e, fabs(pred - corr));
            const double t = corr - sv[q];
            dist += t * t;
        }
        dist = sqrt(dist);
        int dele = 0;
        if (GAS) {
            double r = pp.r;
            double area = 2.0 * kPi * r;
            if (3 == D) area *= 2.0 * r;
            double vr = gs.inv_rho - rcp_nr(r);
            vr *= gs.flux * (area - ov);
            vr += vpr;
            vr *= c.k_param * rcp_nr(area);
            stream_store(field<V>(R.vp[3]) + i, (V)vr);
            vr = (double)(V)vr;  // the stored value drives the corrector
            const double pred = r;
            const double corr = ro + h * (vr0 + vr);
            stream_store(R.xp[3] + i, corr);
            e = fmax(e, fabs(pred - corr));
            dist += corr - sv[3];
            r = corr;
            if (r > c.min_rad) {
                double vol = r * r;
                if (3 == D) vol *= r;
                a.s_v += vol;
            } else {
                dele = 1;
                a.n_del += 1;
            }
            a.max_r = fmax(a.max_r, r);
        } else {
            stream_store(R.xp[3] + i, pp.r);  // radius unchanged without gas exchange
        }
        stream_store(S.del + i, (uint8_t)dele);
        a.max_exp = fmax(a.max_exp, dist);
        if (PATH) {
            double t = xo[0] - xc[0];
            double pd = t * t;
            t = xo[1] - xc[1];
            pd += t * t;
            if (3 == D) {
                t = xo[2] - xc[2];
                pd += t * t;
            }
            stream_store(R.path_new + i, path + sqrt(pd));
        }
        // the largest error so far: most bubbles' stands, and a store less is
        // 1% of the large runs (256 foams 31.54 -> 31.22 ms, 3D 1e6 20.25 -> 20.05);
        // negated, so that a NaN is replaced as fmax does
        if (!(e <= err)) stream_store(field<V>(R.err) + i, (V)fmax(e, err));
        a.max_err = fmax(a.max_err, e);
    }
}

// dt controller and commit: reference src/simulator.cu:239-246, :258-321, by
// one thread, from copies of the header's parts that were read before (the
// pointers' rotation in place took a load's time for each buffer: a load does
// not pass the stores before it).  Returns whether the step removes bubbles that
// the calling workgroup plans.
__device__ __forceinline__ bool control(Foam *F, const Dyn &was, const Roles &R, uint32_t flags,
                                        const CorrAcc &a) {
    Dyn &d = F->d;
    const Consts &c = F->c;
    const double tol = c.tol, skin = c.skin;
    const int dim = c.dim;
    const bool too_large = a.max_err > tol;
    const bool increase = a.max_err < 0.45 * tol && was.dt < 10;
    double ndt = was.dt;
    if (too_large) {
        ndt = was.dt * 0.37;
    } else if (increase) {
        ndt = was.dt * 1.269;
    }
    d.s_v = a.s_v;
    d.max_err = a.max_err;
    d.max_r = a.max_r;
    d.max_exp = a.max_exp;
    d.n_del = a.n_del;
    d.marked = 1;
    d.attempts = was.attempts + 1;
    d.dt = ndt;
    d.accepted = too_large ? 0 : 1;
    if (too_large || !(flags & kCommit)) {
        d.need_remove = 0;  // the last one is done
        return false;
    }
    const bool gas = (flags & kGas) != 0;
    Roles &W = F->r;
    for (int k = 0; k < 4; ++k) {
        if (2 == k && 2 == dim) continue;
        if (3 == k && !gas) continue;
        W.vo[k] = R.v[k];
        W.v[k] = R.vp[k];
        W.vp[k] = R.vo[k];
        W.x[k] = R.xp[k];
        W.xp[k] = R.x[k];
    }
    if (flags & kPath) {
        W.path = R.path_new;
        W.path_new = R.path;
    }
    // the stop rules look at the new state
    Dyn now = was;
    now.max_r = a.max_r;
    now.steps = was.steps + 1;
    const double frac = was.time_frac + ndt;
    const uint64_t whole = (uint64_t)frac;
    now.time_int = was.time_int + whole;
    now.time_frac = frac - (double)whole;
    d.steps = now.steps;
    d.bubble_steps = was.bubble_steps + (double)was.count;
    d.time_int = now.time_int;
    d.time_frac = now.time_frac;
    const bool removes = gas && a.n_del > 0;
    if (gas) d.max_r_cell = a.max_r;
    const bool launched = removes && a.n_del > kBlock && F->nblk > kControlPlans;
    d.need_remove = !removes ? 0 : launched ? kMarked : kPlanned;
    d.need_search = a.max_exp >= 0.5 * skin ? 1 : 0;
    d.ts_min = fmin(was.ts_min, ndt);
    d.ts_max = fmax(was.ts_max, ndt);
    d.ts_sum = was.ts_sum + ndt;
    if (stop_reached(now)) d.halt = 1;
    return removes && !launched;
}

template <int D, bool M, bool W, bool OWN, typename Sums>
__device__ __forceinline__ void correct_dispatch(const Consts &c, const Roles &R, const Scratch &S,
                                                 double dt, int base, int ipt, int n,
                                                 uint32_t flags, Sums &&sums, CorrAcc &a) {
    const bool gas = (flags & kGas) != 0, path = (flags & kPath) != 0;
    if (gas) {
        if (path) correct_range<D, true, true, M, W, OWN>(c, R, S, dt, base, ipt, n, sums, a);
        else correct_range<D, true, false, M, W, OWN>(c, R, S, dt, base, ipt, n, sums, a);
    } else {
        if (path) correct_range<D, false, true, M, W, OWN>(c, R, S, dt, base, ipt, n, sums, a);
        else correct_range<D, false, false, M, W, OWN>(c, R, S, dt, base, ipt, n, sums, a);
    }
}

// One kernel per precision (MIXED: FP32 velocity buffers, recomputed
// prediction), per wall presence (WALLS: some foam of the launch has a
// wall) and per place of the foam's sums (OWN: formed here, behind the block's
// own loads; else k_sums formed them), so that none pays the registers of
// another.
template <bool MIXED, bool WALLS, bool OWN>
__global__ __launch_bounds__(kBlock) void k_correct(Foam *foams, const int2 *bt, uint32_t flags) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (standing(F->d)) return;
    const int n = F->d.count, ipt = F->ipt;
    const Consts c = F->c;
    const Roles R = F->r;
    const Scratch S = F->s;
    const double dt = F->d.dt;
    const int base = cx.lb * kBlock * ipt;
    auto sums = [&]() {
        if (!OWN) return gas_sums(c, n, F->d.s_a, F->d.s_ar, F->d.s_oa, F->d.s_oar);
        double r[4];
        block_foam_sums(S.part, flags & kQuad ? quad_parts(S) : nullptr, F->nblk, r);
        // for the host; the other blocks use their own
        if (0 == cx.lb && 0 == threadIdx.x) {
            F->d.s_a = r[0];
            F->d.s_ar = r[1];
            F->d.s_oa = r[2];
            F->d.s_oar = r[3];
        }
        return gas_sums(c, n, r[0], r[1], r[2], r[3]);
    };
    CorrAcc a{0.0, 0.0, 0.0, 0.0, 0};
    if (3 == c.dim)
        correct_dispatch<3, MIXED, WALLS, OWN>(c, R, S, dt, base, ipt, n, flags, sums, a);
    else
        correct_dispatch<2, MIXED, WALLS, OWN>(c, R, S, dt, base, ipt, n, flags, sums, a);
    // the volume sum, then the maxima of error, radius and expansion
    double r4[4] = {a.s_v, a.max_err, a.max_r, a.max_exp};
    int nd = a.n_del;
    block_reduce_t0(r4, 0xeu, nd);
    if (threadIdx.x == 0) {
        S.part[cx.lb * kPartD + 4] = r4[0];
        S.part[cx.lb * kPartD + 5] = r4[1];
        S.part[cx.lb * kPartD + 6] = r4[2];
        S.part[cx.lb * kPartD + 7] = r4[3];
        S.part_i[cx.lb * kPartI + 0] = nd;
    }
}

// One block per foam: reduce the corrector partials, then the dt controller
// and (when committing) the role rotation and the plan of a removal, which
// the next launch applies.
__device__ __forceinline__ void control_block(Foam *F, uint32_t flags) {
    if (standing(F->d)) {
        // the removal of its last step is done, or waits for the search phase
        // (kApply, or for its plan)
        if (0 == threadIdx.x && !(flags & kApply) && kPlanned == F->d.need_remove)
            F->d.need_remove = 0;
        return;
    }
    __shared__ int s_del;
    __shared__ DeletedBlocks s_blocks;
    if (0 == threadIdx.x) s_blocks.m = 0;
    __syncthreads();
    const Dyn was = F->d;
    const Roles R = F->r;
    const int n = was.count;
    // the volume sum, the maxima of error, radius and expansion, the
    // deletion count
    double r[4];
    int nd;
    const double *const part = F->s.part;
    reduce_parts4(
        [&](int b, double (&v)[4]) {
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = part[b * kPartD + 4 + k];
        },
        F->s.part_i, [&](int b, int c) { s_blocks.add(b, c); }, F->nblk, 0xeu, r, nd);
    if (threadIdx.x == 0) {
        CorrAcc t;
        t.s_v = r[0];
        t.max_err = r[1];
        t.max_r = r[2];
        t.max_exp = r[3];
        t.n_del = nd;
        s_del = control(F, was, R, flags, t) ? nd : 0;
    }
    __syncthreads();
    nd = s_del;
    if (nd > 0) plan_removal(F, s_blocks, n, nd);
}

// mirror: pinned host memory that receives the foams' scalars as they are then
// (a launch less than reading them afterwards), or null.
__global__ __launch_bounds__(kBlock) void k_control(Foam *foams, uint32_t flags, Dyn *mirror) {
    Foam *F = touch_header(foams + blockIdx.x);
    control_block(F, flags);
    if (!mirror) return;
    __syncthreads();
    for (int w = threadIdx.x; w < (int)(sizeof(Dyn) / 8); w += kBlock)
        reinterpret_cast<uint64_t *>(mirror + blockIdx.x)[w] =
            reinterpret_cast<const volatile uint64_t *>(&F->d)[w];
}

// ---------------------------------------------------------------- launches
void launch_predict(const Grid &g, uint32_t flags) {
    if (flags & kApply)
        hipLaunchKernelGGL(k_predict<true>, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams,
                           g.bt_bub, flags);
    else
        hipLaunchKernelGGL(k_predict<false>, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams,
                           g.bt_bub, flags);
}

void launch_pair(const Grid &g, uint32_t flags) {
    if (g.quad) {
        if (flags & kFlow)
            hipLaunchKernelGGL(k_pair_quad<true>, dim3(4 * g.nb_bub), dim3(kBlock), 0, g.stream,
                               g.foams, g.bt_bub, flags);
        else
            hipLaunchKernelGGL(k_pair_quad<false>, dim3(4 * g.nb_bub), dim3(kBlock), 0, g.stream,
                               g.foams, g.bt_bub, flags);
        return;
    }
    if (flags & kFlow)
        hipLaunchKernelGGL(k_pair<true>, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams,
                           g.bt_bub, flags);
    else
        hipLaunchKernelGGL(k_pair<false>, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams,
                           g.bt_bub, flags);
}

void launch_sums(const Grid &g) {
    if (g.big)
        hipLaunchKernelGGL(k_sums, dim3(g.nfoams), dim3(kBlock), 0, g.stream, g.foams, g.quad);
}

// AB2 bootstrap of init (reference src/simulator.cu:739-787): the Euler step
// of the predicted record by the pair velocities in vp (kernel euler,
// src/kernels.cu:958-968), then those velocities become the old ones.  The
// record holds the current positions (zero velocities at creation); in mixed
// precision the stepped FP64 position is recoded into the fixed-point record.
__global__ __launch_bounds__(kBlock) void k_euler(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    const int n = F->d.count, ipt = F->ipt, D = F->c.dim;
    const Consts c = F->c;
    const Roles R = F->r;
    const Scratch S = F->s;
    const double ts = F->d.dt;
    const int base = cx.lb * kBlock * ipt;
    for (int k = 0; k < ipt; ++k) {
        const int i = base + k * kBlock + (int)threadIdx.x;
        if (i >= n) break;
        if (S.q4) {
            Q4 q = S.q4[i];
            auto code = [&](int a) {
                const double x = R.x[a][i] + (double)field<float>(R.vp[a])[i] * ts;
                return fixed_code(x, c.lbb[a], c.interval[a], c.wall[a] != 0);
            };
            q.x = code(0);
            q.y = code(1);
            if (3 == D) q.z = code(2);
            S.q4[i] = q;
        } else {
            D4 p = S.p4[i];
            p.x += field<double>(R.vp[0])[i] * ts;
            p.y += field<double>(R.vp[1])[i] * ts;
            if (3 == D) p.z += field<double>(R.vp[2])[i] * ts;
            S.p4[i] = p;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_old_from_pair(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    const int n = F->d.count, ipt = F->ipt, D = F->c.dim;
    const Roles R = F->r;
    const bool mixed = F->s.q4 != nullptr;
    const int base = cx.lb * kBlock * ipt;
    for (int k = 0; k < ipt; ++k) {
        const int i = base + k * kBlock + (int)threadIdx.x;
        if (i >= n) break;
        for (int a = 0; a < D; ++a) {
            if (mixed) field<float>(R.vo[a])[i] = field<float>(R.vp[a])[i];
            else field<double>(R.vo[a])[i] = field<double>(R.vp[a])[i];
        }
    }
}

void launch_bootstrap(const Grid &g, bool mixed) {
    launch_predict(g, 0);  // zero velocities: the record holds the positions
    if (mixed) launch_pair_mixed(g, 0);
    else launch_pair(g, 0);
    hipLaunchKernelGGL(k_euler, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    if (mixed) launch_pair_mixed(g, 0);
    else launch_pair(g, 0);
    hipLaunchKernelGGL(k_old_from_pair, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams,
                       g.bt_bub);
}

void launch_correct(const Grid &g, uint32_t flags, bool mixed, bool control, Dyn *mirror) {
    const dim3 grid(g.nb_bub), block(kBlock);
    if (g.quad) flags |= kQuad;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, g.stream, g.foams, g.bt_bub, flags);
    };
    if (g.big) {
        if (mixed) g.walls ? launch(k_correct<true, true, false>) : launch(k_correct<true, false, false>);
        else g.walls ? launch(k_correct<false, true, false>) : launch(k_correct<false, false, false>);
    } else {
        if (mixed) g.walls ? launch(k_correct<true, true, true>) : launch(k_correct<true, false, true>);
        else g.walls ? launch(k_correct<false, true, true>) : launch(k_correct<false, false, true>);
    }
    if (control)
        hipLaunchKernelGGL(k_control, dim3(g.nfoams), dim3(kBlock), 0, g.stream, g.foams, flags,
                           mirror);
}

}  // namespace cubble_amd
