// remove_kernels.hip -- removeBubbles (reference src/simulator.cu:180-190).
//
//   the plan:    the sorted deletion list, the moves -- the k-th hole below
//                the new count receives the k-th surviving bubble counted
//                from the back (reference swapDataCountPairs,
//                src/kernels.cu:775-857) --, the marks on the lists that
//                change, and the volume-fix multiplier M / S_V^(1/D)
//                (src/kernels.cu:861-867).  By one workgroup per foam at the
//                end of k_control (remove_plan.hpp), or by k_rm_emit and
//                k_rm_plan for many bubbles of a large foam and for a removal
//                asked for by itself
//   apply_removal (remove_apply.hpp), in k_predict of the foam's next attempt,
//                or k_rm_apply: every slot below the new count applies the
//                volume fix; a hole pulls its tail survivor's state and list, a marked bubble
//                filters its own list -- deleted neighbours dropped, moved
//                ones mapped to their new slots, kept ascending (reference
//                addVolumeFixPairs, src/kernels.cu:859-936)
//
// The reference appends the deletion list with an atomic counter, so its
// hole / survivor pairing depends on thread timing; a sorted list makes the
// pairing deterministic.  Its race-prone pair swap-from-the-back
// (src/kernels.cu:873-909) is replaced by per-bubble list filtering, done
// only for the few lists a removal touches.
#include "dev_util.hpp"
#include "launch.hpp"
#include "remove_apply.hpp"
#include "remove_plan.hpp"

namespace cubble_amd {

constexpr int kFilter = 8;  // list entries loaded together when walking a list

// The deletion marks in each block, for a removal asked for by itself: the
// corrector's counts are of the launch shape and the count it ran with, and
// the planner indexes with what the marks it finds give.
__global__ __launch_bounds__(kBlock) void k_rm_count(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (kMarked != F->d.need_remove) return;
    const int n = F->d.count, ipt = F->ipt;
    int c = 0;
    for (int k = 0; k < ipt; ++k) {
        const int i = (cx.lb * ipt + k) * kBlock + (int)threadIdx.x;
        c += i < n && F->s.del[i] ? 1 : 0;
    }
    c = block_sum_i(c);
    if (0 == threadIdx.x) F->s.part_i[cx.lb * kPartI] = c;
}

// The deletion list, ascending, and the marks on the lists that change: those
// of the neighbours of the deleted bubbles and of the survivors past the new
// count, which move.  Every block takes its own bubbles; its offset is the sum
// of the counts of the blocks before.  Twice the pairs that go (those of the
// deleted bubbles, each once) to the block's partials: two for a list entry of
// a deleted bubble, less one for an entry that is deleted too.
__global__ __launch_bounds__(kBlock) void k_rm_emit(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (kMarked != F->d.need_remove) return;
    const Scratch S = F->s;
    const int n = F->d.count, ipt = F->ipt, nblk = F->nblk;
    const size_t cap = (size_t)F->cap;
    int before = 0, all = 0;
    for (int b = threadIdx.x; b < nblk; b += kBlock) {
        const int c = S.part_i[b * kPartI];
        all += c;
        before += b < cx.lb ? c : 0;
    }
    int off = block_sum_i(before);
    const int nnew = n - block_sum_i(all);
    const int base = cx.lb * ipt * kBlock;
    int gone = 0;
    if (S.part_i[cx.lb * kPartI] > 0 || base + ipt * kBlock > nnew) {  // uniform
        for (int k = 0; k < ipt; ++k) {
            const int i = base + k * kBlock + (int)threadIdx.x;
            const int f = i < n && S.del[i] ? 1 : 0;
            int tot = 0;
            const int pre = block_excl_scan(f, tot);
            if (f) S.del_list[off + pre] = i;
            off += tot;
            auto mark = [&](int j, int f) {
                if (j < nnew) S.dirty[j] = 1;  // same value from every writer
                if (f) gone += S.del[j] ? 1 : 2;
            };
            int m = i < n && (f || i >= nnew) ? S.nn[i] : 0;
            // a long list by the whole wave
            for (unsigned long long t = __builtin_amdgcn_ballot_w64(m > 64); t; t &= t - 1ull) {
                const int l = __builtin_ctzll(t);
                const int b = __builtin_amdgcn_readlane(i, l), g = __builtin_amdgcn_readlane(f, l);
                const int len = __builtin_amdgcn_readlane(m, l);
                for (int q = (int)(threadIdx.x & 63); q < len; q += 64)
                    mark(S.nbr[(size_t)q * cap + b], g);
            }
            if (m > 64) m = 0;
            for (int q0 = 0; q0 < m; q0 += kFilter) {
                int js[kFilter];
#pragma unroll
                for (int u = 0; u < kFilter; ++u)
                    js[u] = q0 + u < m ? S.nbr[(size_t)(q0 + u) * cap + i] : -1;
#pragma unroll
                for (int u = 0; u < kFilter; ++u)
                    if (js[u] >= 0) mark(js[u], f);
            }
        }
    }
    gone = block_sum_i(gone);
    if (0 == threadIdx.x) S.part_i[cx.lb * kPartI + 1] = gone;
}

// The moves and the counters, one workgroup per foam.
__global__ __launch_bounds__(kBlock) void k_rm_plan(Foam *foams) {
    Foam *F = foams + blockIdx.x;
    if (kMarked != F->d.need_remove) return;
    const Scratch S = F->s;
    const int n = F->d.count;
    int nd = 0, gone = 0;
    for (int b = threadIdx.x; b < F->nblk; b += kBlock) {
        nd += S.part_i[b * kPartI];
        gone += S.part_i[b * kPartI + 1];
    }
    nd = block_sum_i(nd);
    gone = block_sum_i(gone);
    const int h = plan_moves(S, n, nd);
    if (0 == threadIdx.x) {
        commit_removal(F, F->d.s_v, h, n - nd, gone / 2);
        F->d.need_remove = kPlanned;
    }
}

// Removals of the last attempt before a search phase, and of foams that stand
// still; k_predict carries out the others.
__global__ __launch_bounds__(kBlock) void k_rm_apply(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    if (kPlanned == cx.F->d.need_remove) apply_removal(cx.F, cx.lb);
}

void launch_apply(const Grid &g) {
    hipLaunchKernelGGL(k_rm_apply, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
}

void launch_plan(const Grid &g) {
    hipLaunchKernelGGL(k_rm_emit, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    hipLaunchKernelGGL(k_rm_plan, dim3(g.nfoams), dim3(kBlock), 0, g.stream, g.foams);
}

void launch_remove(const Grid &g) {
    hipLaunchKernelGGL(k_rm_count, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    launch_plan(g);
    launch_apply(g);
}

}  // namespace cubble_amd
