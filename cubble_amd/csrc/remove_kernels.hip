// remove_kernels.hip -- removeBubbles (reference src/simulator.cu:180-190).
//
//   plan_removal (remove_plan.hpp), by one workgroup per foam: at the end of
//                k_control, or k_rm_plan for a removal asked for by itself.
//                The sorted deletion list, the moves -- the k-th hole below
//                the new count receives the k-th surviving bubble counted
//                from the back (reference swapDataCountPairs,
//                src/kernels.cu:775-857) --, the marks on the lists that
//                change, and the volume-fix multiplier M / S_V^(1/D)
//                (src/kernels.cu:861-867)
//   apply_removal (remove_apply.hpp), in k_predict of the foam's next attempt,
//                or k_rm_apply: every slot below the new count applies the volume fix; a hole
//                pulls its tail survivor's state and list, a marked bubble
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

// The deletion marks in each block, for a removal asked for by itself: the
// corrector's counts are of the launch shape and the count it ran with, and
// the planner indexes with what the marks it finds give.
__global__ __launch_bounds__(kBlock) void k_rm_count(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    Foam *F = cx.F;
    if (!F->d.need_remove) return;
    const int n = F->d.count, ipt = F->ipt;
    int c = 0;
    for (int k = 0; k < ipt; ++k) {
        const int i = (cx.lb * ipt + k) * kBlock + (int)threadIdx.x;
        c += i < n && F->s.del[i] ? 1 : 0;
    }
    c = block_sum_i(c);
    if (0 == threadIdx.x) F->s.part_i[cx.lb * kPartI] = c;
}

// A removal asked for by itself (cubble_remove_bubbles); k_control plans its
// own.
__global__ __launch_bounds__(kBlock) void k_rm_plan(Foam *foams) {
    Foam *F = foams + blockIdx.x;
    if (!F->d.need_remove) return;
    __shared__ DeletedBlocks s_blocks;
    if (0 == threadIdx.x) s_blocks.m = 0;
    __syncthreads();
    int nd = 0;
    for (int b = threadIdx.x; b < F->nblk; b += kBlock) {
        const int c = F->s.part_i[b * kPartI];
        if (c > 0) s_blocks.add(b, c);
        nd += c;
    }
    nd = block_sum_i(nd);  // (and every thread's blocks are in the list)
    plan_removal(F, s_blocks, F->d.count, nd);
}

// Removals of the last attempt before a search phase, and of foams that stand
// still; k_predict carries out the others.
__global__ __launch_bounds__(kBlock) void k_rm_apply(Foam *foams, const int2 *bt) {
    const Ctx cx = bubble_ctx(foams, bt);
    if (cx.F->d.need_remove) apply_removal(cx.F, cx.lb);
}

void launch_apply(const Grid &g) {
    hipLaunchKernelGGL(k_rm_apply, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
}

void launch_remove(const Grid &g) {
    hipLaunchKernelGGL(k_rm_count, dim3(g.nb_bub), dim3(kBlock), 0, g.stream, g.foams, g.bt_bub);
    hipLaunchKernelGGL(k_rm_plan, dim3(g.nfoams), dim3(kBlock), 0, g.stream, g.foams);
    launch_apply(g);
}

}  // namespace cubble_amd
