// remove_plan.hpp -- planning a removal, by one workgroup of the foam: the
// sorted deletion list, the moves of the tail survivors into the holes, the
// marks on the neighbour lists that change, the new count and pair count, and
// the volume-fix multiplier (reference src/kernels.cu:775-867).  k_rm_apply
// then does the work on every slot.
//
// A removal touches few bubbles (one to a few dozen of 1e5 .. 1e7), so its
// planning is a chain of short dependent loads, not work: one workgroup walks
// it with a barrier between the stages (8-10 us with a removal of a few
// bubbles, 0 without), where four launches cost 3-4 us each whether or not a
// foam had a removal (1e5 foam, mixed: 15 us per attempt group with one).
#pragma once

#include "dev_util.hpp"

namespace cubble_amd {

// Blocks holding deletions that the planner sorts in LDS; a removal spread
// over more blocks (thousands of bubbles in one step) takes the block by block
// walk.
constexpr int kPlanBlocks = 1024;

// The deletion list, ascending, from the corrector's marks and block counts.
__device__ __forceinline__ void emit_deleted(const Scratch &S, int n, int ipt, int nblk) {
    __shared__ int s_blk[kPlanBlocks], s_num[kPlanBlocks], s_m;
    if (0 == threadIdx.x) s_m = 0;
    __syncthreads();
    for (int b = threadIdx.x; b < nblk; b += kBlock) {
        const int c = S.part_i[b * kPartI + 0];
        if (c > 0) {
            const int k = atomicAdd(&s_m, 1);
            if (k < kPlanBlocks) {
                s_blk[k] = b;
                s_num[k] = c;
            }
        }
    }
    __syncthreads();
    const int m = s_m, lane = (int)(threadIdx.x & 63);
    if (m <= kPlanBlocks) {
        // one wave per block with deletions: its offset is the sum of the
        // counts of the blocks before it
        for (int e = threadIdx.x >> 6; e < m; e += kWaves) {
            const int b = s_blk[e];
            int before = 0;
            for (int f = lane; f < m; f += 64) before += s_blk[f] < b ? s_num[f] : 0;
            int off = wave_sum_i(before);
            const int base = b * kBlock * ipt;
            for (int k = 0; k < kBlock * ipt; k += 64) {
                const int i = base + k + lane;
                const bool f = i < n && S.del[i];
                const unsigned long long hits = __builtin_amdgcn_ballot_w64(f);
                if (f) S.del_list[off + __popcll(hits & ((1ull << lane) - 1ull))] = i;
                off += __popcll(hits);
            }
        }
        return;
    }
    int off = 0;
    for (int b = 0; b < nblk; ++b) {
        if (0 == S.part_i[b * kPartI + 0]) continue;  // uniform
        for (int k = 0; k < ipt; ++k) {
            const int i = (b * ipt + k) * kBlock + (int)threadIdx.x;
            const int f = i < n && S.del[i] ? 1 : 0;
            int tot = 0;
            const int pre = block_excl_scan(f, tot);
            if (f) S.del_list[off + pre] = i;
            off += tot;
        }
    }
}

// Plans the removal of the `nd` marked bubbles of the foam's n, and commits
// the counters.  The whole workgroup (kBlock threads) calls it.
__device__ __forceinline__ void plan_removal(Foam *F, int n, int nd) {
    const Scratch S = F->s;
    const int nnew = n - nd;
    const size_t cap = (size_t)F->cap;
    emit_deleted(S, n, F->ipt, F->nblk);
    __syncthreads();
    // the k-th hole below the new count receives the k-th surviving bubble
    // counted from the back
    int below = 0;
    for (int k = threadIdx.x; k < nd; k += kBlock) below += S.del_list[k] < nnew ? 1 : 0;
    const int h = block_sum_i(below);
    int got = 0;
    for (int top = n - 1; got < h && top >= nnew; top -= kBlock) {
        const int i = top - (int)threadIdx.x;
        const int f = (i >= nnew && !S.del[i]) ? 1 : 0;
        int tot = 0;
        const int pre = block_excl_scan(f, tot);
        if (f && got + pre < h) {
            S.plan_src[got + pre] = i;
            S.moved_to[i - nnew] = S.del_list[got + pre];
        }
        got += tot;
    }
    __syncthreads();
    // mark the lists that change, those of the neighbours of the deleted
    // bubbles and of the moving survivors: 16 lanes per bubble.  The pairs
    // that go are those of the deleted bubbles, each once: their list entries,
    // less half of the entries that are deleted themselves.
    int gone = 0, both = 0;
    const int items = nd + h;
    for (int t = threadIdx.x >> 4; t < items; t += kBlock / 16) {
        const int s = t < nd ? S.del_list[t] : S.plan_src[t - nd];
        const int m = S.nn[s];
        for (int q = threadIdx.x & 15; q < m; q += 16) {
            const int j = S.nbr[(size_t)q * cap + s];
            if (j < nnew) S.dirty[j] = 1;  // same value from every writer
            if (t < nd) {
                gone += 1;
                both += S.del[j] ? 1 : 0;
            }
        }
    }
    gone = block_sum_i(gone);
    both = block_sum_i(both);
    if (0 == threadIdx.x) {
        Dyn &d = F->d;
        double vm = 3 == F->c.dim ? 1.0 / det_cbrt(d.s_v) : 1.0 / sqrt(d.s_v);
        vm *= F->c.vol_mul;
        d.vol_fix = vm;
        d.n_holes = h;
        d.count = nnew;
        d.removals += 1;
        d.num_pairs -= gone - both / 2;
        if (d.count_stop > 0 && nnew <= d.count_stop) d.halt = 1;
    }
}

}  // namespace cubble_amd
