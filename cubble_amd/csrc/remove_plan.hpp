// remove_plan.hpp -- planning a removal, by one workgroup of the foam: the
// sorted deletion list, the moves of the tail survivors into the holes, the
// marks on the neighbour lists that change, the new count and pair count, and
// the volume-fix multiplier (reference src/kernels.cu:775-867).  apply_removal
// then does the work on every slot.
//
// A removal touches few bubbles (one to a few dozen of 1e5 .. 1e7), so its
// planning is a chain of short dependent loads, not work: one workgroup walks
// it with a barrier between the stages, where four launches cost 3-4 us each
// whether or not a foam had a removal (1e5 foam, mixed: 15 us per attempt group
// with one).  Up to kBlock deletions, plan_few keeps the lists in LDS and loads
// ahead what does not depend on them; more take plan_many.
//
// Thousands of deletions in one step (bubbles set below the smallest radius,
// coarsening of a large foam at a large time step) are work, which one
// workgroup takes too long for; foams of more than kControlPlans blocks leave
// them to the launches of remove_kernels.hip.
#pragma once

#include "dev_util.hpp"

namespace cubble_amd {

// Most blocks with deletions in a removal planned here: foams of that many
// blocks, or removals of at most kBlock bubbles.
constexpr int kPlanBlocks = kControlPlans;
static_assert(kPlanBlocks >= kBlock, "a deletion per block");

// The blocks with deletions, as k_control comes to their counts.
struct DeletedBlocks {
    int blk[kPlanBlocks], num[kPlanBlocks], m;
    __device__ __forceinline__ void add(int b, int c) {
        const int k = atomicAdd(&m, 1);
        if (k < kPlanBlocks) {
            blk[k] = b;
            num[k] = c;
        }
    }
};

// The deletion list, ascending, from the corrector's marks (and into `lds`, if
// given, which has room for it): by one wave per block with deletions, whose
// offset is the sum of the counts of the blocks before it.  The marks are
// bytes, four a lane.  Ends without a barrier.
__device__ __forceinline__ void emit_blocks(const Scratch &S, const DeletedBlocks &B, int n,
                                            int ipt, int *lds) {
    const int lane = (int)threadIdx.x & 63;
    for (int e = (int)threadIdx.x >> 6; e < B.m; e += kWaves) {
        const int b = B.blk[e];
        int before = 0;
        for (int f = lane; f < B.m; f += 64) before += B.blk[f] < b ? B.num[f] : 0;
        int off = wave_sum_i(before);
        for (int k0 = 0; k0 < ipt; k0 += 4) {
            uint32_t w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int base = (b * ipt + min(k0 + u, ipt - 1)) * kBlock;
                // (marks are padded to whole words)
                w[u] = base + 4 * lane < n
                           ? *reinterpret_cast<const uint32_t *>(S.del + base + 4 * lane) : 0u;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i0 = (b * ipt + k0 + u) * kBlock + 4 * lane;
                if (k0 + u >= ipt) w[u] = 0u;
                if (i0 + 4 > n) w[u] = i0 < n ? w[u] & ((1u << 8 * (n - i0)) - 1u) : 0u;
                if (__builtin_amdgcn_ballot_w64(w[u] != 0u) == 0ull) continue;
                const int c = __popc(w[u]);  // marks are 0 or 1
                const unsigned long long below = (1ull << lane) - 1ull;
                int at = off;
#pragma unroll
                for (int bit = 0; bit < 3; ++bit) {
                    const unsigned long long h = __builtin_amdgcn_ballot_w64((c >> bit) & 1);
                    at += __popcll(h & below) << bit;
                    off += __popcll(h) << bit;
                }
                for (int v = 0; v < 4; ++v)
                    if ((w[u] >> (8 * v)) & 1u) {
                        if (lds) lds[at] = i0 + v;
                        S.del_list[at++] = i0 + v;
                    }
            }
        }
    }
}

// What a planned removal changes in the foam's header; one thread.
__device__ __forceinline__ void commit_removal(Foam *F, double s_v, int h, int nnew, int pairs) {
    Dyn &d = F->d;
    double vm = 3 == F->c.dim ? 1.0 / det_cbrt(s_v) : 1.0 / sqrt(s_v);
    vm *= F->c.vol_mul;
    d.vol_fix = vm;
    d.n_holes = h;
    d.count = nnew;
    d.removals += 1;
    d.marked = 0;
    d.num_pairs -= pairs;
    if (d.count_stop > 0 && nnew <= d.count_stop) d.halt = 1;
}

// The moves, from the deletion list of `nd` bubbles of n: the k-th hole below
// the new count receives the k-th surviving bubble counted from the back.
// Returns the number of holes.  By the whole workgroup; ends without a barrier.
__device__ __forceinline__ int plan_moves(const Scratch &S, int n, int nd) {
    const int nnew = n - nd;
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
    return h;
}

// Plans the removal of the `nd` marked bubbles of the foam's n, which are in
// the blocks B, and commits the counters.  The whole workgroup (kBlock threads)
// calls it.
__device__ __forceinline__ void plan_many(Foam *F, const DeletedBlocks &B, int n, int nd) {
    const Scratch S = F->s;
    const int nnew = n - nd;
    const size_t cap = (size_t)F->cap;
    emit_blocks(S, B, n, F->ipt, nullptr);
    __syncthreads();
    const int h = plan_moves(S, n, nd);
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
    if (0 == threadIdx.x) commit_removal(F, F->d.s_v, h, nnew, gone - both / 2);
}

// The same for nd <= kBlock deletions (in as many blocks at most).
__device__ __forceinline__ void plan_few(Foam *F, const DeletedBlocks &B, int n, int nd) {
    __shared__ int s_del[kBlock], s_src[kBlock], s_sum[2][kWaves];
    const Scratch S = F->s;
    const int nnew = n - nd, nbr_cap = F->nbr_cap;
    const size_t cap = (size_t)F->cap;
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    const double s_v = F->d.s_v;
    // the tail [nnew, n), from the back
    const int top = n - 1 - t;
    const int stays = t < nd && !S.del[max(top, 0)] ? 1 : 0;
    emit_blocks(S, B, n, F->ipt, s_del);
    // the k-th hole below the new count receives the k-th surviving bubble
    // counted from the back: as many as survive
    int h = 0;
    const int pre = block_excl_scan(stays, h);
    if (stays) {
        s_src[pre] = top;
        S.plan_src[pre] = top;
        S.moved_to[top - nnew] = s_del[pre];
    }
    __syncthreads();
    // mark the lists that change, as in plan_many: the first 16 entries of a
    // list together with its length
    int gone = 0, both = 0;
    const int items = nd + h;
    for (int k = t >> 4; k < items; k += kBlock / 16) {
        const int s = k < nd ? s_del[k] : s_src[k - nd];
        const int q0 = t & 15;
        int j = S.nbr[(size_t)min(q0, nbr_cap - 1) * cap + s];
        const int m = S.nn[s];
        for (int q = q0; q < m; q += 16) {
            if (q != q0) j = S.nbr[(size_t)q * cap + s];
            if (j < nnew) S.dirty[j] = 1;  // same value from every writer
            if (k < nd) {
                gone += 1;
                both += S.del[j] ? 1 : 0;
            }
        }
    }
    gone = wave_sum_i(gone);
    both = wave_sum_i(both);
    if (0 == lane) {
        s_sum[0][wave] = gone;
        s_sum[1][wave] = both;
    }
    __syncthreads();
    if (0 == t) {
        gone = both = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            gone += s_sum[0][w];
            both += s_sum[1][w];
        }
        commit_removal(F, s_v, h, nnew, gone - both / 2);
    }
}

__device__ __forceinline__ void plan_removal(Foam *F, const DeletedBlocks &B, int n, int nd) {
    if (nd <= kBlock) plan_few(F, B, n, nd);
    else plan_many(F, B, n, nd);
}

}  // namespace cubble_amd
