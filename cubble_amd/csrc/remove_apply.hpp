// remove_apply.hpp -- a planned removal, carried out on one block of slots.
#pragma once

#include "dev_util.hpp"

namespace cubble_amd {

// The state of the tail survivor `src` into the hole i, by one wave: lane f
// moves field f (x, v, v_old, saved by component, path, error, wrap counters,
// index, list length at the last search), so all fields' loads are in flight
// together; one after another, each waiting for the store before it, they
// took most of a removal's time.  The radius takes the volume fix on the way.
__device__ __forceinline__ void move_state(const Foam *F, int i, int src, double vm) {
    const int lane = (int)(threadIdx.x & 63), q = lane & 3, D = F->c.dim;
    const bool fvel = CUBBLE_PREC_MIXED == F->precision;
    const Roles *R = &F->r;
    void *p = nullptr;
    bool wide = !fvel;  // an FP64 field
    if (lane < 16) {
        if (q != 2 || 3 == D)
            p = lane < 4 ? R->x[q] : lane < 8 ? R->v[q] : lane < 12 ? R->vo[q] : R->saved[q];
        wide = wide || lane < 4;
    } else if (16 == lane) {
        p = R->path;
        wide = true;
    } else if (17 == lane) {
        p = R->err;
    } else {
        wide = false;
        if (lane < 18 + D) p = R->wc[lane - 18];
        if (21 == lane) p = R->idx;
        if (22 == lane) p = F->s.deg;  // the reference moves numNeighbors unchanged
    }
    if (!p) return;
    if (wide) {
        double v = static_cast<const double *>(p)[src];
        if (3 == lane) v = v * vm;
        static_cast<double *>(p)[i] = v;
    } else {
        static_cast<uint32_t *>(p)[i] = static_cast<const uint32_t *>(p)[src];
    }
}

// Bubble i's list from src's, by one wave: deleted neighbours dropped, moved
// ones mapped to their new slots, ascending.  Up to 64 entries one lane each
// (their marks and new slots are then one load each, and an entry's place is
// the number of smaller ones); longer lists 64 entries at a time.
__device__ __forceinline__ void filter_list(const Scratch &S, size_t cap, int nnew, int i,
                                            int src) {
    const int lane = (int)(threadIdx.x & 63);
    const int m = uniform_i(S.nn[src]);
    if (m <= 64) {
        const int j = lane < m ? S.nbr[(size_t)lane * cap + src] : -1;
        const bool keep = j >= 0 && !S.del[j];
        const bool moved = keep && j >= nnew;
        const int jj = moved ? S.moved_to[j - nnew] : j;
        const unsigned long long kept = __builtin_amdgcn_ballot_w64(keep);
        int pos = __popcll(kept & ((1ull << lane) - 1ull));
        if (__builtin_amdgcn_ballot_w64(moved)) {
            pos = 0;
            for (unsigned long long t = kept; t; t &= t - 1ull)
                pos += __builtin_amdgcn_readlane(jj, __builtin_ctzll(t)) < jj ? 1 : 0;
        }
        if (keep) S.nbr[(size_t)pos * cap + i] = jj;
        if (0 == lane) S.nn[i] = __popcll(kept);
        return;
    }
    // Entries below the new count keep their order; writes stay at positions <=
    // those read, so this also runs in place (src == i).
    constexpr int kNone = 0x7fffffff;
    const unsigned long long below = (1ull << lane) - 1ull;
    auto at = [&](int q, int of) -> int & { return S.nbr[(size_t)q * cap + of]; };
    int out = 0, first = m;  // the moved ones, with the largest indices, come last
    for (int q = 0; q < m; q += 64) {
        const int j = q + lane < m ? at(q + lane, src) : kNone;
        const bool keep = j < nnew && !S.del[j];
        const unsigned long long kept = __builtin_amdgcn_ballot_w64(keep);
        if (keep) at(out + __popcll(kept & below), i) = j;
        out += __popcll(kept);
        const unsigned long long low = __builtin_amdgcn_ballot_w64(j < nnew);
        if (~low) {
            first = q + __popcll(low);
            break;
        }
    }
    // 64 moved ones merged into the list at a time, from its back: an entry goes
    // up by as many as are smaller than it
    for (int q = first; q < m; q += 64) {
        const int j = q + lane < m ? at(q + lane, src) : -1;
        const bool keep = j >= 0 && !S.del[j];
        const int e = keep ? S.moved_to[j - nnew] : kNone;
        const unsigned long long kept = __builtin_amdgcn_ballot_w64(keep);
        if (!kept) continue;
        int pos = 0;  // of e: the smaller moved ones and list entries
        for (unsigned long long t = kept; t; t &= t - 1ull)
            pos += __builtin_amdgcn_readlane(e, __builtin_ctzll(t)) < e ? 1 : 0;
        for (int top = out; top > 0; top -= 64) {
            const int k = top - 64 + lane;
            wave_sync();  // entries that other lanes wrote
            const int v = k >= 0 ? at(k, i) : kNone;
            int up = 0;
            for (unsigned long long t = kept; t; t &= t - 1ull) {
                const int l = __builtin_ctzll(t), n = __builtin_amdgcn_readlane(e, l);
                const int smaller = __popcll(__builtin_amdgcn_ballot_w64(v < n));
                up += k >= 0 && n < v ? 1 : 0;
                if (lane == l) pos += smaller;
            }
            wave_sync();
            if (up > 0) at(k + up, i) = v;
            // the rest is smaller than all of them once its last one is
            if (0 == __builtin_amdgcn_readlane(up, max(64 - top, 0))) {
                pos += max(top - 64, 0);
                break;
            }
        }
        wave_sync();
        if (keep) at(pos, i) = e;
        out += __popcll(kept);
    }
    if (0 == lane) S.nn[i] = out;
}

// Bubble i's own list of at most 16 entries, filtered by 16 lanes (g: which of
// the wave's four groups).  j: this lane's entry, -1 past the end.
__device__ __forceinline__ void filter_short(const Scratch &S, size_t cap, int nnew, int i, int j,
                                             int g) {
    const int lane = (int)(threadIdx.x & 15);
    const bool keep = j >= 0 && !S.del[j];
    const bool moved = keep && j >= nnew;
    const int jj = moved ? S.moved_to[j - nnew] : j;
    const unsigned kept = (unsigned)(__builtin_amdgcn_ballot_w64(keep) >> (16 * g)) & 0xffffu;
    int pos = __popc(kept & ((1u << lane) - 1u));
    if (__builtin_amdgcn_ballot_w64(moved)) {
        pos = 0;
        for (int k = 0; k < 16; ++k) {
            const int v = __shfl(jj, 16 * g + k);
            pos += (kept >> k & 1u) && v < jj ? 1 : 0;
        }
    }
    if (keep) S.nbr[(size_t)pos * cap + i] = jj;
    if (0 == lane && i >= 0) S.nn[i] = __popc(kept);
}

// The planned removal on the slots of bubble-space block lb, by its whole
// workgroup: each thread applies the volume fix to its bubbles; the few holes
// and marked bubbles are listed in LDS and rebuilt, a marked bubble with a short
// list by 16 lanes, the others by one wave each.  No block reads a slot that
// another one writes: the survivors lie past the new count.  What bounds it is
// the rebuild's chain of dependent loads (list, marks, new slots) behind one
// pass over marks and radii; the ten or so neighbours of a deleted bubble are
// in few blocks, so that rebuilt by a wave each they took three such chains.
__device__ __forceinline__ void apply_removal(const Foam *F, int lb) {
    // marked bubbles from the front of the list, holes from its back
    __shared__ int s_cnt, s_holes, s_list[kBlock];
    const Scratch S = F->s;
    double *const r = F->r.x[3];
    const int nnew = F->d.count, h = F->d.n_holes, ipt = F->ipt;
    const double vm = F->d.vol_fix;
    const size_t cap = (size_t)F->cap;
    const int nbr_cap = F->nbr_cap;
    const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6);
    for (int k = 0; k < ipt; ++k) {
        const int base = (lb * ipt + k) * kBlock;
        if (base >= nnew) break;  // uniform per block
        const int i = base + (int)threadIdx.x;
        if (0 == threadIdx.x) s_cnt = s_holes = 0;
        __syncthreads();
        if (i < nnew) {
            const bool hole = S.del[i] != 0;
            const bool marked = S.dirty[i] != 0;
            if (!hole) r[i] = r[i] * vm;
            if (marked) S.dirty[i] = 0;
            if (hole) s_list[kBlock - 1 - atomicAdd(&s_holes, 1)] = i;
            else if (marked) s_list[atomicAdd(&s_cnt, 1)] = i;
        }
        __syncthreads();
        const int cnt = s_cnt, holes = s_holes;
        // the last waves first: the marked bubbles go to the first
        for (int e = kWaves - 1 - wave; e < holes; e += kWaves) {
            const int b = uniform_i(s_list[kBlock - 1 - e]);
            int src = b;  // the k-th entry of the deletion list is the k-th hole
            int k0 = 0;
            for (int len = h; len > 256;) {  // (ascending: 64 steps at once)
                const int step = (len + 63) >> 6;
                const int at = k0 + lane * step;
                const bool reached = lane * step < len && S.del_list[at] <= b;
                const int c = __popcll(__builtin_amdgcn_ballot_w64(reached)) - 1;
                len = min(step, len - c * step);
                k0 += c * step;
            }
            for (; k0 < h; k0 += 64) {
                const bool in = k0 + lane < h;
                const int d = in ? S.del_list[k0 + lane] : -1;
                const int s = in ? S.plan_src[k0 + lane] : -1;
                const unsigned long long at = __builtin_amdgcn_ballot_w64(d == b);
                if (at) {
                    src = __builtin_amdgcn_readlane(s, __builtin_ctzll(at));
                    break;
                }
            }
            move_state(F, b, src, vm);
            filter_list(S, cap, nnew, b, src);
        }
        // (a wave's four groups together: the ballots need them)
        for (int e0 = 4 * wave; e0 < cnt; e0 += kBlock / 16) {
            const int e = e0 + (lane >> 4), q = lane & 15;
            const int b = e < cnt ? s_list[e] : -1;
            int j = -1, m = 0;
            if (b >= 0) {
                j = S.nbr[(size_t)min(q, nbr_cap - 1) * cap + b];
                m = S.nn[b];
            }
            const bool brief = m <= 16;
            filter_short(S, cap, nnew, brief ? b : -1, brief && q < m ? j : -1, lane >> 4);
            for (unsigned long long t = __builtin_amdgcn_ballot_w64(!brief && 0 == q); t;
                 t &= t - 1ull) {
                const int v = __builtin_amdgcn_readlane(b, __builtin_ctzll(t));
                filter_list(S, cap, nnew, v, v);
            }
        }
        __syncthreads();
    }
}

}  // namespace cubble_amd
