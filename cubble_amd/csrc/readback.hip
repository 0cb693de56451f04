// readback.hip -- device arrays to caller-owned host arrays.
//
// A copy per field costs a host call and a wait each (10-15 us), and the
// runtime moves pageable memory at 14 GB/s.  Here one kernel writes a chunk of
// all fields into pinned host memory, in the caller's order, at the
// rate of the link (51 GB/s), and the host copies the chunks before it into
// the caller's arrays meanwhile.  One thread reads what the device just wrote
// at 25 GB/s, so larger reads take helpers.  Attempt outputs of 2e5 bubbles
// (3D FP64, 16 MB) 1180 -> 460 us, of 4e3 150 -> 56; a state of 3e4 (2D, 5 MB)
// 900 -> 300, of 1e6 (3D) 70 -> 17 ms, most of it first touches of new arrays.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>

#include "dev_util.hpp"
#include "engine.hpp"
#include "readback.hpp"

namespace cubble_amd {

namespace {

// One kernel's piece of an item: elements [first, first + n) to byte `dst` of
// the chunk, by the workgroups from tile0 on.
struct PackSeg {
    const void *src;
    uint64_t first;
    uint32_t n, dst, tile0;
    int32_t kind;
};

constexpr int kPackSegs = 32;
constexpr unsigned kPackTile = 4 * kBlock;  // elements per workgroup
// The pinned block: room for the chunk that the host copies and the two whose
// kernels are in flight meanwhile, the one behind it and the one after.
constexpr int kSlots = 3;
constexpr size_t kRoom = (size_t)1 << 20;
// Reads above it go in chunks of kRoom and copy with three threads more
// (starting them takes 30 us); smaller ones in half of it at most, so that their
// copies start early.
constexpr size_t kHelpFrom = (size_t)4 << 20;
constexpr int kHelpers = 3;
constexpr size_t kPiece = (size_t)64 << 10;  // bytes a thread copies at a time

struct PackArgs {
    PackSeg seg[kPackSegs];
    int32_t nseg;
    int32_t bubbles;
    const uint32_t *ends;
    const int64_t *base;
    const int32_t *nbr;
    uint64_t cap;
};

constexpr int kEndsTile = 4 * kBlock;  // bubbles per workgroup of k_ends

__global__ __launch_bounds__(kBlock) void k_pack(PackArgs a, char *out) {
    int s = 0;
    while (s + 1 < a.nseg && blockIdx.x >= a.seg[s + 1].tile0) ++s;  // uniform
    const PackSeg g = a.seg[s];
    const unsigned e0 = (blockIdx.x - g.tile0) * kPackTile + threadIdx.x;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const unsigned e = e0 + u * kBlock;
        if (e >= g.n) break;
        const uint64_t k = g.first + e;
        if (Readback::kWords8 == g.kind) {
            reinterpret_cast<uint64_t *>(out + g.dst)[e] =
                static_cast<const uint64_t *>(g.src)[k];
        } else if (Readback::kLists == g.kind) {
            // the tile, and in it the bubble, whose lists hold entry k: the first
            // that ends past it
            int t = 0, hi = (a.bubbles - 1) / kEndsTile;
            while (t < hi) {
                const int mid = (t + hi) >> 1;
                if ((uint64_t)a.base[mid + 1] > k) hi = mid;
                else t = mid + 1;
            }
            const uint32_t first = (uint32_t)a.base[t], rel = (uint32_t)k - first;
            int lo = t * kEndsTile;
            hi = min(a.bubbles, lo + kEndsTile) - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (a.ends[mid] - first > rel) hi = mid;
                else lo = mid + 1;
            }
            const uint32_t q = rel - (lo > t * kEndsTile ? a.ends[lo - 1] - first : 0u);
            reinterpret_cast<int32_t *>(out + g.dst)[e] = a.nbr[q * a.cap + lo];
        } else {  // FP32 as it is; bytes in words of four
            reinterpret_cast<uint32_t *>(out + g.dst)[e] =
                static_cast<const uint32_t *>(g.src)[k];
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_ends_part(const int32_t *nn, int n, int32_t *part) {
    int s = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = blockIdx.x * kEndsTile + u * kBlock + (int)threadIdx.x;
        if (i < n) s += nn[i];
    }
    s = block_sum_i(s);
    if (0 == threadIdx.x) part[blockIdx.x] = s;
}

// (A foam's lists may hold more than 2^31 entries, those of 1024 bubbles not.)
__global__ __launch_bounds__(kBlock) void k_ends(const int32_t *nn, int n, const int32_t *part,
                                                 uint32_t *ends, int64_t *base) {
    double acc = 0.0;  // whole numbers: exact
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += kBlock) acc += (double)part[b];
    int64_t off = (int64_t)block_sum(acc);
    if (0 == threadIdx.x) base[blockIdx.x] = off;
    for (int u = 0; u < 4; ++u) {
        const int i = blockIdx.x * kEndsTile + u * kBlock + (int)threadIdx.x;
        const int v = i < n ? nn[i] : 0;
        int tot = 0;
        const int pre = block_excl_scan(v, tot);
        if (i < n) ends[i] = (uint32_t)(off + pre + v);
        off += tot;
    }
    if (0 == threadIdx.x && blockIdx.x + 1 == gridDim.x) base[gridDim.x] = off;
}

// Pinned memory in slots and the events of the kernels that fill them.
struct Bounce {
    char *mem = nullptr;
    hipEvent_t done[kSlots] = {};
    int device = 0;
};

std::mutex g_lock;
constexpr int kIdle = 2;
Bounce g_idle[kIdle];  // emptied with the last engine
int g_num_idle = 0;
int g_engines = 0;

void destroy(Bounce &b) {
    for (hipEvent_t &d : b.done)
        if (d) (void)hipEventDestroy(d);
    if (b.mem) (void)hipHostFree(b.mem);
    b = Bounce{};
}

// A block for the duration of one call (one per thread that reads).
class Lease {
  public:
    Bounce b;
    hipError_t take(int device) {
        {
            std::lock_guard<std::mutex> l(g_lock);
            for (int k = 0; k < g_num_idle; ++k)
                if (g_idle[k].device == device) {
                    b = g_idle[k];
                    g_idle[k] = g_idle[--g_num_idle];
                    return hipSuccess;
                }
        }
        b.device = device;
        // an event belongs to the device that is current, which need not be the
        // engine's in the calling thread
        int was = device;
        hipError_t e = hipGetDevice(&was);
        if (hipSuccess == e && was != device) e = hipSetDevice(device);
        if (hipSuccess == e) e = hipHostMalloc((void **)&b.mem, kSlots * kRoom, hipHostMallocDefault);
        for (hipEvent_t &d : b.done)
            if (hipSuccess == e) e = hipEventCreateWithFlags(&d, hipEventDisableTiming);
        if (was != device) (void)hipSetDevice(was);
        return e;
    }
    // complete: nothing on the device uses the block any more
    bool complete = true;
    ~Lease() {
        if (complete && b.done[kSlots - 1]) {
            std::lock_guard<std::mutex> l(g_lock);
            if (g_engines > 0 && g_num_idle < kIdle) {
                g_idle[g_num_idle++] = b;
                return;
            }
        }
        if (!complete) (void)hipDeviceSynchronize();
        destroy(b);
    }
};

struct Copy {
    char *dst;
    const char *src;
    size_t bytes;  // at src
    bool widen;    // FP32 there, FP64 at dst
    void run() const {
        if (!widen) {
            std::memcpy(dst, src, bytes);
            return;
        }
        const float *const s = reinterpret_cast<const float *>(src);
        double *const d = reinterpret_cast<double *>(dst);
        for (size_t k = 0; k < bytes / 4; ++k) d[k] = (double)s[k];
    }
};

// Copies lists of pieces with the threads it started, all of which end with
// the object.  run() returns when the list is copied.
class Copier {
  public:
    explicit Copier(int helpers) {
        for (int k = 0; k < helpers; ++k) {
            try {
                threads_.emplace_back([this] { help(); });
            } catch (...) {  // no thread to be had: the caller copies
                break;
            }
        }
    }
    ~Copier() {
        stop_.store(true, std::memory_order_release);
        for (std::thread &t : threads_) t.join();
    }
    void run(const std::vector<Copy> &list) {
        if (threads_.empty()) {
            for (const Copy &c : list) c.run();
            return;
        }
        list_ = &list;
        left_.store((int)list.size(), std::memory_order_relaxed);
        // takers of the round before are out (left_ was 0), so the round and
        // its first piece can be set together
        next_.store((int)list.size(), std::memory_order_release);
        take();
        while (left_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
    }

  private:
    // pieces from the last one down; next_ <= 0: none
    void take() {
        for (int k; (k = next_.fetch_sub(1, std::memory_order_acq_rel) - 1) >= 0;) {
            (*list_)[(size_t)k].run();
            left_.fetch_sub(1, std::memory_order_acq_rel);
        }
    }
    void help() {
        while (!stop_.load(std::memory_order_acquire)) {
            if (next_.load(std::memory_order_acquire) > 0) take();
            else std::this_thread::yield();
        }
    }
    const std::vector<Copy> *list_ = nullptr;
    std::atomic<int> next_{0}, left_{0};
    std::atomic<bool> stop_{false};
    std::vector<std::thread> threads_;
};

}  // namespace

void bounce_engine_opened() {
    std::lock_guard<std::mutex> l(g_lock);
    ++g_engines;
}

void bounce_engine_closed() {
    std::lock_guard<std::mutex> l(g_lock);
    if (--g_engines > 0) return;
    while (g_num_idle > 0) destroy(g_idle[--g_num_idle]);
}

void Readback::lists(int32_t *dst, const ListEnds &ends, const int32_t *nbr, size_t cap, int n,
                     size_t total) {
    ends_ = ends;
    nbr_ = nbr;
    cap_ = cap;
    bubbles_ = n;
    add(dst, nullptr, total, kLists, 4);
}

int Readback::run(Engine &e) {
    if (items_.empty()) return CUBBLE_OK;
    Lease lease;
    auto bad = [&](hipError_t err, const char *what) {
        return e.fail(err == hipErrorOutOfMemory ? CUBBLE_E_NOMEM : CUBBLE_E_HIP,
                      std::string(what) + ": " + hipGetErrorString(err));
    };
    hipError_t err = lease.take(e.device);
    if (err != hipSuccess) return bad(err, "readback: pinned memory");
    size_t all = 0;
    for (const Item &it : items_) all += it.n * it.size;
    // (a small read in equal parts, so that the copies overlap the kernels)
    const size_t chunk = std::min(all > kHelpFrom ? kRoom : kRoom / 2,
                                  std::max((all / 4 + 255) & ~(size_t)255, (size_t)128 << 10));
    std::vector<Copy> copies[kSlots];
    size_t item = 0, at = 0;  // the next element to fetch
    // the next chunk's kernel, into slot h; false: nothing is left
    auto launch = [&](int h) {
        PackArgs a{};
        a.ends = ends_.ends;
        a.base = ends_.base;
        a.nbr = nbr_;
        a.cap = cap_;
        a.bubbles = bubbles_;
        copies[h].clear();
        char *const out = lease.b.mem + (size_t)h * kRoom;
        size_t off = 0;
        unsigned tiles = 0;
        while (item < items_.size() && a.nseg < kPackSegs) {
            const Item &it = items_[item];
            // bytes in words of four (device arrays are padded to 256 bytes)
            const size_t size = it.size < 4 ? 4 : it.size;
            const size_t n = it.size < 4 ? (it.n * it.size + 3) / 4 : it.n;
            size_t take = std::min(n - at, (chunk - off) / size);
            if (take < n - at) take -= take % kPackTile;
            if (0 == take) break;
            PackSeg &g = a.seg[a.nseg++];
            g.src = it.src;
            g.first = at;
            g.n = (uint32_t)take;
            g.dst = (uint32_t)off;
            g.tile0 = tiles;
            g.kind = it.kind;
            tiles += (unsigned)((take + kPackTile - 1) / kPackTile);
            const size_t bytes = std::min(take * size, it.n * it.size - at * size);
            const bool widen = kWiden == it.kind;
            for (size_t b = 0; b < bytes; b += kPiece)
                copies[h].push_back(Copy{it.dst + (widen ? 2 : 1) * (at * size + b),
                                         out + off + b, std::min(kPiece, bytes - b), widen});
            off = std::min(chunk, (off + take * size + 255) & ~(size_t)255);
            at += take;
            if (at == n) {
                ++item;
                at = 0;
            }
        }
        if (0 == a.nseg) return false;
        hipLaunchKernelGGL(k_pack, dim3(tiles), dim3(kBlock), 0, e.stream, a, out);
        err = hipGetLastError();
        if (hipSuccess == err) err = hipEventRecord(lease.b.done[h], e.stream);
        return true;
    };
    lease.complete = false;
    bool busy[kSlots] = {};
    int ahead = 0;  // the slot to launch into next
    // (two to begin with: the first copy waits for their launches)
    for (; ahead < 2 && hipSuccess == err && (busy[ahead] = launch(ahead)); ++ahead) {}
    Copier copier(all > kHelpFrom ? kHelpers : 0);
    for (int h = 0; hipSuccess == err && busy[h]; h = (h + 1) % kSlots) {
        // the slot copied last takes the chunk after the one in flight
        if (!busy[ahead] && (busy[ahead] = launch(ahead))) ahead = (ahead + 1) % kSlots;
        if (hipSuccess == err) err = hipEventSynchronize(lease.b.done[h]);
        if (err != hipSuccess) break;
        copier.run(copies[h]);
        busy[h] = false;
    }
    if (err != hipSuccess) return bad(err, "readback");
    lease.complete = true;
    return CUBBLE_OK;
}

ListEnds launch_list_ends(const int32_t *nn, int n, int32_t *ends, int32_t *scratch,
                          hipStream_t stream) {
    const int nb = (n + kEndsTile - 1) / kEndsTile;
    ListEnds e;
    e.ends = reinterpret_cast<uint32_t *>(ends);
    e.base = reinterpret_cast<int64_t *>(scratch);
    e.total = e.base + nb;
    int32_t *const part = scratch + 2 * (nb + 1);
    hipLaunchKernelGGL(k_ends_part, dim3(nb), dim3(kBlock), 0, stream, nn, n, part);
    hipLaunchKernelGGL(k_ends, dim3(nb), dim3(kBlock), 0, stream, nn, n, part, e.ends, e.base);
    return e;
}

}  // namespace cubble_amd
