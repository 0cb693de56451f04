// readback.hpp -- device arrays of one engine copied to caller-owned host
// arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

namespace cubble_amd {

class Engine;

// Where the lists of n bubbles end when stored one after another: ends[i] =
// nn[0] + .. + nn[i], its low 32 bits; base[t], in full, where the lists of
// bubbles 1024 t on begin; the total, base's last.
struct ListEnds {
    uint32_t *ends = nullptr;
    int64_t *base = nullptr, *total = nullptr;
};

class Readback {
  public:
    // n elements of 8 bytes, 4 bytes or 1 byte; FP32 elements as FP64.  A null
    // dst is skipped.
    void f64(double *dst, const void *src, size_t n) { add(dst, src, n, kWords8, 8); }
    void i64(int64_t *dst, const void *src, size_t n) { add(dst, src, n, kWords8, 8); }
    void i32(int32_t *dst, const void *src, size_t n) { add(dst, src, n, kWords4, 4); }
    void u8(uint8_t *dst, const void *src, size_t n) { add(dst, src, n, kWords1, 1); }
    void f32_as_f64(double *dst, const void *src, size_t n) { add(dst, src, n, kWiden, 4); }
    // The entries of n bubbles' neighbour lists one after another, `total` in
    // all: entry q of bubble i's is nbr[q * cap + i].
    void lists(int32_t *dst, const ListEnds &ends, const int32_t *nbr, size_t cap, int n,
               size_t total);
    // Copies them all; the arrays are complete when it returns.
    int run(Engine &e);

    enum Kind { kWords1, kWords4, kWords8, kWiden, kLists };

  private:
    struct Item {
        char *dst;
        const void *src;
        size_t n;
        int kind, size;
    };
    void add(void *dst, const void *src, size_t n, int kind, int size) {
        if (dst && n) items_.push_back(Item{static_cast<char *>(dst), src, n, kind, size});
    }
    std::vector<Item> items_;
    ListEnds ends_;
    const int32_t *nbr_ = nullptr;
    size_t cap_ = 0;
    int bubbles_ = 0;
};

// The ends of n > 0 lists, into ends (n ints); scratch (8-byte aligned): 12 bytes
// per 1024 lists and 20 more.
ListEnds launch_list_ends(const int32_t *nn, int n, int32_t *ends, int32_t *scratch,
                          hipStream_t stream);

// The pinned blocks that Readback::run copies through are shared by the
// process's engines and freed with the last of them.
void bounce_engine_opened();
void bounce_engine_closed();

}  // namespace cubble_amd
