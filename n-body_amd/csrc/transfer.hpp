// Host copies of state arrays: several device rows of n floats to or from the
// caller's memory.
//
// A blocking copy of pageable memory costs some 18 us each way however small
// it is, and a system's state is six to nine of them.  Here one kernel packs
// the rows into pinned memory (or unpacks them from it), one wait, and the
// host moves them to or from the caller's arrays: out, a member of 512 bodies
// with its accelerations 164 -> 27 us.  Large states go through eight slots in
// turn, packed while four threads copy and touch the caller's fresh pages:
// 1,048,576 bodies' state 2.3 -> 1.7 ms, their accelerations 1.6 -> 0.4.
#pragma once

#include <atomic>
#include <cstdint>
#include <mutex>

#include "host_util.hpp"
#include "launch.hpp"

namespace nbg {

constexpr int kSlotCount = 8;
constexpr int64_t kSlotWords = 1 << 18;  // 1 MiB
constexpr int kCopyThreads = 4;
constexpr int64_t kThreadedWords = 1 << 21;  // 8 MiB: below, starting threads costs more than they save

// A context's pinned slots: allocated with the first transfer, freed with the
// context, used by one transfer at a time.
struct Staging {
    std::mutex mu;
    bool tried = false;
    float *words = nullptr;   // kSlotCount slots, then one line for an error word
    hipEvent_t ev[kSlotCount] = {};
    bool ready();             // with mu held
    void release();
    float *slot(int i) const { return words + i * kSlotWords; }
    volatile uint32_t *err() const { return reinterpret_cast<volatile uint32_t *>(words + kSlotCount * kSlotWords); }
};

// Copies rows R (n floats each) into dst[0 .. R.k - 1]; with R.xyz the last
// three rows go interleaved to dst[R.k - 3].  err (device, may be null) is read
// first: if it holds a value, that goes to *err_value and nothing is copied.
// The stream must have no unfinished work that another thread could wait for.
int rows_out(nbg_ctx *ctx, hipStream_t s, const RowSet &R, float *const *dst, int64_t n, const uint32_t *err = nullptr,
             uint32_t *err_value = nullptr);

// Copies src[j] (null: zeros) into row j.
int rows_in(nbg_ctx *ctx, hipStream_t s, const RowSet &R, const float *const *src, int64_t n);

}  // namespace nbg
