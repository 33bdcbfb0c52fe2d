#include "transfer.hpp"

#include <cstring>
#include <thread>

namespace nbg {

bool Staging::ready() {
    if (tried) return words != nullptr;
    tried = true;
    if (hipHostMalloc((void **)&words, (kSlotCount * kSlotWords + 64) * sizeof(float), hipHostMallocDefault) !=
        hipSuccess) {
        words = nullptr;
        (void)hipGetLastError();
        return false;
    }
    for (auto &e : ev)
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            release();
            return false;
        }
    return true;
}

void Staging::release() {
    for (auto &e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (words) (void)hipHostFree(words);
    words = nullptr;
}

namespace {

// Without pinned memory: one blocking copy a row.
int plain_out(const RowSet &R, float *const *dst, int64_t n) {
    const int whole = R.xyz ? R.k - 3 : R.k;
    for (int j = 0; j < whole; ++j) NBG_HIP(hipMemcpy(dst[j], R.row[j], (size_t)n * 4, hipMemcpyDeviceToHost));
    if (!R.xyz) return NBG_OK;
    float v[4096];
    for (int64_t i0 = 0; i0 < n; i0 += 4096) {
        const int64_t cnt = n - i0 < 4096 ? n - i0 : 4096;
        for (int c = 0; c < 3; ++c) {
            NBG_HIP(hipMemcpy(v, R.row[whole + c] + i0, (size_t)cnt * 4, hipMemcpyDeviceToHost));
            for (int64_t i = 0; i < cnt; ++i) dst[whole][3 * (i0 + i) + c] = v[i];
        }
    }
    return NBG_OK;
}

int read_err(const uint32_t *err, uint32_t *value) {
    *value = 0;
    if (err) NBG_HIP(hipMemcpy(value, err, 4, hipMemcpyDeviceToHost));
    return NBG_OK;
}

}  // namespace

int rows_out(nbg_ctx *ctx, hipStream_t s, const RowSet &R, float *const *dst, int64_t n, const uint32_t *err,
             uint32_t *err_value) {
    uint32_t none = 0;
    if (!err_value) err_value = &none;
    *err_value = 0;
    if (n <= 0 || R.k <= 0) return read_err(err, err_value);
    Staging &S = *ctx->staging;
    std::lock_guard<std::mutex> lk(S.mu);
    if (!S.ready()) {
        if (int r = read_err(err, err_value)) return r;
        return *err_value ? NBG_OK : plain_out(R, dst, n);
    }
    const int64_t most = (kSlotWords / R.k) & ~(int64_t)3;
    const int64_t chunks = (n + most - 1) / most;
    const int whole = R.xyz ? R.k - 3 : R.k;
    auto count = [&](int64_t c) { return c + 1 < chunks ? most : n - c * most; };
    auto stride = [&](int64_t c) { return (count(c) + 3) & ~(int64_t)3; };
    auto pack = [&](int64_t c) -> hipError_t {
        launch_rows_out(R, c * most, (int)count(c), (int)stride(c), S.slot((int)(c % kSlotCount)), c == 0 ? err : nullptr,
                        (uint32_t *)S.err(), s);
        const hipError_t e = hipGetLastError();
        return e != hipSuccess ? e : hipEventRecord(S.ev[c % kSlotCount], s);
    };
    auto unload = [&](int64_t c) {
        const float *p = S.slot((int)(c % kSlotCount));
        const int64_t i0 = c * most, cnt = count(c), st = stride(c);
        for (int j = 0; j < whole; ++j) std::memcpy(dst[j] + i0, p + j * st, (size_t)cnt * 4);
        if (R.xyz) std::memcpy(dst[whole] + 3 * i0, p + whole * st, (size_t)cnt * 12);
    };
    // Every launched pack is waited for before the slots are given back.
    hipError_t bad = hipSuccess;
    for (int64_t c = 0; c < chunks && c < kSlotCount && bad == hipSuccess; ++c) bad = pack(c);
    if (bad == hipSuccess) bad = hipEventSynchronize(S.ev[0]);
    if (bad != hipSuccess) {
        (void)hipStreamSynchronize(s);
        return fail(NBG_ERR_HIP, std::string("state copy: ") + hipGetErrorString(bad));
    }
    if (err && *S.err()) {
        *err_value = *S.err();
        NBG_HIP(hipStreamSynchronize(s));
        return NBG_OK;
    }
    std::atomic<int> failed{(int)hipSuccess};
    // Chunks t, t + T, ...: a slot's next chunk is packed as soon as the slot is empty.
    auto run = [&](int t, int T) {
        for (int64_t c = t; c < chunks; c += T) {
            hipError_t e = hipEventSynchronize(S.ev[c % kSlotCount]);
            if (e == hipSuccess) {
                unload(c);
                if (c + kSlotCount < chunks) e = pack(c + kSlotCount);
            }
            if (e != hipSuccess) {
                failed = (int)e;
                return;
            }
        }
    };
    const bool threaded = n * R.k >= kThreadedWords && chunks >= kCopyThreads;
    if (!threaded) {
        run(0, 1);
    } else {
        static_assert(kSlotCount % kCopyThreads == 0, "a slot's chunks are one thread's");
        std::thread helpers[kCopyThreads];
        int started = 1;
        try {
            for (; started < kCopyThreads; ++started)
                helpers[started] = std::thread([&run, &failed, ctx, t = started] {
                    if (hipSetDevice(ctx->device) != hipSuccess) failed = (int)hipErrorInvalidDevice;
                    else run(t, kCopyThreads);
                });
        } catch (...) {
            // no thread to be had: its chunks are done here
        }
        run(0, kCopyThreads);
        for (int t = started; t < kCopyThreads; ++t) run(t, kCopyThreads);
        for (int t = 1; t < started; ++t) helpers[t].join();
    }
    if (failed != (int)hipSuccess) {
        (void)hipStreamSynchronize(s);
        return fail(NBG_ERR_HIP, std::string("state copy: ") + hipGetErrorString((hipError_t)failed.load()));
    }
    return NBG_OK;
}

int rows_in(nbg_ctx *ctx, hipStream_t s, const RowSet &R, const float *const *src, int64_t n) {
    if (n <= 0) return NBG_OK;
    const int64_t stride = (n + 3) & ~(int64_t)3;
    if (R.k * stride <= kSlotWords) {
        Staging &S = *ctx->staging;
        std::lock_guard<std::mutex> lk(S.mu);
        if (S.ready()) {
            uint32_t absent = 0;
            for (int j = 0; j < R.k; ++j) {
                if (src[j]) std::memcpy(S.slot(0) + j * stride, src[j], (size_t)n * 4);
                else absent |= 1u << j;
            }
            launch_rows_in(R, (int)n, (int)stride, S.slot(0), absent, s);
            const hipError_t e = hipGetLastError();
            const hipError_t w = hipStreamSynchronize(s);
            if (e != hipSuccess || w != hipSuccess)
                return fail(NBG_ERR_HIP, std::string("state copy: ") + hipGetErrorString(e != hipSuccess ? e : w));
            return NBG_OK;
        }
    }
    for (int j = 0; j < R.k; ++j) {
        if (src[j]) NBG_HIP(hipMemcpyAsync(R.row[j], src[j], (size_t)n * 4, hipMemcpyHostToDevice, s));
        else launch_fill_u32((uint32_t *)R.row[j], 0u, n, s);
    }
    NBG_HIP(hipStreamSynchronize(s));
    return NBG_OK;
}

}  // namespace nbg

