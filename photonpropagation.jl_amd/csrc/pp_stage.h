// pp_stage.h - results on their way from the device to pageable host memory,
// through two pinned halves that their owner keeps. The runtime's own copy from
// device to pageable memory took 408 us for 1 MB and 1450 us for 20 MB (to fresh
// pages); through the pinned halves, one being filled by the device while the
// other is emptied by the host, 40 us and 700 us. Measured on MI355X.
// Kernels may write the halves themselves: the memory is coherent, so that their
// stores are visible once an event or stream behind them is done.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>

namespace pp {

struct PinnedPair {
    char* p = nullptr;
    size_t half = 0;    // bytes of each half
    int halves = 0;     // one where all the work is a single piece, two, or a third for
                        // work that runs two pieces ahead
    hipEvent_t ev[3] = {};

    static constexpr size_t kMost = (size_t)4 << 20;  // half of copy_out's own choice

    // At least `bytes` per half. Work that still uses the old halves must be done.
    hipError_t ensure(size_t bytes, int n = 2) {
        for (auto& e : ev)
            if (!e)
                if (hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming)) return r;
        if (bytes <= half && n <= halves) return hipSuccess;
        bytes = std::max(bytes, half);
        n = std::max(n, halves);
        // in eighths of a power of two: pinning takes its time by the page
        size_t want = (size_t)64 << 10;
        while (want < bytes) want *= 2;
        const size_t step = want / 8;
        want = std::max((size_t)64 << 10, (bytes + step - 1) / step * step);
        if (p) (void)hipHostFree(p);
        p = nullptr;
        half = 0;
        halves = 0;
        if (hipError_t r = hipHostMalloc((void**)&p, n * want, hipHostMallocCoherent)) return r;
        half = want;
        halves = n;
        return hipSuccess;
    }
    char* at(int k) const { return p + (size_t)k * half; }
    void release() {
        if (p) (void)hipHostFree(p);
        for (auto& e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        p = nullptr;
        half = 0;
        halves = 0;
    }

    // dst (host) <- src (device), ordered on the stream; returns when dst is written.
    // Where no pinned memory is left, the runtime's own copy.
    hipError_t copy_out(hipStream_t st, void* dst, const void* src, size_t bytes) {
        if (bytes == 0) return hipStreamSynchronize(st);
        if (ensure(std::min(bytes, kMost), bytes > kMost ? 2 : 1) != hipSuccess) {
            (void)hipGetLastError();
            if (hipError_t r = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st)) return r;
            return hipStreamSynchronize(st);
        }
        const size_t n = (bytes + half - 1) / half;
        auto part = [&](size_t k) { return std::min(half, bytes - k * half); };
        for (size_t k = 0; k <= n; ++k) {
            if (k < n) {
                if (hipError_t r = hipMemcpyAsync(at((int)(k & 1)), (const char*)src + k * half, part(k),
                                                  hipMemcpyDeviceToHost, st))
                    return r;
                if (hipError_t r = hipEventRecord(ev[k & 1], st)) return r;
            }
            if (k > 0) {
                if (hipError_t r = hipEventSynchronize(ev[(k - 1) & 1])) return r;
                std::memcpy((char*)dst + (k - 1) * half, at((int)((k - 1) & 1)), part(k - 1));
            }
        }
        return hipSuccess;
    }
};

}  // namespace pp
