// Host-side check of PinnedPair (pp_stage.h) over stand-ins of the runtime calls it
// makes: every byte arrives for sizes of one and several pieces, a pair that grows
// keeps two halves, and copies without pinned memory go through the runtime.
// Built by tests/test_stage_host.py.
//   usage: stage_check      prints: copies checked, of them without pinned memory
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

namespace fake {
size_t limit = 0, held = 0;
std::vector<std::pair<void*, size_t>> live;
hipError_t host_malloc(void** p, size_t n, unsigned) {
    if (held + n > limit) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    std::memset(*p, 0xEE, n);
    held += n;
    live.push_back({*p, n});
    return hipSuccess;
}
hipError_t host_free(void* p) {
    for (auto& e : live)
        if (e.first == p) {
            held -= e.second;
            e = live.back();
            live.pop_back();
            std::free(p);
            return hipSuccess;
        }
    return hipErrorInvalidValue;
}
hipError_t copy(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
int events = 0;
hipError_t event_create(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>((intptr_t)++events);
    return hipSuccess;
}
hipError_t event_ok(hipEvent_t e) { return e ? hipSuccess : hipErrorInvalidHandle; }
hipError_t event_record(hipEvent_t e, hipStream_t) { return event_ok(e); }
hipError_t stream_sync(hipStream_t) { return hipSuccess; }
hipError_t last_error() { return hipSuccess; }
}  // namespace fake
#undef hipHostMalloc
#define hipHostMalloc(p, n, f) fake::host_malloc(p, n, f)
#define hipHostFree(p) fake::host_free(p)
#define hipMemcpyAsync(d, s, n, k, st) fake::copy(d, s, n, k, st)
#define hipEventCreateWithFlags(e, f) fake::event_create(e, f)
#define hipEventRecord(e, st) fake::event_record(e, st)
#define hipEventSynchronize(e) fake::event_ok(e)
#define hipEventDestroy(e) fake::event_ok(e)
#define hipStreamSynchronize(st) fake::stream_sync(st)
#define hipGetLastError() fake::last_error()

#include "../../photonpropagation.jl_amd/csrc/pp_stage.h"

int main() {
    const size_t most = pp::PinnedPair::kMost;
    const size_t sizes[] = {0, 1, 65535, 65536, 65537, most, most - 1, most + 1, 2 * most, 2 * most + 7,
                            3 * most + 1, 100, 5 * most};
    long checked = 0, without = 0;
    for (size_t limit : {(size_t)0, (size_t)100000, most, 64 * most}) {
        fake::limit = limit;
        pp::PinnedPair pair;
        for (size_t n : sizes) {
            std::vector<unsigned char> src(n), dst(n + 16, 0x55);
            for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(i * 131 + (i >> 13));
            if (pair.copy_out(nullptr, dst.data(), src.data(), n) != hipSuccess) {
                std::fprintf(stderr, "limit %zu size %zu failed\n", limit, n);
                return 1;
            }
            for (size_t i = 0; i < dst.size(); ++i)
                if (dst[i] != (i < n ? src[i] : 0x55)) {
                    std::fprintf(stderr, "limit %zu size %zu byte %zu\n", limit, n, i);
                    return 1;
                }
            ++checked;
            without += n > 0 && pair.p == nullptr;
        }
        // one half, then two, then one piece again: never fewer than before
        if (limit == 64 * most) {
            pp::PinnedPair grow;
            if (grow.ensure(1000, 1) || grow.halves != 1) return 2;
            if (grow.ensure(500, 2) || grow.halves != 2 || grow.half < 1000) return 2;
            if (grow.ensure(200000, 1) || grow.halves != 2 || grow.half < 200000) return 2;
            std::memset(grow.at(0), 1, grow.half);
            std::memset(grow.at(1), 2, grow.half);
            grow.release();
        }
        pair.release();
        if (fake::held != 0 || !fake::live.empty()) return 3;
    }
    std::printf("%ld %ld\n", checked, without);
    return 0;
}
