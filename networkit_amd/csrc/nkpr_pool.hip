// Memory and streams kept between handles.
//
// Making and destroying a handle takes about a hundred device allocations, most of them the
// temporaries of the sorts.  hipMalloc and hipFree cost 20 to 150 us each (hipFree waits for the
// device and unmaps), and their cost grows with what the process has allocated before: a handle
// over 1.5e7 arcs with one solve, made and destroyed in a loop, took 30 ms in a fresh process and
// 163 ms in one that had held a 40 GB handle, of which the kernels are 12 ms.  Freed blocks are
// therefore kept for the next request of about their size.
//
//   bounded     at most kKeepBytes per process (NKPR_POOL_MB overrides; 0 keeps nothing), blocks of
//               at most kLargest; larger ones go straight to hipMalloc and hipFree.  A released
//               block that would pass the bound takes the place of those kept longest: blocks
//               left by a large handle otherwise held the room that the next handles need
//               (72 ms instead of 12.5 for the solve above, until they were old enough).
//   given back  all blocks by release_kept (nkpr_release_memory), and when an allocation of this
//               library fails, which is then tried again; a block unused for kKeepSeconds at the
//               next request or release.  There is no timer: a process that stops calling the
//               library keeps what it had until it asks for the release.
//   ordering    hipFree waits for all work on the device before the memory can be used again.  The
//               same holds here: a block is handed out only after a device synchronisation that
//               came after its release (one for all blocks released before it).
//   threads     one lock; blocks belong to the device they were allocated on.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdlib>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "nkpr_internal.hpp"

namespace nkpr {
namespace {

using Clock = std::chrono::steady_clock;

constexpr size_t kKeepBytes = (size_t)4 << 30;
constexpr size_t kLargest = (size_t)1 << 30;
constexpr double kKeepSeconds = 10.0;
constexpr size_t kPinnedBytes = 4096;  // pinned buffers are control blocks and dot results
constexpr size_t kMostPinned = 64, kMostStreams = 16;

struct Kept {
    void *p;
    uint64_t released;  // position in the order of releases
    Clock::time_point at;
};
struct Live {
    int device;
    size_t bytes;
};
struct DevicePool {
    std::multimap<size_t, Kept> kept;
    std::vector<hipStream_t> streams;
    uint64_t synced = 0;  // every block released up to here is idle
};

struct Pool {
    std::mutex mu;
    std::unordered_map<void *, Live> live;  // blocks in use that go back to the pool
    std::map<int, DevicePool> dev;
    std::vector<void *> pinned;
    uint64_t releases = 0;
    size_t kept_bytes = 0, limit = kKeepBytes;

    Pool() {
        if (const char *e = std::getenv("NKPR_POOL_MB"); e && *e) limit = (size_t)std::strtoull(e, nullptr, 10) << 20;
    }

    void drop(DevicePool &d, std::multimap<size_t, Kept>::iterator it) {
        (void)hipFree(it->second.p);
        kept_bytes -= it->first;
        d.kept.erase(it);
    }
    void drop_old(Clock::time_point now) {
        for (auto &d : dev)
            for (auto it = d.second.kept.begin(); it != d.second.kept.end();) {
                const auto cur = it++;
                if (std::chrono::duration<double>(now - cur->second.at).count() > kKeepSeconds) drop(d.second, cur);
            }
    }
    void drop_oldest() {
        DevicePool *of = nullptr;
        std::multimap<size_t, Kept>::iterator old;
        for (auto &d : dev)
            for (auto it = d.second.kept.begin(); it != d.second.kept.end(); ++it)
                if (!of || it->second.released < old->second.released) {
                    of = &d.second;
                    old = it;
                }
        if (of) drop(*of, old);
    }
    void drop_all() {
        for (auto &d : dev)
            while (!d.second.kept.empty()) drop(d.second, d.second.kept.begin());
    }
};

// never destroyed: handles may be released while the process ends
Pool &pool() {
    static Pool *p = new Pool();
    return *p;
}

// 512-byte steps up to 1 MiB, 2 MiB steps above: sizes that recur for one structure stay equal
size_t rounded(size_t bytes) {
    const size_t step = bytes <= ((size_t)1 << 20) ? 512 : (size_t)2 << 20;
    return (bytes + step - 1) / step * step;
}

}  // namespace

void *device_alloc(size_t bytes) {
    int device = 0;
    NKPR_HIP(hipGetDevice(&device));
    Pool &P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    const bool keep = bytes <= kLargest && P.limit > 0;
    const size_t want = keep ? rounded(bytes) : bytes;
    if (keep) {
        DevicePool &d = P.dev[device];
        P.drop_old(Clock::now());
        // the smallest block that fits and wastes less than a quarter
        const auto it = d.kept.lower_bound(want);
        if (it != d.kept.end() && it->first <= want + want / 4) {
            if (it->second.released > d.synced) {
                NKPR_HIP(hipDeviceSynchronize());
                d.synced = P.releases;
            }
            void *p = it->second.p;
            P.live[p] = {device, it->first};
            P.kept_bytes -= it->first;
            d.kept.erase(it);
            return p;
        }
    }
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, want);
    if (e != hipSuccess && P.kept_bytes > 0) {
        (void)hipGetLastError();
        P.drop_all();
        e = hipMalloc(&p, want);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        throw Error(NKPR_ERR_NOMEM, "hipMalloc(" + std::to_string(bytes) + " bytes) failed: " + hipGetErrorString(e));
    }
    if (keep) P.live[p] = {device, want};
    return p;
}

void device_free(void *p) {
    if (!p) return;
    Pool &P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    const auto it = P.live.find(p);
    if (it == P.live.end()) {
        (void)hipFree(p);
        return;
    }
    const Live b = it->second;
    P.live.erase(it);
    const Clock::time_point now = Clock::now();
    P.drop_old(now);
    if (b.bytes > P.limit) {
        (void)hipFree(p);
        return;
    }
    while (P.kept_bytes + b.bytes > P.limit) P.drop_oldest();
    P.dev[b.device].kept.emplace(b.bytes, Kept{p, ++P.releases, now});
    P.kept_bytes += b.bytes;
}

void release_kept() {
    Pool &P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    P.drop_all();
}

void *pinned_alloc(size_t bytes) {
    Pool &P = pool();
    void *p = nullptr;
    if (bytes <= kPinnedBytes) {
        std::lock_guard<std::mutex> lock(P.mu);
        if (!P.pinned.empty()) {
            p = P.pinned.back();
            P.pinned.pop_back();
            return p;
        }
    }
    NKPR_CHECK(bytes <= kPinnedBytes, "pinned buffers are small");
    NKPR_HIP(hipHostMalloc(&p, kPinnedBytes, hipHostMallocDefault));
    return p;
}

void pinned_free(void *p) {
    if (!p) return;
    Pool &P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    if (P.pinned.size() < kMostPinned) P.pinned.push_back(p);
    else (void)hipHostFree(p);
}

hipStream_t stream_get() {
    int device = 0;
    NKPR_HIP(hipGetDevice(&device));
    {
        Pool &P = pool();
        std::lock_guard<std::mutex> lock(P.mu);
        std::vector<hipStream_t> &idle = P.dev[device].streams;
        if (!idle.empty()) {
            const hipStream_t s = idle.back();
            idle.pop_back();
            return s;
        }
    }
    hipStream_t s = nullptr;
    NKPR_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    return s;
}

void stream_put(hipStream_t s, int device) {
    if (!s) return;
    // an idle, healthy stream can serve the next handle
    const bool idle = hipStreamSynchronize(s) == hipSuccess;
    Pool &P = pool();
    std::lock_guard<std::mutex> lock(P.mu);
    std::vector<hipStream_t> &kept = P.dev[device].streams;
    if (idle && kept.size() < kMostStreams) kept.push_back(s);
    else (void)hipStreamDestroy(s);
}

}  // namespace nkpr
