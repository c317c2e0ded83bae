// Device buffers the library allocates and frees on every call of a kind: the
// outputs of vj_join and vj_join_rows and the latter's transposed key columns.
//
// hipMalloc and hipFree of tens of megabytes cost up to a few hundred
// microseconds each (and hipFree waits for the device), more than the join of
// such tables. A buffer that comes back is kept here and handed out again to a
// request of at most its size and at least half of it.
//
//  - A buffer enters the list only when nothing on its device can still use
//    it: its last user waited for the device (or, inside the library, for the
//    stream of all its work), as hipFree would have. So it may go to any
//    stream and any thread next.
//  - At most kCacheBytes per device are kept, the oldest go first. Everything
//    is given back when the last context on a device is destroyed, and before
//    any allocation of the library is reported as failed.
//  - Buffers are ordinary hipMalloc allocations: an output may also be passed
//    to hipFree by its owner. What the list knows of such a buffer is checked
//    against the runtime's own record before it is trusted.
//  - Contexts under an HBM budget neither take from the list nor add to it.
#include <deque>
#include <mutex>
#include <unordered_map>

#include "vj_internal.hpp"

namespace vj {

namespace {

constexpr size_t kCacheBytes = (size_t)1 << 30;

struct Buf {
    void *p;
    size_t bytes;
    int device;
};

struct Cache {
    std::mutex m;
    std::deque<Buf> idle;                     // oldest first
    std::unordered_map<void *, Buf> out;      // handed out and to be kept on return
    std::unordered_map<int, int> contexts;    // live contexts per device
};

Cache &cache() {
    static Cache *c = new Cache();  // never destroyed: no device calls at process exit
    return *c;
}

int current_device() {
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess) {
        (void)hipGetLastError();
        d = -1;
    }
    return d;
}

// Frees the idle buffers of `device` beyond `keep` bytes, oldest first (m held).
void trim(Cache &c, int device, size_t keep) {
    size_t held = 0;
    for (const Buf &b : c.idle)
        if (b.device == device) held += b.bytes;
    for (auto it = c.idle.begin(); it != c.idle.end() && held > keep;) {
        if (it->device != device) {
            ++it;
            continue;
        }
        held -= it->bytes;
        (void)hipFree(it->p);
        it = c.idle.erase(it);
    }
}

}  // namespace

void cache_context(int device, int delta) {
    Cache &c = cache();
    std::lock_guard<std::mutex> lock(c.m);
    if ((c.contexts[device] += delta) <= 0) trim(c, device, 0);
}

hipError_t device_malloc(void **p, size_t bytes) {
    *p = nullptr;
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    *p = nullptr;
    {
        Cache &c = cache();
        std::lock_guard<std::mutex> lock(c.m);
        trim(c, current_device(), 0);
    }
    e = hipMalloc(p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
    }
    return e;
}

hipError_t cache_malloc(void **p, size_t bytes, bool keep) {
    if (!keep) return device_malloc(p, bytes);
    const int device = current_device();
    Cache &c = cache();
    {
        std::lock_guard<std::mutex> lock(c.m);
        auto best = c.idle.end();
        for (auto it = c.idle.begin(); it != c.idle.end(); ++it)
            if (it->device == device && it->bytes >= bytes && it->bytes / 2 <= bytes &&
                (best == c.idle.end() || it->bytes < best->bytes))
                best = it;
        if (best != c.idle.end()) {
            const Buf b = *best;
            c.idle.erase(best);
            c.out[b.p] = b;
            *p = b.p;
            return hipSuccess;
        }
    }
    // an eighth of its power of two at most is rounded up, so that calls of about the same size share buffers
    size_t step = 4096;
    while (step * 16 <= bytes) step <<= 1;
    const size_t want = (bytes + step - 1) / step * step;
    const hipError_t e = device_malloc(p, want);
    if (e != hipSuccess) return device_malloc(p, bytes);
    if (want <= kCacheBytes / 2) {
        std::lock_guard<std::mutex> lock(c.m);
        c.out[*p] = Buf{*p, want, device};
    }
    return hipSuccess;
}

void cache_free(void *p, bool idle) {
    if (!p) return;
    Cache &c = cache();
    Buf b{nullptr, 0, -1};
    {
        std::lock_guard<std::mutex> lock(c.m);
        auto it = c.out.find(p);
        if (it != c.out.end()) {
            b = it->second;
            c.out.erase(it);
        }
    }
    if (b.p) {
        hipDeviceptr_t base = nullptr;
        size_t size = 0;
        const hipError_t e = hipMemGetAddressRange(&base, &size, p);
        if (e != hipSuccess) (void)hipGetLastError();
        if (e == hipSuccess && base == p && size >= b.bytes) {
            const int cur = current_device();
            bool ok = true;
            if (!idle) {  // as hipFree: whatever still uses it ends first
                ok = hipSetDevice(b.device) == hipSuccess && hipDeviceSynchronize() == hipSuccess;
                if (cur >= 0 && cur != b.device) (void)hipSetDevice(cur);
            }
            if (ok) {
                std::lock_guard<std::mutex> lock(c.m);
                if (c.contexts[b.device] > 0) {
                    c.idle.push_back(b);
                    trim(c, b.device, kCacheBytes);
                    return;
                }
            } else {
                (void)hipGetLastError();
            }
        }
    }
    (void)hipFree(p);
}

}  // namespace vj
