#pragma once
// Device buffers of a context's states between uses (host code).
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <mutex>
#include <vector>

namespace qd {

// State buffers given up (a state closed, or grown) and not yet returned to
// the device, for the context's next ones: mapping and unmapping 10 MB to
// 1 GB costs 25-300 us each time, and a program that makes a state per step
// (the gradient's forward pass) spent a quarter of its time on it.  Bounded
// (kPoolBytes); given back when an allocation does not fit, when the context
// is trimmed or destroyed, and before free memory decides anything.
struct StatePool {
    struct Buf {
        void *p;
        size_t cap;
    };
    std::mutex m;
    std::vector<Buf> bufs;  // oldest first
    size_t bytes = 0;
    // the smallest buffer of at least `want` bytes, and at most twice that
    // (plus 1 MB), or nothing
    Buf take(size_t want) {
        std::lock_guard<std::mutex> g(m);
        size_t best = bufs.size();
        for (size_t i = 0; i < bufs.size(); ++i)
            if (bufs[i].cap >= want && bufs[i].cap <= 2 * want + (1 << 20) &&
                (best == bufs.size() || bufs[i].cap < bufs[best].cap))
                best = i;
        if (best == bufs.size()) return {nullptr, 0};
        const Buf b = bufs[best];
        bufs.erase(bufs.begin() + long(best));
        bytes -= b.cap;
        return b;
    }
    // The device has finished with a buffer that is kept (an unmapping waits
    // for it, whatever stream used it); where that cannot be waited for, while
    // a stream is captured for instance, the buffer is unmapped.
    void give(void *p, size_t cap) {
        constexpr size_t kSmall = 64 << 10;  // the runtime hands these out in a microsecond itself
        if (hipDeviceSynchronize() != hipSuccess) {
            (void)hipGetLastError();
            (void)hipFree(p);
            return;
        }
        if (cap < kSmall || cap > kPoolBytes / 2) {
            (void)hipFree(p);
            return;
        }
        std::lock_guard<std::mutex> g(m);
        while (!bufs.empty() && (bytes + cap > kPoolBytes || bufs.size() >= 64)) {
            (void)hipFree(bufs.front().p);
            bytes -= bufs.front().cap;
            bufs.erase(bufs.begin());
        }
        bufs.push_back({p, cap});
        bytes += cap;
    }
    size_t held() {
        std::lock_guard<std::mutex> g(m);
        return bytes;
    }
    void trim() {
        std::lock_guard<std::mutex> g(m);
        for (Buf &b : bufs) (void)hipFree(b.p);
        bufs.clear();
        bytes = 0;
    }
    static constexpr size_t kPoolBytes = 4ull << 30;
};

}  // namespace qd
