// The library's plain host code, called by tests/test_host_arithmetic.py.
#include "../../quids_amd/csrc/qd_pool.hpp"
#include "../../quids_amd/csrc/qd_sizes.hpp"

// The HIP calls of the pool: what is freed is counted, and the wait for the
// device ends as the test says.
static hipError_t sync_result = hipSuccess;
static uint64_t freed;
extern "C" hipError_t hipDeviceSynchronize(void) { return sync_result; }
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }
extern "C" hipError_t hipFree(void *) {
    ++freed;
    return hipSuccess;
}

// First bytes of n <= 4 objects, and the byte after the last.
extern "C" uint64_t host_place_run(const uint32_t *size, uint32_t n, uint32_t align, uint64_t *at) {
    uint64_t a[4];
    const uint64_t end = qd::place_run(size, n, align, a);
    for (int k = 0; k < 4; ++k) at[k] = a[k];
    return end;
}

extern "C" uint64_t host_state_room(uint64_t begin, uint64_t size, uint64_t mag) {
    return qd::state_room(begin, size, mag);
}

// Gives n buffers of `bytes` to a new pool, the first `failing` of them while
// the device cannot be waited for; returns the bytes kept, and how many
// buffers were freed.
extern "C" uint64_t host_pool_give(uint64_t n, uint64_t failing, uint64_t bytes, uint64_t *num_freed) {
    qd::StatePool pool;
    freed = 0;
    for (uint64_t i = 0; i < n; ++i) {
        sync_result = i < failing ? hipErrorStreamCaptureUnsupported : hipSuccess;
        pool.give(reinterpret_cast<void *>((i + 1) << 40), bytes);
    }
    sync_result = hipSuccess;
    *num_freed = freed;
    return pool.held();
}
