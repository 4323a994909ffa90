// The library's plain host arithmetic, called by tests/test_host_arithmetic.py.
#include "../../quids_amd/csrc/qd_sizes.hpp"

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
