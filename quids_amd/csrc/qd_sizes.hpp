#pragma once
// Sizes and places of objects in a state's buffers: plain integer arithmetic
// of the kernels and of the host code (no HIP, so that a host compiler builds
// it for the tests).
#include <cstddef>

#include "qd_rules.hpp"

namespace qd {

// Zero bytes that follow an object (quids::get_alignment_offset, src/quids.hpp:93-102).
QD_HD u32 align_pad(u32 size, u32 align) {
    if (align <= 1) return 0;
    const u32 off = align - size % align;
    return off == align ? 0 : off;
}

// First bytes at[k] of the n <= PER objects of the given sizes, one after the
// other from 0; returns the byte after the last.  (64 bits: one object and
// its padding may pass 2^32, and so may a tile of objects of 1 MB each.)
template <u32 PER>
QD_HD u64 place_run(const u32 *size, u32 n, u32 align, u64 (&at)[PER]) {
    u64 end = 0;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
    for (u32 k = 0; k < PER; ++k) {
        at[k] = end;
        if (k < n) end += u64(size[k]) + align_pad(size[k], align);
    }
    return end;
}

// Objects that a state's begin, size and magnitude buffers of these bytes
// hold (begin has one entry more than there are objects; a buffer whose
// allocation failed has 0 bytes).
QD_HD u64 state_room(u64 begin, u64 size, u64 mag) {
    u64 n = begin / sizeof(u64);
    if (n) --n;
    if (size / sizeof(u32) < n) n = size / sizeof(u32);
    if (mag / (2 * sizeof(double)) < n) n = mag / (2 * sizeof(double));
    return n;
}

}  // namespace qd
