// row_slot.hh -- offsets of a row's entries in an ELL array of 4-byte elements
// read through a buffer.  Plain C++ on the host, HIP on the device, so the
// host-side check runs the very code the kernels use.
#pragma once

#include <cstdint>

#include "exact_div.hh"   // HONEI_HD

namespace honei {
namespace hipx {

constexpr uint32_t kOutside = 0x80000000u;   // beyond every buffer (they end below 2^31)

// Byte offsets of entry k of `row`: the lane's and the wavefront's.  Entries
// past the row's length are asked for outside the buffer (no memory access)
// by the lane's offset; the wavefront's is at most the buffer's size also
// where k is past the stored width (only entries from `least` on can be), so
// a range check that takes it off that size cannot wrap.
struct RowSlot {
    uint32_t lane, wave;
};
HONEI_HD inline RowSlot row_slot(uint32_t row, uint32_t k, uint32_t len, uint32_t stride, uint32_t bytes,
                                 uint32_t least) {
    const uint32_t at = k * stride * 4u;
    return RowSlot{k < len ? row * 4u : kOutside, k >= least && at > bytes ? bytes : at};
}

}  // namespace hipx
}  // namespace honei
