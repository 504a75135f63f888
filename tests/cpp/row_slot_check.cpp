// row_slot_check.cpp -- row_slot (honei_amd/csrc/row_slot.hh), the buffer
// offsets of the wide-row product, for every stored width the kernels take,
// entries up to their compile-time widths and strides up to the largest
// buffer: an entry of the row lies at its place inside the buffer, any other
// is outside whichever way the range check combines the two offsets.
// Exit status 0 when all hold.

#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "row_slot.hh"

using namespace honei::hipx;

int main() {
    for (uint32_t width = 17; width <= 28; ++width) {
        const uint32_t least = width <= 24 ? 17 : 25, entries = width <= 24 ? 24 : 28;
        const uint32_t most = (uint32_t)((((uint64_t)1 << 31) - 1) / 4 / width / 32 * 32);
        for (uint32_t stride : {98304u, 1000032u, most}) {
            const uint32_t bytes = width * stride * 4;
            for (uint32_t row : {0u, 1u, stride / 2, stride - 1})
                for (uint32_t len = 0; len <= width; ++len)
                    for (uint32_t k = 0; k < entries; ++k) {
                        const RowSlot e = row_slot(row, k, len, stride, bytes, least);
                        bool ok;
                        if (k < len)
                            ok = (uint64_t)e.lane + e.wave == ((uint64_t)k * stride + row) * 4;
                        else
                            ok = e.lane >= bytes && e.lane >= (uint32_t)(bytes - e.wave) &&
                                 (uint64_t)e.lane + e.wave >= bytes && (uint64_t)e.lane + e.wave + 4 <= UINT32_MAX;
                        if (!ok) {
                            std::printf("width %u stride %u row %u length %u entry %u: %u + %u of %u\n", width, stride,
                                        row, len, k, e.lane, e.wave, bytes);
                            return 1;
                        }
                    }
        }
    }
    std::printf("every entry in place\n");
    return 0;
}
