// The 17-64-row kernel of mnb_rows64.hpp: blocks of 32.
#include "mnb_rows64.hpp"

namespace mnb {

hipError_t launch_rows64_bs32(const Rows64Geom& g, const void* a, const uint8_t* b,
                             const uint8_t* strips, const void* s, const uint8_t* z, void* y,
                             int64_t m, int64_t n, int64_t k, hipStream_t st) {
    return rows64_bs<32>(g, a, b, strips, s, z, y, m, n, k, st);
}

}  // namespace mnb
