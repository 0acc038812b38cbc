// The prefill GEMM of mnb_gemm_direct.hpp: 8-bit weights.
#include "mnb_gemm_direct.hpp"

namespace mnb {

hipError_t launch_gemm_direct_b8(int bs, const GemmConfig& c, const void* a, const uint8_t* b,
                                 const void* s, const uint8_t* z, void* y, int64_t m, int64_t n,
                                 int64_t k, float* part, hipStream_t st) {
    return direct_bs<8, false>(bs, c, a, b, s, z, y, m, n, k, part, st);
}

}  // namespace mnb
