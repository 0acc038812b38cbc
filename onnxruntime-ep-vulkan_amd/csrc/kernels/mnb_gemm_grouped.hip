// The prefill GEMM of mnb_gemm_direct.hpp over the experts of a mixture of experts: every expert's
// rows times its own int4 weights in one launch.
//
// Tiles of 128 rows x 192 columns (128 for blocks of 64 and 128), as many row tiles as the experts'
// row counts need; a tile with at most 64 or 32 rows multiplies only those quarters, so an expert's last tile costs what its
// rows cost (1024 tokens over 32 experts, 4 each: 128 rows per expert on average, half of the
// experts with a few rows in a second tile).
#include "mnb_gemm_direct.hpp"

namespace mnb {

bool gemm_grouped_supported(int64_t rows, int64_t a_rows, int64_t experts, int64_t n, int64_t k,
                            int bs, const void* a, const void* b) {
    if (bs != 32 && bs != 64 && bs != 128) return false;
    if (rows < 1 || experts < 1 || rows + experts >= (int64_t)1 << 24) return false;
    if (!gemm_supported(std::max(rows, a_rows), n, k, 4, bs, false)) return false;
    return reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(b) % 16 == 0;
}

template <int BS, bool NATIVE, int MODE>
static hipError_t grouped_go(const DirectGroups& grp, const void* a, const uint8_t* b,
                             const void* s, void* y, int64_t rows, int64_t a_rows, int64_t n,
                             int64_t k, hipStream_t st) {
    using T = DirectTile<4, BS, kTile128x192>;
    constexpr int kBM = 16 * T::MT, kBN = 16 * T::S * T::NW;
    auto kern = gemm_direct<4, BS, false, T::MT, T::S, T::NW, NATIVE, MODE>;
    const int64_t tiles_n = (n + kBN - 1) / kBN;
    // at most one partial row tile per expert that has rows
    const int64_t items = (rows / kBM + std::min<int64_t>(grp.experts, rows)) * tiles_n;
    const dim3 grid((unsigned)(8 * ((items + 7) / 8)), 1, 1);
    hipLaunchKernelGGL(kern, grid, dim3(64 * T::NW), 2 * kBM * 256, st, static_cast<const f16*>(a),
                       b, static_cast<const f16*>(s), nullptr, static_cast<f16*>(y), 0, (int)n,
                       (int)k, 0, (int)tiles_n, 1, nullptr, (uint32_t)(a_rows * k * 2), grp);
    return hipGetLastError();
}

hipError_t launch_gemm_grouped(const void* a, int64_t a_rows, const int32_t* row_index,
                               const int32_t* offsets, int64_t experts, const uint8_t* b,
                               const uint8_t* b_strips, const void* s, void* y, int64_t rows,
                               int64_t n, int64_t k, int bs, hipStream_t st,
                               const StripSwiglu* sw) {
    if (rows == 0) return hipSuccess;
    DirectGroups g{offsets, row_index, nullptr, (int)experts, 0.f, 0.f, 0.f, 0};
    if (sw) {
        if (n % 2) return hipErrorInvalidValue;
        g.bias = static_cast<const f16*>(sw->bias);
        g.alpha = sw->alpha;
        g.beta = sw->beta;
        g.limit = sw->limit;
        g.has_limit = sw->has_limit;
    }
#define MNB_GG(BS_)                                                                              \
    case BS_:                                                                                    \
        if (b_strips)                                                                            \
            return sw ? grouped_go<BS_, true, kGroupedSwiglu>(g, a, b_strips, s, y, rows,        \
                                                              a_rows, n, k, st)                  \
                      : grouped_go<BS_, true, kGrouped>(g, a, b_strips, s, y, rows, a_rows, n,   \
                                                        k, st);                                  \
        return sw ? grouped_go<BS_, false, kGroupedSwiglu>(g, a, b, s, y, rows, a_rows, n, k,    \
                                                           st)                                   \
                  : grouped_go<BS_, false, kGrouped>(g, a, b, s, y, rows, a_rows, n, k, st)
    switch (bs) {
        MNB_GG(32);
        MNB_GG(64);
        MNB_GG(128);
        default: return hipErrorInvalidValue;
    }
#undef MNB_GG
}

}  // namespace mnb
