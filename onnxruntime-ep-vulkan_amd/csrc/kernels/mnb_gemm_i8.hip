// accuracy_level 4 above 64 rows: int8 MFMA GEMM on gfx950 (int8 activation codes with one
// fp32 scale per row and block, int4 weights, fp16 scales and output).
//
// What bounds it.  As in the fp16 prefill GEMM (mnb_gemm_direct.hpp, whose tiling and loads it
// shares) the VALU: each output of each block takes int32 -> fp32, the weight scale and the
// activation scale.  Two FMAs do it: the MFMA's accumulator starts at the bits of 1.5 * 2^23, so
// its int32 result, read as a float, is 1.5 * 2^23 + dot exactly (|dot| < 2^22), and
//   t = fma(that, sb, -1.5 * 2^23 * sb) = dot * sb, rounded once;  acc = fma(t, sa, acc).
// At 512 rows of 3072 x 8192 (block 32) the row-tiled int8 GEMV, one wavefront per strip and 64
// rows with A gathered through the caches, took 305 us; this kernel 53.
//
// Work split.  A workgroup of four wavefronts, side by side along N, owns 16 MT rows x 64 S
// columns and walks K in quads of 128 k; A's codes (128 bytes per row and quad) and activation
// scales come a pair of quads ahead by LDS DMA, the weights likewise into registers (the int8
// strip copy, or ORT's layout and the 4 x 4 dword transpose).  16-byte slot s of row r sits at
// s ^ ((r >> 1) & 7), so the 8-byte operand reads of 16 rows touch every bank once.
#include <algorithm>
#include <type_traits>

#include "mnb_common.hpp"
#include "mnb_gemm_direct.hpp"
#include "mnb_launch.hpp"

namespace mnb {

namespace {

constexpr int kI8Waves = 4;

template <int BS, bool HAS_ZP, int MT, int S, bool NATIVE>
__global__ void __launch_bounds__(64 * kI8Waves) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_i8(const int8_t* __restrict__ A, const float* __restrict__ Sa, const uint8_t* __restrict__ B,
        const f16* __restrict__ Sc, const uint8_t* __restrict__ Z, f16* __restrict__ Y, int M, int N,
        int K, int tiles_m, int tiles_n) {
    constexpr int NW = kI8Waves;
    constexpr int CPB = BS / 32;                         // 32-k chunks per block
    constexpr int BPQ = 4 / CPB;                         // blocks per quad
    constexpr int kRows = 16 * MT;
    constexpr int AI = (kRows / 8) / NW;                 // A loads per wavefront: 8 rows each
    constexpr int SI = BPQ * kRows / 64;                 // 4-byte loads of activation scales
    constexpr int SPW = (SI + NW - 1) / NW;              // ... per wavefront
    constexpr int kQuad = kRows * 128 + SI * 256;        // a quad's codes and scales
    static_assert(AI >= 1 && kRows % 64 == 0, "loads per wavefront");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15;
    const int g = lane >> 4;
    const int V = tiles_m * tiles_n;
    const int per_xcd = (V + 7) >> 3;
    const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || item >= V) return;   // before any barrier
    const int tile_m = item / tiles_n;
    const int tile_n = item - tile_m * tiles_n;
    const int m0 = tile_m * kRows;
    const int bpc = K / BS;
    const int zpb = (bpc + 1) >> 1;
    const int strips = (N + 15) >> 4;
    const int KQ = (K + 127) >> 7;
    const int strip0 = (tile_n * NW + wave) * S;
    const bool active = strip0 < strips;                 // else: only its share of the loads

    uint32_t a_off[AI];
#pragma unroll
    for (int j = 0; j < AI; ++j) {
        const int row = 8 * (AI * wave + j) + (lane >> 3);
        const int gm = min(m0 + row, M - 1);             // clamped rows are never stored
        a_off[j] = (uint32_t)((int64_t)gm * K + 16 * ((lane & 7) ^ ((row >> 1) & 7)));
    }
    // scales [block][M]: load i of a quad takes 64 rows of one block (rows past M read the next
    // block's and are never stored)
    auto sa_off = [&](int i) {
        return (uint32_t)(((64 * i / kRows) * (int64_t)M + m0 + 64 * i % kRows + lane) * 4);
    };
    const auto ra = buffer_of(A, (uint32_t)((int64_t)M * K));
    const auto rs = buffer_of(Sa, (uint32_t)((int64_t)bpc * M * 4));
    const auto rb = buffer_of(B, (uint32_t)(NATIVE ? (int64_t)strips * KQ * 1024 : (int64_t)N * (K / 2)));
    // quad q lands in one of four places: the pair in use and the next
    auto issue_a = [&](int q) {
        uint8_t* dst = smem + (q & 3) * kQuad;
#pragma unroll
        for (int j = 0; j < AI; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                ra, (lds_void_ptr)(dst + (wave * AI + j) * 1024), 16, (int)a_off[j],
                __builtin_amdgcn_readfirstlane(128 * q), 0, 0);
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            const int i = wave * SPW + j;
            if (i < SI)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rs, (lds_void_ptr)(dst + kRows * 128 + i * 256), 4, (int)sa_off(i),
                    __builtin_amdgcn_readfirstlane(q * BPQ * M * 4), 0, 0);
        }
    };
    uint32_t b_off[S], s_off[S], z_off[S];
#pragma unroll
    for (int t = 0; t < S; ++t) {
        const int col = min(16 * (strip0 + t) + nl, N - 1);
        if constexpr (NATIVE)
            b_off[t] = (uint32_t)((int64_t)min(strip0 + t, strips - 1) * KQ * 1024 + 64 * nl + 16 * g);
        else
            b_off[t] = (uint32_t)((int64_t)col * (K / 2) + 16 * g);
        s_off[t] = (uint32_t)(col * bpc * 2);
        z_off[t] = (uint32_t)(col * zpb);
    }
    auto load_w = [&](u32x4 (&w)[S], int q) {
        const int so = __builtin_amdgcn_readfirstlane(q * (NATIVE ? 1024 : 64));
#pragma unroll
        for (int t = 0; t < S; ++t) w[t] = buffer_load16(rb, b_off[t], (uint32_t)so);
    };
    using Pair = ScalePair<4, BS, HAS_ZP, S>;

    f32x4 acc[MT][S];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < S; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the lane part of the operand reads: row 16 i + nl, chunk c, bytes 8 g .. + 7 of its 32
    int a_lane[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        a_lane[c] = nl * 128 + (((2 * c + (g >> 1)) ^ ((nl >> 1) & 7)) << 4) + 8 * (g & 1);
    constexpr float kMagic = 12582912.f;                 // 1.5 * 2^23, bits 0x4B400000
    const i32x4 magic = {0x4B400000, 0x4B400000, 0x4B400000, 0x4B400000};

    auto compute = [&](const u32x4 (&rw)[S], const Pair& r, int q, auto half_c) {
        constexpr int half = decltype(half_c)::value;    // quad of the pair
        const uint8_t* base = smem + (q & 3) * kQuad;
        const uint8_t* sbase = base + kRows * 128 + 16 * g;
        uint32_t wv[S][4];
#pragma unroll
        for (int t = 0; t < S; ++t) {
            wv[t][0] = rw[t].x;
            wv[t][1] = rw[t].y;
            wv[t][2] = rw[t].z;
            wv[t][3] = rw[t].w;
            if constexpr (!NATIVE) transpose_rows(wv[t][0], wv[t][1], wv[t][2], wv[t][3]);
        }
        const int blocks = min(BPQ, ((K >> 5) - 4 * q) / CPB);
#pragma unroll
        for (int bq = 0; bq < BPQ; ++bq) {
            if (bq >= blocks) break;                     // uniform: the missing half of a quad
            long bop[S][CPB];
            float sb[S], nb[S];
#pragma unroll
            for (int t = 0; t < S; ++t) {
                sb[t] = r.scale(t, half * BPQ + bq);
                nb[t] = -kMagic * sb[t];                 // exact: 13 bits
                const uint32_t zb = (128u - r.zero(t, half * BPQ + bq)) * 0x01010101u;
#pragma unroll
                for (int cc = 0; cc < CPB; ++cc)
                    bop[t][cc] = __builtin_bit_cast(long, qz_i8(wv[t][bq * CPB + cc], zb));
            }
            // Four row tiles of all strips at a time: reads, MFMAs, then the scaled adds (a tile
            // at a time every MFMA waited for its reads and every add for its MFMA, 110 cycles).
#pragma unroll
            for (int f = 0; f < MT / 4; ++f) {
                long a[4][CPB];
                f32x4 sa[4];
                i32x4 d[4][S];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
#pragma unroll
                    for (int cc = 0; cc < CPB; ++cc)
                        a[i][cc] = *reinterpret_cast<const long*>(base + a_lane[bq * CPB + cc] +
                                                                  2048 * (4 * f + i));
                    sa[i] = *reinterpret_cast<const f32x4*>(sbase + (bq * MT + 4 * f + i) * 64);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int t = 0; t < S; ++t) {
                        d[i][t] = magic;
#pragma unroll
                        for (int cc = 0; cc < CPB; ++cc)
                            d[i][t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[i][cc], bop[t][cc],
                                                                           d[i][t], 0, 0, 0);
                    }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int t = 0; t < S; ++t) {
                        const f32x4 v = __builtin_bit_cast(f32x4, d[i][t]);
                        f32x4& o = acc[4 * f + i][t];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[e] = __builtin_fmaf(__builtin_fmaf(v[e], sb[t], nb[t]), sa[i][e], o[e]);
                    }
            }
        }
    };

    // Pairs of quads, everything one pair ahead: with few workgroups the time of a step is the
    // latency of its loads (1.75 us a quad with quads as steps).
    u32x4 w0[2][S], w1[2][S];
    Pair p0, p1;
    auto fetch = [&](int q, u32x4 (&w)[2][S], Pair& p) {
        issue_a(q);
        load_w(w[0], q);
        if (q + 1 < KQ) {
            issue_a(q + 1);
            load_w(w[1], q + 1);
        }
        p.load(Sc, Z, s_off, z_off, q * BPQ, bpc, zpb);
    };
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    auto step = [&](int q, u32x4 (&now)[2][S], u32x4 (&next)[2][S], const Pair& p, Pair& pn) {
        __builtin_amdgcn_s_waitcnt(0x7 << 4);            // vmcnt(0) lgkmcnt(0)
        wg_barrier();
        if (q + 2 < KQ) fetch(q + 2, next, pn);
        __builtin_amdgcn_sched_barrier(0);
        if (!active) return;
        compute(now[0], p, q, H0{});
        if (q + 1 < KQ) compute(now[1], p, q + 1, H1{});
    };
    fetch(0, w0, p0);
    for (int q = 0; q < KQ; q += 4) {
        step(q, w0, w1, p0, p1);
        if (q + 2 >= KQ) break;
        step(q + 2, w1, w0, p1, p0);
    }
    if (!active) return;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < S; ++t) {
            const int col = 16 * (strip0 + t) + nl;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + 16 * i + 4 * g + e;
                if (row < M && col < N) Y[(int64_t)row * N + col] = (f16)acc[i][t][e];
            }
        }
}

template <int BS, int MT, int S>
hipError_t i8_go(const GemmI8Geom& c, const int8_t* qa, const float* sa, const uint8_t* b,
                 const uint8_t* strips, const void* s, const uint8_t* z, void* y, int64_t m,
                 int64_t n, int64_t k, hipStream_t st) {
    constexpr int kLds = 4 * 16 * MT * (128 + 128 / BS * 4);
    const int64_t items = c.tiles_m * c.tiles_n;
    const dim3 grid((unsigned)(8 * ((items + 7) / 8)), 1, 1);
    auto go = [&](auto kern, const uint8_t* w) {
        const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), kLds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, grid, dim3(64 * kI8Waves), kLds, st, qa, sa, w,
                           static_cast<const f16*>(s), z, static_cast<f16*>(y), (int)m, (int)n,
                           (int)k, (int)c.tiles_m, (int)c.tiles_n);
        return hipGetLastError();
    };
    if (strips)
        return z ? go(gemm_i8<BS, true, MT, S, true>, strips)
                 : go(gemm_i8<BS, false, MT, S, true>, strips);
    return z ? go(gemm_i8<BS, true, MT, S, false>, b) : go(gemm_i8<BS, false, MT, S, false>, b);
}

template <int BS>
hipError_t i8_tile(const GemmI8Geom& c, const int8_t* qa, const float* sa, const uint8_t* b,
                   const uint8_t* strips, const void* s, const uint8_t* z, void* y, int64_t m,
                   int64_t n, int64_t k, hipStream_t st) {
    if (c.bm == 128) return i8_go<BS, 8, 2>(c, qa, sa, b, strips, s, z, y, m, n, k, st);
    if (c.bm == 64) return i8_go<BS, 4, 2>(c, qa, sa, b, strips, s, z, y, m, n, k, st);
    return hipErrorInvalidValue;
}

}  // namespace

bool gemm_i8_geometry(int64_t m, int64_t n, int64_t k, int bits, int bs, GemmI8Geom* out) {
    // Up to 64 rows, and on small nodes up to 256, the row-tiled GEMV's shorter chains win (its time
    // steps up past 64 rows): 3072 x 8192 at 64 / 96 / 256 / 512 rows 33.8 / 34.7 / 37.2 / 57.7 us
    // here, 36.1 / 55.1 / 153 / 307 there; 8192 x 3072 (block 128) 49.9 / 50.8 / 52.0 / 54.2
    // against 42.8 / 62.2 / 107 / 234; 1024 x 1000 at 96 / 256 / 512 rows 12.8 / 13.0 / 13.2
    // against 11.6 / 12.0 / 19.5.
    if (m <= 64 || (m <= 256 && n * k < (int64_t)4 << 20)) return false;
    if (bits != 4 || (bs != 32 && bs != 64 && bs != 128)) return false;
    if (!gemm_supported(m, n, k, bits, bs, false)) return false;
    GemmI8Geom g{};
    g.bn = 128;
    if (m * (k / bs) * 4 >= (int64_t)1 << 32) return false;
    g.tiles_n = (n + 127) / 128;
    // 128-row tiles read and convert B half as often, and win once they fill every CU twice: 64- /
    // 128-row tiles on 3072 x 8192 (block 32) at 512 / 768 / 1024 / 2048 rows 60.4 / 84.3 / 102 /
    // 194 us against 61.7 / 86.5 / 91.9 / 169; 3072 x 3072 at 1024 / 2048 rows (192 and 384
    // 128-row tiles) 52.0 / 80.2 against 56.4 / 85.0.
    g.bm = (m + 127) / 128 * g.tiles_n >= 512 ? 128 : 64;
    g.tiles_m = (m + g.bm - 1) / g.bm;
    *out = g;
    return true;
}

hipError_t launch_gemm_i8(const GemmI8Geom& c, const int8_t* qa, const float* sa,
                          const uint8_t* b, const uint8_t* strips, const void* s,
                          const uint8_t* z, void* y, int64_t m, int64_t n, int64_t k, int bs,
                          hipStream_t st) {
    switch (bs) {
        case 32: return i8_tile<32>(c, qa, sa, b, strips, s, z, y, m, n, k, st);
        case 64: return i8_tile<64>(c, qa, sa, b, strips, s, z, y, m, n, k, st);
        case 128: return i8_tile<128>(c, qa, sa, b, strips, s, z, y, m, n, k, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mnb
