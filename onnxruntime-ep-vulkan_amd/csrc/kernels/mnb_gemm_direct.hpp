// Prefill MatMulNBits on gfx950, blocks of 32, 64 or 128: fp16 MFMA GEMM whose weights go from
// memory straight into each wavefront's registers (fp16 A; 4- or 8-bit weights).
//
// What bounds it.  The exact per-block rescale: one fp32 FMA per output and block, as many VALU
// cycles as a 32-block's MFMAs take (4 FMAs of 4 cycles per v_mfma_f32_16x16x32_f16 of 16), plus
// the unpacking of the weights.  So the VALU is the busiest pipe and everything else has to stay
// out of its way.  The kernel this one replaced dequantised a step's weights into LDS for all its
// wavefronts (one barrier per 64 k, 190 KB of LDS traffic per 64-k step and CU, LDS round trips
// between unpacking and use); here only A goes through LDS (half the operand reads), a barrier
// comes once per 128 k, and the wavefronts of a SIMD drift apart between barriers, so that one's
// FMAs run under the other's MFMAs.
//   Measured, M = 2048, int4 block 32 with zero points, qkv / o / gate_up / down of the
//   Phi-3.5-mini layer: 224 / 72 / 302 / 177 us before, 136 / 57 / 248 / 136 us (803 TFLOP/s)
//   on the MFMA-native strip copy and 147 / 61 / 263 / 146 us on ORT's layout.
//
// Work split.  A workgroup of NW wavefronts, side by side along N, owns 16 MT rows; wavefront w
// owns 16 S columns of all of them (S strips).  K is walked in quads of 128.  Workgroup ids are
// mapped to tiles XCD by XCD (the eight XCDs take consecutive ids in turn; each gets one
// contiguous run of tiles, so a band of A stays in that XCD's L2).
//
// Data movement.  A: one quad ahead into one of two LDS stages with the LDS DMA (buffer loads of
// 16 bytes per lane); a row's 256 bytes are 16 slots of 16 bytes, slot s of row r stored at
// s ^ (r & 15), so the DMA reads whole lines and an operand read (16 rows, one slot each) is free
// of bank conflicts.  B: per strip and quad one 16-byte (8-bit: two) load per lane, one quad
// ahead; lane (n, g) takes chunk g of column n and the 4 x 4 dword transpose across the lane rows
// gives it the MFMA operand dwords, which the strip copy stores directly.  Scales and zero points:
// one load each per strip and pair of quads.  (Loaded quad by quad, two scattered loads each, they
// alone took 1,200-2,000 of a quad's 5,000-6,000 cycles: a load whose lanes touch 16 lines holds
// the wavefront far longer than its bytes are worth.)  Buffer loads keep the addresses to one
// 32-bit register each and make reads past the end of a tensor (the half quad of K % 128 == 64)
// return zeros.
//
// Arithmetic.  Each 16 x 16 tile's partial over one quant block is accumulated by MFMAs over the
// exact (q - zp) operands in fp32 (fp16 a x integer q - zp is exact in fp32) -- the reference
// kernel's per-block fp32 partial (rust/shaders/glsl/templates/q_gemv.comp:571-579) -- and added
// to the tile's accumulator scaled by the block's scale, while the next tile's MFMAs run.
#pragma once

#include <algorithm>
#include <type_traits>

#include "mnb_common.hpp"
#include "mnb_launch.hpp"

namespace mnb {

namespace {

typedef __attribute__((address_space(3))) void* lds_void_ptr;

// What a launch does: one dense problem; the expert-grouped problems of a mixture of experts; the
// same with SwiGLU applied to interleaved (gate, linear) columns as they are stored.
enum : int { kDense = 0, kGrouped = 1, kGroupedSwiglu = 2 };

// The expert-grouped launch: expert e's rows are offsets[e] .. offsets[e + 1] - 1 of Y, each
// multiplying row row_index[r] of A (row r itself without an index).
struct DirectGroups {
    const int32_t* offsets;      // [experts + 1]
    const int32_t* row_index;    // or null
    const f16* bias;             // SwiGLU: [experts][N] or null
    int experts;
    float alpha, beta, limit;
    int has_limit;
};

template <int BM>
__device__ __forceinline__ int group_tiles_of(const DirectGroups& g, int e) {
    return e < g.experts ? (g.offsets[e + 1] - g.offsets[e] + BM - 1) / BM : 0;
}

// Row tiles of all experts: ceil(rows / BM) each.
template <int BM>
__device__ __forceinline__ int group_row_tiles(const DirectGroups& g, int lane) {
    int n = 0;
    for (int e = lane; e < g.experts; e += 64) n += group_tiles_of<BM>(g, e);
    for (int d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d);
    return __builtin_amdgcn_readfirstlane(n);
}

// The expert that row tile `tile` belongs to (tile < group_row_tiles), the tile's first row and
// the end of the expert's rows: 64 experts at a time, their tile counts summed along the lanes.
template <int BM>
__device__ __forceinline__ void group_tile(const DirectGroups& g, int tile, int lane, int* expert,
                                           int* row0, int* row_end) {
    int e0 = 0, seen = 0;
    for (;; e0 += 64) {
        int sum = group_tiles_of<BM>(g, e0 + lane);
        const int own = sum;
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(sum, d);
            if (lane >= d) sum += v;
        }
        const uint64_t past = __ballot(seen + sum > tile);
        if (past || e0 + 64 >= g.experts) {
            const int l = past ? __builtin_ctzll(past) : 63;
            *expert = __builtin_amdgcn_readfirstlane(min(e0 + l, g.experts - 1));
            const int before = __builtin_amdgcn_readfirstlane(__shfl(seen + sum - own, l));
            *row0 = __builtin_amdgcn_readfirstlane(g.offsets[*expert]) + (tile - before) * BM;
            *row_end = __builtin_amdgcn_readfirstlane(g.offsets[*expert + 1]);
            return;
        }
        seen += __shfl(sum, 63);
    }
}

// Buffer descriptor over `bytes` bytes (loads past them return zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                             __builtin_amdgcn_readfirstlane((int)bytes), 0x00027000);
}
__device__ __forceinline__ u32x4 buffer_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

__device__ __forceinline__ void wg_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Unaligned loads of W bytes (global loads take any byte address).
template <class T>
__device__ __forceinline__ T load_any(const void* p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

// Block scales and zero points of a pair of quads (from an even one) for S strips: a column's
// 2 BPQ scales and zero points are consecutive bytes, read by one load each (scattered loads cost
// the wavefront far more than their bytes).  A pair that runs past the column's end is read block
// by block.
template <int BITS, int BS, bool HAS_ZP, int S>
struct ScalePair {
    static constexpr int NSC = 2 * 128 / BS;             // 8, 4 or 2 blocks
    uint32_t sc[S][NSC / 2];
    uint32_t z[S][BITS == 8 ? 2 : 1];

    // s_off, z_off: byte offset of each strip's column; b: the pair's first block
    __device__ __forceinline__ void load(const f16* Sc, const uint8_t* Z, const uint32_t (&s_off)[S],
                                         const uint32_t (&z_off)[S], int b, int bpc, int zpb) {
        if (b + NSC <= bpc) {
#pragma unroll
            for (int t = 0; t < S; ++t) {
                const uint8_t* sp = reinterpret_cast<const uint8_t*>(Sc) + (int64_t)b * 2 + s_off[t];
                if constexpr (NSC == 8) {
                    const u32x4 v = load_any<u32x4>(sp);
                    sc[t][0] = v.x;
                    sc[t][1] = v.y;
                    sc[t][NSC / 2 - 2] = v.z;
                    sc[t][NSC / 2 - 1] = v.w;
                } else if constexpr (NSC == 4) {
                    const u32x2 v = load_any<u32x2>(sp);
                    sc[t][0] = v.x;
                    sc[t][1] = v.y;
                } else {
                    sc[t][0] = load_any<uint32_t>(sp);
                }
                if constexpr (HAS_ZP) {
                    const uint8_t* zp = Z + (BITS == 8 ? b : b >> 1) + z_off[t];
                    constexpr int ZB = NSC * BITS / 8;   // 1 to 8 bytes
                    if constexpr (ZB == 8) {
                        const u32x2 v = load_any<u32x2>(zp);
                        z[t][0] = v.x;
                        z[t][BITS == 8] = v.y;
                    } else if constexpr (ZB == 4) {
                        z[t][0] = load_any<uint32_t>(zp);
                    } else if constexpr (ZB == 2) {
                        z[t][0] = load_any<uint16_t>(zp);
                    } else {
                        z[t][0] = *zp;
                    }
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < S; ++t) {
                const uint16_t* sp = reinterpret_cast<const uint16_t*>(
                    reinterpret_cast<const uint8_t*>(Sc) + s_off[t]);
#pragma unroll
                for (uint32_t& v : z[t]) v = 0;
#pragma unroll
                for (int i = 0; i < NSC; i += 2) {
                    sc[t][i / 2] = sp[min(b + i, bpc - 1)] |
                                   ((uint32_t)sp[min(b + i + 1, bpc - 1)] << 16);
                    if constexpr (HAS_ZP && BITS == 8) {
                        z[t][i / 4] |= ((uint32_t)Z[z_off[t] + min(b + i, zpb - 1)] |
                                        (uint32_t)Z[z_off[t] + min(b + i + 1, zpb - 1)] << 8)
                                       << (8 * (i & 3));
                    } else if constexpr (HAS_ZP) {
                        z[t][0] |= (uint32_t)Z[z_off[t] + min((b + i) >> 1, zpb - 1)] << (4 * i);
                    }
                }
            }
        }
    }
    // scale and zero point of block bi of the pair (a compile-time constant)
    __device__ __forceinline__ float scale(int t, int bi) const {
        const uint32_t w = sc[t][bi >> 1];
        return (float)__builtin_bit_cast(f16, (uint16_t)(bi & 1 ? w >> 16 : w & 0xFFFFu));
    }
    __device__ __forceinline__ uint32_t zero(int t, int bi) const {
        if constexpr (!HAS_ZP) return 1u << (BITS - 1);
        return __builtin_amdgcn_ubfe(z[t][BITS == 8 ? bi >> 2 : 0],
                                     BITS == 8 ? 8 * (bi & 3) : 4 * bi, BITS);
    }
};

}  // namespace

// MT: 16-row tiles per workgroup; S: 16-column strips per wavefront; NW: wavefronts per workgroup,
// side by side along N; NATIVE: B is the strip copy.
template <int BITS, int BS, bool HAS_ZP, int MT, int S, int NW, bool NATIVE,
          int MODE>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_direct(const f16* __restrict__ A, const uint8_t* __restrict__ B, const f16* __restrict__ Sc,
            const uint8_t* __restrict__ Z, f16* __restrict__ Y, int M, int N, int K, int tiles_m,
            int tiles_n, int ksplit, float* __restrict__ part,
            uint32_t a_bytes, DirectGroups grp) {
    static_assert(BITS == 4 || (BITS == 8 && !NATIVE), "form");
    static_assert(MODE == kDense || (BITS == 4 && !HAS_ZP), "expert weights are symmetric int4");
    constexpr int CPB = BS / 32;                         // 32-k chunks per block
    constexpr int BPQ = 4 / CPB;                         // blocks per quad
    constexpr int kBM = 16 * MT;
    constexpr int kStage = kBM * 256;
    constexpr int AI = MT * 4 / NW;                      // A loads per wavefront and quad
    constexpr int WPL = BITS / 4;                        // 16-byte weight loads per strip and quad
    static_assert(AI % 4 == 0, "the A swizzle repeats every 16 rows");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 15;
    const int g = lane >> 4;

    // Grouped: the row tiles are those of the experts in order, as many as their row counts (known
    // on the device only) need; every wavefront counts them from the offsets.
    if constexpr (MODE != kDense) tiles_m = group_row_tiles<kBM>(grp, lane);
    const int V = tiles_m * tiles_n * ksplit;
    const int per_xcd = (V + 7) >> 3;
    if ((int)(blockIdx.x >> 3) >= per_xcd) return;
    const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= V) return;                               // whole workgroups, before any barrier
    const int tile = item / ksplit;
    const int split = item - tile * ksplit;
    const int tile_m = tile / tiles_n;
    const int tile_n = tile - tile_m * tiles_n;
    int m0 = tile_m * kBM;
    const int bpc = K / BS;
    const int zpb = BITS == 8 ? bpc : (bpc + 1) >> 1;
    const int cb = K * BITS / 8;                         // bytes per column of B
    const int strips = (N + 15) >> 4;
    const int KQ = (K + 127) >> 7;
    int expert = 0;
    if constexpr (MODE != kDense) {
        // M: the end of the expert's rows; B, Sc: its weights
        group_tile<kBM>(grp, tile_m, lane, &expert, &m0, &M);
        B += NATIVE ? (int64_t)expert * strips * KQ * 1024 : (int64_t)expert * N * cb;
        Sc += (int64_t)expert * N * bpc;
    }
    const int strip0 = (tile_n * NW + wave) * S;
    const bool active = strip0 < strips;                 // else: only its share of the A loads
    const int per_split = ((KQ + ksplit - 1) / ksplit + 1) & ~1;   // pairs of quads
    const int q0 = split * per_split;
    const int q1 = min(KQ, q0 + per_split);

    // A: instruction j of the wavefront lands 4 rows x 256 bytes
    uint32_t a_off[AI];
    const int a_slot = lane & 15;
#pragma unroll
    for (int j = 0; j < AI; ++j) {
        const int row = 4 * (AI * wave + j) + (lane >> 4);
        int gm = m0 + row;
        gm = gm < M ? gm : M - 1;                        // clamped rows are never stored
        if constexpr (MODE != kDense) {
            if (grp.row_index) gm = grp.row_index[gm];
        }
        a_off[j] = (uint32_t)(((int64_t)gm * K + 8 * (a_slot ^ (row & 15))) * 2);
    }
    const auto ra = buffer_of(A, a_bytes);
    auto issue_a = [&](int q, int rows) {                // the wavefronts whose rows are needed
        if (4 * AI * wave >= rows) return;
        uint8_t* dst = smem + (q & 1) * kStage + wave * AI * 1024;
#pragma unroll
        for (int j = 0; j < AI; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_ptr)(dst + j * 1024), 16,
                                                     (int)a_off[j],
                                                     __builtin_amdgcn_readfirstlane(256 * q), 0, 0);
    };

    // B: per strip this lane's column, 16 (8-bit: 32) bytes per quad
    uint32_t b_off[S], s_off[S], z_off[S];
#pragma unroll
    for (int t = 0; t < S; ++t) {
        const int col = min(16 * (strip0 + t) + nl, N - 1);
        if constexpr (NATIVE)
            b_off[t] = (uint32_t)((int64_t)min(strip0 + t, strips - 1) * KQ * 1024 + 64 * nl + 16 * g);
        else
            b_off[t] = (uint32_t)((int64_t)col * cb + 16 * WPL * g);
        s_off[t] = (uint32_t)(col * bpc * 2);
        z_off[t] = (uint32_t)(col * zpb);
    }
    const auto rb = buffer_of(B, (uint32_t)(NATIVE ? (int64_t)strips * KQ * 1024 : (int64_t)N * cb));
    auto load_w = [&](u32x4 (&w)[S][WPL], int q) {
        const int so = __builtin_amdgcn_readfirstlane(q * (NATIVE ? 1024 : 64 * WPL));
#pragma unroll
        for (int t = 0; t < S; ++t)
#pragma unroll
            for (int h = 0; h < WPL; ++h) w[t][h] = buffer_load16(rb, b_off[t] + 16 * h, (uint32_t)so);
    };
    using Pair = ScalePair<BITS, BS, HAS_ZP, S>;

    // The K loop and the stores over the first MV row tiles.
    auto body = [&](auto mt_c) {
        constexpr int MV = decltype(mt_c)::value;
        f32x4 acc[MV][S];
#pragma unroll
        for (int i = 0; i < MV; ++i)
#pragma unroll
            for (int t = 0; t < S; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

        // the lane part of the A operand reads: row 16 i + nl, chunk c, 16-byte slot 4 c + g
        int a_lane[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) a_lane[c] = nl * 256 + (((4 * c + g) ^ nl) << 4);

        // half: which quad of the pair
        auto compute = [&](const u32x4 (&rw)[S][WPL], const Pair& r, int q, auto half_c) {
            constexpr int half = decltype(half_c)::value;
            const uint8_t* base = smem + (q & 1) * kStage;
            // the operand dwords of each chunk: dword g of the chunk (8-bit: dwords 2g and 2g + 1)
            uint32_t wv[S][WPL][4];
#pragma unroll
            for (int t = 0; t < S; ++t) {
                if constexpr (BITS == 4) {
                    wv[t][0][0] = rw[t][0].x;
                    wv[t][0][1] = rw[t][0].y;
                    wv[t][0][2] = rw[t][0].z;
                    wv[t][0][3] = rw[t][0].w;
                } else {
                    wv[t][0][0] = rw[t][0].x;
                    wv[t][WPL - 1][0] = rw[t][0].y;
                    wv[t][0][1] = rw[t][0].z;
                    wv[t][WPL - 1][1] = rw[t][0].w;
                    wv[t][0][2] = rw[t][WPL - 1].x;
                    wv[t][WPL - 1][2] = rw[t][WPL - 1].y;
                    wv[t][0][3] = rw[t][WPL - 1].z;
                    wv[t][WPL - 1][3] = rw[t][WPL - 1].w;
                }
                if constexpr (!NATIVE) {
#pragma unroll
                    for (int h = 0; h < WPL; ++h)
                        transpose_rows(wv[t][h][0], wv[t][h][1], wv[t][h][2], wv[t][h][3]);
                }
            }
            const int blocks = min(BPQ, ((K >> 5) - 4 * q) / CPB);
            constexpr int AH = 3 < MV ? 3 : MV;                            // operand reads in flight
            f16x8 a[AH][CPB];
            auto read_a = [&](int f) {                       // f = block * MV + row tile
#pragma unroll
                for (int cc = 0; cc < CPB; ++cc)
                    a[f % AH][cc] = *reinterpret_cast<const f16x8*>(
                        base + a_lane[(f / MV) * CPB + cc] + 4096 * (f % MV));
            };
#pragma unroll
            for (int f = 0; f < AH; ++f) read_a(f);
            f32x4 p[2][S];
            float psc[S];
#pragma unroll
            for (int t = 0; t < S; ++t) psc[t] = 0.f;
            auto retire = [&](int f, int t) {                // tile f's partial of strip t, scaled
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[f % MV][t][e] = __builtin_fmaf(p[f & 1][t][e], psc[t], acc[f % MV][t][e]);
            };
#pragma unroll
            for (int bq = 0; bq < BPQ; ++bq) {
                if (bq >= blocks) break;                     // uniform: the missing half of a quad
                f16x8 bop[S][CPB];
                float sc[S];
#pragma unroll
                for (int t = 0; t < S; ++t) {
                    const int bi = half * BPQ + bq;          // block of the pair
                    sc[t] = r.scale(t, bi);
                    asm volatile("" : "+v"(sc[t]));
                    const uint32_t z = r.zero(t, bi);
#pragma unroll
                    for (int cc = 0; cc < CPB; ++cc) {
                        const uint32_t w = wv[t][0][bq * CPB + cc];
                        if constexpr (BITS == 8) {
                            const uint32_t w1 = wv[t][WPL - 1][bq * CPB + cc];
                            const f16x2 zo = as_h2(0xE400E400u + z * 0x10001u);   // -(1024 + z) twice
                            bop[t][cc].s01 = byte_pair_lo(w, zo);
                            bop[t][cc].s23 = byte_pair_hi(w, zo);
                            bop[t][cc].s45 = byte_pair_lo(w1, zo);
                            bop[t][cc].s67 = byte_pair_hi(w1, zo);
                        } else if constexpr (NATIVE) {
                            bop[t][cc] = native_pairs(w, as_h2(0xE400E400u + z * 0x10001u),
                                                      as_h2(0xD400D400u + z * 0x100010u));
                        } else {
                            const f16x2 zo = zoff4((int)z);
                            bop[t][cc].s01 = nib_pair<0>(w, zo);
                            bop[t][cc].s23 = nib_pair<1>(w, zo);
                            bop[t][cc].s45 = nib_pair<2>(w, zo);
                            bop[t][cc].s67 = nib_pair<3>(w, zo);
                        }
                    }
                }
#pragma unroll
                for (int i = 0; i < MV; ++i) {
                    const int f = bq * MV + i;
#pragma unroll
                    for (int t = 0; t < S; ++t) {
                        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int cc = 0; cc < CPB; ++cc)
                            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[f % AH][cc], bop[t][cc], c, 0, 0, 0);
                        p[f & 1][t] = c;
                        if (f > 0) retire(f - 1, t);
                        if (i == 0) psc[t] = sc[t];
                        if (t == S - 1 && f + AH < BPQ * MV) read_a(f + AH);
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < S; ++t) retire(BPQ * MV - 1, t);
        };

        // Quads in pairs from an even one: (A, w) one quad ahead, a pair's scales one pair ahead.
        u32x4 w0[S][WPL], w1[S][WPL];
        Pair p0, p1;
        auto step = [&](int q, u32x4 (&now)[S][WPL], u32x4 (&next)[S][WPL], const Pair& p,
                        Pair& pn, auto half) {
            __builtin_amdgcn_s_waitcnt(0x7 << 4);            // vmcnt(0) lgkmcnt(0)
            wg_barrier();
            if (q + 1 < q1) {
                issue_a(q + 1, 16 * MV);
                load_w(next, q + 1);
                if constexpr (decltype(half)::value == 0) {
                    if (q + 2 < q1) pn.load(Sc, Z, s_off, z_off, (q + 2) * BPQ, bpc, zpb);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (active) compute(now, p, q, half);
        };
        using H0 = std::integral_constant<int, 0>;
        using H1 = std::integral_constant<int, 1>;
        issue_a(q0, 16 * MV);
        load_w(w0, q0);
        p0.load(Sc, Z, s_off, z_off, q0 * BPQ, bpc, zpb);
        for (int q = q0; q < q1; q += 4) {
            step(q, w0, w1, p0, p1, H0{});
            if (q + 1 >= q1) break;
            step(q + 1, w1, w0, p0, p1, H1{});
            if (q + 2 >= q1) break;
            step(q + 2, w0, w1, p1, p0, H0{});
            if (q + 3 >= q1) break;
            step(q + 3, w1, w0, p1, p0, H1{});
        }
        if (!active) return;

        if constexpr (MODE == kGroupedSwiglu) {
            // Columns 2i, 2i + 1 are neighbouring lanes.  Of each pair of rows the even lane takes
            // the first and the odd lane the second: it hands over its own half of the other row.
            const bool odd = lane & 1;
#pragma unroll
            for (int t = 0; t < S; ++t) {
                const int col = 16 * (strip0 + t) + (nl & ~1);
                float bg = 0.f, bl = 0.f;
                if (grp.bias && col < N) {
                    const f16x2 b = *reinterpret_cast<const f16x2*>(grp.bias + (int64_t)expert * N + col);
                    bg = (float)b.x;
                    bl = (float)b.y;
                }
#pragma unroll
                for (int i = 0; i < MV; ++i)
#pragma unroll
                    for (int e = 0; e < 4; e += 2) {
                        const float own = odd ? acc[i][t][e + 1] : acc[i][t][e];
                        const float got = dpp_f<0xB1>(odd ? acc[i][t][e] : acc[i][t][e + 1]);
                        // h is rounded to fp16 before its bias, as where h is stored
                        float gt = (float)(f16)(odd ? got : own) + bg;
                        float lt = (float)(f16)(odd ? own : got) + bl;
                        if (grp.has_limit) {
                            gt = fminf(gt, grp.limit);
                            lt = fminf(fmaxf(lt, -grp.limit), grp.limit);
                        }
                        const float a = gt / (1.f + expf(-grp.alpha * gt)) * (lt + grp.beta);
                        const int row = m0 + 16 * i + 4 * g + e + (odd ? 1 : 0);
                        if (row < M && col < N) Y[(int64_t)row * (N >> 1) + (col >> 1)] = (f16)a;
                    }
            }
            return;
        }
        float* const pbase = part ? part + (int64_t)split * M * N : nullptr;
#pragma unroll
        for (int i = 0; i < MV; ++i) {
#pragma unroll
            for (int t = 0; t < S; ++t) {
                const int col = 16 * (strip0 + t) + nl;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int row = m0 + 16 * i + 4 * g + e;
                    if (row < M && col < N) {
                        if (MODE == kDense && pbase) pbase[(int64_t)row * N + col] = acc[i][t][e];
                        else Y[(int64_t)row * N + col] = (f16)acc[i][t][e];
                    }
                }
            }
        }
    };
    if constexpr (MODE == kDense) {
        body(std::integral_constant<int, MT>{});
    } else {
        // experts leave tiles part full: only the quarters of the tile that have rows
        if (M - m0 > kBM / 2) body(std::integral_constant<int, MT>{});
        else if (M - m0 > kBM / 4) body(std::integral_constant<int, MT / 2>{});
        else body(std::integral_constant<int, MT / 4>{});
    }
}

// The tile of each GemmTile: 16-row tiles, strips per wavefront, wavefronts.
template <int BITS, int BS, int TILE>
struct DirectTile {
    static constexpr int MT = TILE == kTile64x128 ? 4 : 8;
    static constexpr int S = TILE == kTile128x192 && BITS == 4 && BS == 32 ? 3 : 2;
    static constexpr int NW = TILE == kTile128x256 ? 8 : 4;
};

template <int BITS, int BS, bool HAS_ZP, int TILE, bool NATIVE>
hipError_t direct_go(const GemmConfig& c, const void* a, const uint8_t* b, const void* s,
                     const uint8_t* z, void* y, int64_t m, int64_t n, int64_t k, float* part,
                     hipStream_t st) {
    using T = DirectTile<BITS, BS, TILE>;
    if (c.bm != 16 * T::MT || c.bn != 16 * T::S * T::NW) return hipErrorInvalidValue;
    auto kern = gemm_direct<BITS, BS, HAS_ZP, T::MT, T::S, T::NW, NATIVE, kDense>;
    constexpr int lds = 2 * 16 * T::MT * 256;
    const int ks = part ? c.ksplit : 1;
    const int64_t items = c.tiles_m * c.tiles_n * ks;
    const dim3 grid((unsigned)(8 * ((items + 7) / 8)), 1, 1);
    hipLaunchKernelGGL(kern, grid, dim3(64 * T::NW), lds, st, static_cast<const f16*>(a), b,
                       static_cast<const f16*>(s), z, static_cast<f16*>(y), (int)m, (int)n,
                       (int)k, (int)c.tiles_m, (int)c.tiles_n, ks, ks > 1 ? part : nullptr,
                       (uint32_t)(m * k * 2), DirectGroups{});
    if (ks > 1) return launch_splitk_sum(part, y, m * n, ks, st);
    return hipGetLastError();
}

template <int BITS, int BS, bool NATIVE>
hipError_t direct_tile(const GemmConfig& c, const void* a, const uint8_t* b, const void* s,
                       const uint8_t* z, void* y, int64_t m, int64_t n, int64_t k, float* part,
                       hipStream_t st) {
#define MNB_GD(T_)                                                                              \
    case T_:                                                                                    \
        return z ? direct_go<BITS, BS, true, T_, NATIVE>(c, a, b, s, z, y, m, n, k, part, st)   \
                 : direct_go<BITS, BS, false, T_, NATIVE>(c, a, b, s, z, y, m, n, k, part, st)
    switch (c.tile) {
        MNB_GD(kTile128x256);
        MNB_GD(kTile128x192);
        MNB_GD(kTile64x128);
        default: return hipErrorInvalidValue;
    }
#undef MNB_GD
}

template <int BITS, bool NATIVE>
hipError_t direct_bs(int bs, const GemmConfig& c, const void* a, const uint8_t* b, const void* s,
                     const uint8_t* z, void* y, int64_t m, int64_t n, int64_t k, float* part,
                     hipStream_t st) {
    switch (bs) {
        case 32: return direct_tile<BITS, 32, NATIVE>(c, a, b, s, z, y, m, n, k, part, st);
        case 64: return direct_tile<BITS, 64, NATIVE>(c, a, b, s, z, y, m, n, k, part, st);
        case 128: return direct_tile<BITS, 128, NATIVE>(c, a, b, s, z, y, m, n, k, part, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mnb
