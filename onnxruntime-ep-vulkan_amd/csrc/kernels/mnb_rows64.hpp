// MatMulNBits for 17 to 64 fp16 rows (a large decode batch, drafted tokens) on gfx950: int4
// weights, blocks of 32, 64 or 128, without any workspace.
//
// What bounds it.  The weights are read once and would stream in 3-6 us per node, but every
// workgroup needs all of A (up to 1 MB at K = 8192), and without a workspace the sum over K has to
// stay inside a workgroup.  So a CU's share of the time is the L2 -> LDS copy of A (64 bytes per
// clock) plus, per strip, the unpacking and the per-block rescale of its outputs.
//
// Work split.  A workgroup of eight wavefronts owns S strips of 16 columns and all 16 MT rows;
// wavefront w takes the w-th of eight contiguous runs of quads (128 k) of K, on its own from the
// first load to the final sum: no barrier inside the loop, so the two wavefronts of a SIMD cover
// each other's waits.  S makes the workgroups fit the 256 CUs in as few rounds as pay (see
// rows64_geometry).  The eight partial tiles are added in LDS in wavefront order.
//
// Data movement.  A by LDS DMA into the wavefront's two stages of 64 k (8 rows x 128 bytes per
// instruction: whole lines; 16-byte slot s of row r at s ^ (r & 7), so operand reads are free of
// bank conflicts), one stage ahead; weights one quad ahead straight into registers (the strip
// copy, or ORT's layout and the 4 x 4 dword transpose); scales and zero points of a pair of quads
// by one load each.  Arithmetic as in mnb_gemm_direct.hpp: exact (q - z) operands, each block's
// fp32 partial scaled once.
#pragma once

#include <algorithm>
#include <type_traits>

#include "mnb_common.hpp"
#include "mnb_gemm_direct.hpp"
#include "mnb_launch.hpp"

namespace mnb {

namespace {

constexpr int kR64Waves = 8;

template <int BS, bool HAS_ZP, int MT, int S, bool NATIVE>
__global__ void __launch_bounds__(64 * kR64Waves) __attribute__((amdgpu_waves_per_eu(2, 2)))
rows64(const f16* __restrict__ A, const uint8_t* __restrict__ B, const f16* __restrict__ Sc,
       const uint8_t* __restrict__ Z, f16* __restrict__ Y, int M, int N, int K) {
    constexpr int CPB = BS / 32;                         // 32-k chunks per block
    constexpr int BPQ = 4 / CPB;                         // blocks per quad
    constexpr int kStage = 16 * MT * 128;                // 64 k of the rows
    constexpr int AI = 2 * MT;                           // DMA instructions per stage
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nl = lane & 15;
    const int g = lane >> 4;
    const int bpc = K / BS;
    const int zpb = (bpc + 1) >> 1;
    const int strips = (N + 15) >> 4;
    const int KQ = (K + 127) >> 7;
    const int strip0 = blockIdx.x * S;
    // contiguous runs of pairs of quads (a run starts on an even quad)
    const int pairs = (KQ + 1) >> 1;
    const int q0 = 2 * (wave * pairs / kR64Waves);
    const int q1 = min(KQ, 2 * ((wave + 1) * pairs / kR64Waves));

    uint8_t* const slot = smem + wave * 2 * kStage;
    const auto ra = buffer_of(A, (uint32_t)((int64_t)M * K * 2));
    const auto rb = buffer_of(B, (uint32_t)(NATIVE ? (int64_t)strips * KQ * 1024 : (int64_t)N * (K / 2)));
    uint32_t a_off[AI];
#pragma unroll
    for (int j = 0; j < AI; ++j) {
        const int row = 8 * j + (lane >> 3);
        const int gm = row < M ? row : M - 1;            // clamped rows are never stored
        a_off[j] = (uint32_t)(((int64_t)gm * K + 8 * ((lane & 7) ^ (row & 7))) * 2);
    }
    auto issue_a = [&](int h) {                          // h: 64-k stage
#pragma unroll
        for (int j = 0; j < AI; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                ra, (lds_void_ptr)(slot + (h & 1) * kStage + j * 1024), 16, (int)a_off[j],
                __builtin_amdgcn_readfirstlane(128 * h), 0, 0);
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
        for (int t = 0; t < S; ++t)                      // read once: past the caches (nt)
            w[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 rb, (int)b_off[t], so, 2));
    };
    using Pair = ScalePair<4, BS, HAS_ZP, S>;

    f32x4 acc[MT][S];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < S; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the lane part of the A operand reads: row 16 i + nl, chunk c of the stage, slot 4 c + g
    int a_lane[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) a_lane[c] = nl * 128 + (((4 * c + g) ^ (nl & 7)) << 4);

    // One 64-k stage: chunks 2 hq and 2 hq + 1 of the quad.  Partials of blocks of 64 and 32 end
    // inside it; those of a 128 block carry over from the quad's first half in `carry`.
    f32x4 carry[CPB == 4 ? MT : 1][CPB == 4 ? S : 1];
    auto compute = [&](const u32x4 (&rw)[S], const Pair& r, int q, auto half_c, auto hq_c) {
        constexpr int half = decltype(half_c)::value;    // quad of the pair
        constexpr int hq = decltype(hq_c)::value;        // half of the quad
        const uint8_t* base = slot + hq * kStage;        // 2 q + hq: hq is its parity
        f16x8 bop[S][2];
        float sc[S][2];
#pragma unroll
        for (int t = 0; t < S; ++t) {
            uint32_t v[4] = {rw[t].x, rw[t].y, rw[t].z, rw[t].w};
            if constexpr (!NATIVE) transpose_rows(v[0], v[1], v[2], v[3]);
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int bi = half * BPQ + (2 * hq + c) / CPB;   // block of the pair
                sc[t][c] = r.scale(t, bi);
                const uint32_t z = r.zero(t, bi);
                const uint32_t w = v[2 * hq + c];
                if constexpr (NATIVE) {
                    bop[t][c] = native_pairs(w, as_h2(0xE400E400u + z * 0x10001u),
                                             as_h2(0xD400D400u + z * 0x100010u));
                } else {
                    const f16x2 zo = zoff4((int)z);
                    bop[t][c].s01 = nib_pair<0>(w, zo);
                    bop[t][c].s23 = nib_pair<1>(w, zo);
                    bop[t][c].s45 = nib_pair<2>(w, zo);
                    bop[t][c].s67 = nib_pair<3>(w, zo);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            f16x8 a[2];
#pragma unroll
            for (int c = 0; c < 2; ++c)
                a[c] = *reinterpret_cast<const f16x8*>(base + a_lane[c] + 2048 * i);
#pragma unroll
            for (int t = 0; t < S; ++t) {
                f32x4 p = {0.f, 0.f, 0.f, 0.f};
                if constexpr (CPB == 4 && hq == 1) p = carry[CPB == 4 ? i : 0][CPB == 4 ? t : 0];
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c], bop[t][c], p, 0, 0, 0);
                    if (CPB == 1 || (CPB == 2 && c == 1) || (CPB == 4 && hq == 1 && c == 1)) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[i][t][e] = __builtin_fmaf(p[e], sc[t][c], acc[i][t][e]);
                        p = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                }
                if constexpr (CPB == 4 && hq == 0) carry[CPB == 4 ? i : 0][CPB == 4 ? t : 0] = p;
            }
        }
    };

    u32x4 w0[S], w1[S];
    Pair p0, p1;
    const int hq_end = 2 * KQ - ((K & 64) ? 1 : 0);      // 64-k stages of K
    const int h1 = min(2 * q1, hq_end);
    // Every stage: its A is in (all older loads are; the wavefront is alone in its slot), the
    // next stage's A and, on a quad's first half, the next quad's weights go out, then it is
    // multiplied.  The stage it overwrites was read in the previous step (lgkmcnt(0)).
    auto stage = [&](int q, u32x4 (&now)[S], u32x4 (&next)[S], const Pair& p, Pair& pn, auto half,
                     auto hq) {
        const int h = 2 * q + decltype(hq)::value;
        __builtin_amdgcn_s_waitcnt(0x7 << 4);            // vmcnt(0) lgkmcnt(0)
        asm volatile("" ::: "memory");
        if (h + 1 < h1) issue_a(h + 1);
        if constexpr (decltype(hq)::value == 0) {
            if (q + 1 < q1) load_w(next, q + 1);
            if constexpr (decltype(half)::value == 1) {
                if (q + 1 < q1) pn.load(Sc, Z, s_off, z_off, (q + 1) * BPQ, bpc, zpb);
            }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        compute(now, p, q, half, hq);
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    if (q0 < q1) {
        issue_a(2 * q0);
        load_w(w0, q0);
        p0.load(Sc, Z, s_off, z_off, q0 * BPQ, bpc, zpb);
        for (int q = q0; q < q1; q += 2) {
            stage(q, w0, w1, p0, p1, C0{}, C0{});
            if (2 * q + 1 < h1) stage(q, w0, w1, p0, p1, C0{}, C1{});
            if (q + 1 >= q1) break;
            stage(q + 1, w1, w0, p0, p1, C1{}, C0{});
            if (2 * q + 3 < h1) stage(q + 1, w1, w0, p0, p1, C1{}, C1{});
            p0 = p1;
        }
    }

    // ---- the eight partial tiles, added in wavefront order (run-to-run deterministic); the A
    // stages are free once every wavefront is here ----
    __syncthreads();
    f32x4* const red = reinterpret_cast<f32x4*>(smem);   // [wave][MT * S][64]
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int t = 0; t < S; ++t) red[(wave * MT * S + i * S + t) * 64 + lane] = acc[i][t];
    __syncthreads();
    const float* const rf = reinterpret_cast<const float*>(smem);
    for (int o = threadIdx.x; o < MT * S * 256; o += 64 * kR64Waves) {
        // output o: column on (fastest), row orow of tile ot
        const int on = o & 15, orow = (o >> 4) & 15, ot = o >> 8;
        const int src = ((ot * 64 + (orow >> 2) * 16 + on) << 2) + (orow & 3);
        float v = rf[src];
#pragma unroll
        for (int w = 1; w < kR64Waves; ++w) v += rf[w * MT * S * 256 + src];
        const int row = 16 * (ot / S) + orow;
        const int col = 16 * (strip0 + ot % S) + on;
        if (row < M && col < N) Y[(int64_t)row * N + col] = (f16)v;
    }
}

template <int BS, bool HAS_ZP, bool NATIVE>
hipError_t rows64_go(const Rows64Geom& g, const void* a, const uint8_t* b, const void* s,
                     const uint8_t* z, void* y, int64_t m, int64_t n, int64_t k, hipStream_t st) {
#define MNB_R64(MT_, S_)                                                                          \
    if (g.mt == MT_ && g.s == S_) {                                                               \
        auto kern = rows64<BS, HAS_ZP, MT_, S_, NATIVE>;                                          \
        const hipError_t e = allow_dynamic_lds(reinterpret_cast<const void*>(kern), g.lds);       \
        if (e != hipSuccess) return e;                                                            \
        hipLaunchKernelGGL(kern, dim3((unsigned)g.gx), dim3(64 * kR64Waves), g.lds, st,           \
                           static_cast<const f16*>(a), b, static_cast<const f16*>(s), z,          \
                           static_cast<f16*>(y), (int)m, (int)n, (int)k);                         \
        return hipGetLastError();                                                                 \
    }
    MNB_R64(2, 1) MNB_R64(2, 2) MNB_R64(2, 3) MNB_R64(2, 4)
    MNB_R64(3, 1) MNB_R64(3, 2) MNB_R64(3, 3) MNB_R64(3, 4)
    MNB_R64(4, 1) MNB_R64(4, 2) MNB_R64(4, 3) MNB_R64(4, 4)
#undef MNB_R64
    return hipErrorInvalidValue;
}

template <int BS>
hipError_t rows64_bs(const Rows64Geom& g, const void* a, const uint8_t* b, const uint8_t* strips,
                     const void* s, const uint8_t* z, void* y, int64_t m, int64_t n, int64_t k,
                     hipStream_t st) {
    if (strips)
        return z ? rows64_go<BS, true, true>(g, a, strips, s, z, y, m, n, k, st)
                 : rows64_go<BS, false, true>(g, a, strips, s, z, y, m, n, k, st);
    return z ? rows64_go<BS, true, false>(g, a, b, s, z, y, m, n, k, st)
             : rows64_go<BS, false, false>(g, a, b, s, z, y, m, n, k, st);
}

}  // namespace

}  // namespace mnb
