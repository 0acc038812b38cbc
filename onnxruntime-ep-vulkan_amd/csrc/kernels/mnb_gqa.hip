// com.microsoft::GroupQueryAttention, packed QKV with fused half-rotation (neox) RoPE and a KV
// cache, fp16 tensors, fp32 softmax and accumulation.
//
// Semantics follow the reference kernel (rust/shaders/glsl/gqa_f16.comp, dispatched by
// rust/src/ops/attention.rs:388-735):
//   * packed_qkv [B, S, (Nq + 2 Nkv) D]; per batch past_len = seqlens_k[b] + 1 - S (at least 0);
//     query s sits at position tok_pos = past_len + s;
//   * RoPE on Q and the new K: pairs (x[i], x[i + rd/2]), i < rd/2, rotated by the cos/sin cache
//     rows at tok_pos; dims at or past rd are copied;
//   * the new K (rotated) and V are written to present at tok_pos when tok_pos < present_len;
//     under the growing convention (present is a separate buffer) present also receives the past
//     tokens [0, past_len);
//   * each query attends to keys [0, tok_pos] of KV head h / (Nq / Nkv): keys t < past_len from
//     the past buffer, later keys from this call's own (rotated) K and V.  These are read where
//     the append put them in present (written by the launch before, at positions no launch reads
//     as past, also when present aliases past), or, for a batch row whose new tokens do not all
//     fit in present, from a copy in the workspace.
//
// Bounds the reference leaves to the caller are clamped here so that every access stays inside
// the buffers the problem describes: past_len is clamped to [0, past_stride] and the cos/sin row
// to [0, max_seq - 1].
//
// Three kernels:
//   gqa_prep     RoPE and append, 8 dims per thread: rotated Q in a per-KV-head row order (row
//                r = s * G + g) as fp16 high and low parts, and the present writes.  Bound by its
//                bytes (S = 2048, 32 + 64 heads of 96: 88 MB); one dim per thread and 64-bit
//                divisions took 80 us there, and new K and V also went to the workspace.
//   gqa_attend   flash attention on v_mfma_f32_16x16x32_f16.  A workgroup takes 16 x W query
//                rows of one (batch, KV head) and walks 64-key blocks staged in LDS (K row-major,
//                V transposed), the next block in flight in registers.  Scores are computed
//                transposed, S^T = K Q^T, so each lane holds one query's 16 scores of a block:
//                the softmax statistics stay per lane (two shuffles per block) and P^T feeds the
//                second MFMA (O^T = V^T P^T) straight from registers.  Rows of a workgroup are the
//                G query heads of every position, so one K/V block serves all of them.  Q and P
//                enter the MFMAs as fp16 high + low pairs (two MFMAs each), so scores and weights
//                keep fp32 precision as in the reference's fp32 kernel; rounding either to one
//                fp16 costs up to 6e-3 relative on outputs.
//                Long prompts are bound by the matrix cores and the softmax's VALU work about
//                equally, three wavefronts per SIMD overlapping them.  (Two query tiles per
//                wavefront halve the LDS operand reads but leave two wavefronts per SIMD: 99
//                against 91 us for 2048 tokens of 32 heads of 96.)  Few rows (W = 1, decode) are
//                bound by streaming the cache: the key range is split until about four wavefronts
//                per CU stream, each with a whole block (16 KB of K and of V at D = 128) in flight.
//   gqa_combine  merges the split partials (max, sum, unnormalised O) into attn_output.
#include <algorithm>
#include <cmath>

#include "mnb_common.hpp"
#include "mnb_launch.hpp"

namespace mnb {

namespace {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));

constexpr int kBN = 64;            // keys per block
constexpr int kVP = kBN + 8;       // transposed-V row pitch in halves (conflict-free reads)
constexpr float kMasked = -1.0e30f;   // the maximum of no scores: finite, below any real one
constexpr int kMaxSplits = 64;

struct GqaDims {
    int64_t S, R;                  // new tokens; query rows per (batch, KV head) = S * G
    int64_t past_stride, present_len, max_seq, chunk;
    int nq, nkv, G, rh, rot, row_blocks, splits, copy_past;
    int64_t work;                  // workgroups of gqa_attend
    int64_t q_elems;               // B * Nq * S * D: offset of the low halves of rotated Q
    float scale_log2;              // factor of the scores, > 0 (|scale| log2 e)
    float q_factor;                // factor of Q: the scale's sign, or all of a vanishing scale
};

__device__ __forceinline__ int64_t past_len_of(const int32_t* seqlens, int b, const GqaDims& g) {
    const int64_t p = (int64_t)seqlens[b] + 1 - g.S;
    return p < 0 ? 0 : (p > g.past_stride ? g.past_stride : p);
}

// Whether batch row b's new tokens all have their place in present (else: the workspace copy).
__device__ __forceinline__ bool new_in_present(int64_t past_len, const GqaDims& g) {
    return past_len + g.S <= g.present_len;
}

// Buffer descriptor over `bytes` bytes at a wave-uniform address (loads past them return zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const f16* p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint64_t u = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a) |
                       (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32;
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(u), 0,
                                             __builtin_amdgcn_readfirstlane((int)bytes), 0x00027000);
}
__device__ __forceinline__ u32x4 buffer_load16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)soff, 0));
}

// v - h[I], exact to fp32: one mixed FMA instead of a conversion and a subtraction.
template <int I>
__device__ __forceinline__ float minus_half(float v, f16x2 h) {
    float r;
    if constexpr (I == 0)
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(as_u32(h)), "v"(v));
    else
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
            : "=v"(r)
            : "v"(as_u32(h)), "v"(v));
    return r;
}

// LDS row of key kk within a 64-key block: the 16 keys one score MFMA reads (see gqa_attend)
// sit in 16 consecutive rows.
__device__ __forceinline__ int lds_row(int kk) {
    return (kk & ~31) | (((kk >> 2) & 1) << 4) | (((kk >> 3) & 3) << 2) | (kk & 3);
}

}  // namespace

// Thread: one chunk of 8 dims of one head of one token; blockIdx.x: token b * S + s.
// VEC: rh % 8 == 0, so a rotated chunk's partner and its cos/sin values are chunks too.
template <bool VEC>
__global__ void __launch_bounds__(256)
gqa_prep(const f16* __restrict__ qkv, const int32_t* __restrict__ seqlens,
         const f16* __restrict__ cosc, const f16* __restrict__ sinc, f16* __restrict__ qr,
         f16* __restrict__ kn, f16* __restrict__ vn, f16* pres_k, f16* pres_v, int D, GqaDims g) {
    const int cpr = D >> 3;
    const int heads = g.nq + 2 * g.nkv;
    const int i = blockIdx.y * 256 + threadIdx.x;
    if (i >= heads * cpr) return;
    const int hh = i / cpr;
    const int d0 = (i - hh * cpr) * 8;
    const int64_t tok = blockIdx.x;
    const int b = (int)(tok / g.S);
    const int64_t s = tok - b * g.S;
    const int64_t past = past_len_of(seqlens, b, g);
    const int64_t tp = past + s;
    const f16* row = qkv + (tok * heads + hh) * D;
    const f16x8 x = *reinterpret_cast<const f16x8*>(row + d0);
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (float)x[e];
    if (hh < g.nq + g.nkv && d0 < g.rot) {
        const int64_t pr = (tp < g.max_seq ? tp : g.max_seq - 1) * g.rh;
        if constexpr (VEC) {
            const bool lo = d0 < g.rh;
            const f16x8 o = *reinterpret_cast<const f16x8*>(row + (lo ? d0 + g.rh : d0 - g.rh));
            const int ri = lo ? d0 : d0 - g.rh;
            const f16x8 c = *reinterpret_cast<const f16x8*>(cosc + pr + ri);
            const f16x8 sn = *reinterpret_cast<const f16x8*>(sinc + pr + ri);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float t = (float)o[e] * (float)sn[e];
                y[e] = y[e] * (float)c[e] + (lo ? -t : t);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int d = d0 + e;
                if (d >= g.rot) break;
                const bool lo = d < g.rh;
                const int ri = lo ? d : d - g.rh;
                const float t = (float)row[lo ? d + g.rh : d - g.rh] * (float)sinc[pr + ri];
                y[e] = y[e] * (float)cosc[pr + ri] + (lo ? -t : t);
            }
        }
    }
    if (hh < g.nq) {                                     // Q: rotated, rows grouped per KV head
        const int kvh = hh / g.G;
        const int64_t r = s * g.G + (hh - kvh * g.G);
        const int64_t o = (((int64_t)b * g.nkv + kvh) * g.R + r) * D + d0;
        f16x8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; ++e) {                    // y = hi + lo to 2^-22
            const float v = y[e] * g.q_factor;
            hi[e] = (f16)v;
            lo[e] = (f16)(v - (float)hi[e]);
        }
        *reinterpret_cast<f16x8*>(qr + o) = hi;
        *reinterpret_cast<f16x8*>(qr + o + g.q_elems) = lo;
        return;
    }
    const bool is_v = hh >= g.nq + g.nkv;                // K: rotated; V: copied
    const int kvh = hh - g.nq - (is_v ? g.nkv : 0);
    f16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (f16)y[e];
    const int64_t bk = (int64_t)b * g.nkv + kvh;
    if (tp < g.present_len)
        *reinterpret_cast<f16x8*>((is_v ? pres_v : pres_k) + (bk * g.present_len + tp) * D + d0) = v;
    if (!new_in_present(past, g))
        *reinterpret_cast<f16x8*>((is_v ? vn : kn) + (bk * g.S + s) * D + d0) = v;
}

// W wavefronts of 16 query rows each.
template <int D, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W == 1 ? 1 : 2)))
gqa_attend(const f16* __restrict__ qr, const f16* __restrict__ past_k,
           const f16* __restrict__ past_v, const f16* __restrict__ kn,
           const f16* __restrict__ vn, const int32_t* __restrict__ seqlens,
           f16* __restrict__ out, f16* pres_k, f16* pres_v, float* __restrict__ part_o,
           float* __restrict__ part_ml, GqaDims g) {
    constexpr int KS = (D + 31) / 32;          // k-steps of the score MFMA
    constexpr bool TAIL = (D % 32) != 0;       // the last one half empty: zeros past D
    constexpr int DT = D / 16;                 // 16-wide d tiles of O
    constexpr int KP = D + 8;                  // K row pitch in halves
    constexpr int CPR = D / 8;                 // 16-byte chunks per key row
    constexpr int NT = 64 * W;
    constexpr int KCH = kBN * CPR;
    constexpr int KIT = (KCH + NT - 1) / NT;
    constexpr int VITEMS = (kBN / 4) * CPR;    // 4 keys x 8 dims each
    constexpr int VIT = (VITEMS + NT - 1) / NT;

    __shared__ __align__(16) f16 Ks[kBN * KP];
    __shared__ __align__(16) f16 Vt[D * kVP];

    // Work items: row blocks of one batch row and KV head share K and V, so each XCD (workgroups
    // are dealt to the 8 XCDs round-robin) gets whole heads where it can.  Within an XCD the
    // blocks go longest first (causal: the last rows see the most keys), every other 32 of them
    // (one per CU) in reverse, so that the workgroups sharing a CU add up to about the same.
    int64_t w = blockIdx.x;
    int rb, split;
    int64_t bk;
    if ((g.work & 7) == 0 && (g.work >> 3) % g.row_blocks == 0 && g.splits == 1) {
        const int n = (int)(g.work >> 3);                // items of an XCD
        const int l = (int)(w >> 3);
        const int hx = n / g.row_blocks;                 // heads of an XCD
        const int c0 = l & ~31;
        const int rank = (l >> 5) & 1 ? c0 + (min(32, n - c0) - 1 - (l - c0)) : l;
        rb = g.row_blocks - 1 - rank / hx;
        bk = (w & 7) * hx + rank % hx;
        split = 0;
    } else {
        if ((g.work & 7) == 0) w = (w & 7) * (g.work >> 3) + (w >> 3);
        rb = g.row_blocks - 1 - (int)(w % g.row_blocks); // longest rows first
        const int64_t t2 = w / g.row_blocks;
        split = (int)(t2 % g.splits);
        bk = t2 / g.splits;
    }
    const int b = (int)(bk / g.nkv);

    const int64_t past_len = past_len_of(seqlens, b, g);
    const int64_t r0 = (int64_t)rb * 16 * W;
    const int64_t r_hi = std::min<int64_t>(r0 + 16 * W, g.R);
    const int64_t key_end = past_len + (r_hi - 1) / g.G + 1;
    const int64_t k_begin = (int64_t)split * g.chunk;
    const int64_t k_stop = std::min<int64_t>(k_begin + g.chunk, key_end);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int j = lane & 15;
    const int grp = lane >> 4;
    const int64_t wr0 = r0 + 16 * wave;                  // the wavefront's first row
    const bool wave_active = wr0 < g.R;
    const int64_t r = wr0 + j;
    const bool rvalid = r < g.R;

    if (k_begin >= k_stop) {                             // no keys in this split
        if (!rvalid) return;
        const int64_t prow = ((int64_t)split * (g.work / (g.splits * g.row_blocks)) + bk) * g.R + r;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            *reinterpret_cast<f32x4*>(part_o + prow * D + 16 * dt + 4 * grp) = f32x4{0, 0, 0, 0};
        if (grp == 0) {
            part_ml[2 * prow] = kMasked;
            part_ml[2 * prow + 1] = 0.f;
        }
        return;
    }

    const int64_t rc = rvalid ? r : g.R - 1;
    const int64_t tp = past_len + rc / g.G;              // this lane's query, the wavefront's first
    const int64_t tp_lo = past_len + std::min<int64_t>(wr0, g.R - 1) / g.G;   // and last
    const int64_t tp_hi = past_len + (std::min<int64_t>(wr0 + 15, g.R - 1)) / g.G;
    // Q^T fragments (B operand of the score MFMA): query j, dims 32 ks + 8 grp .. + 7, as fp16
    // high and low parts (two MFMAs), so the scores carry the fp32 rotation of Q.
    f16x8 qf[2][KS];
#pragma unroll
    for (int hl = 0; hl < 2; ++hl) {
        const f16* qrow = qr + hl * g.q_elems + (bk * g.R + rc) * D;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            qf[hl][ks] = rvalid && (!TAIL || ks + 1 < KS || grp < 2)
                             ? *reinterpret_cast<const f16x8*>(qrow + 32 * ks + 8 * grp)
                             : f16x8{};
    }

    f32x4 oacc[DT];
    float m_run = kMasked, l_run = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

    const bool copy = g.copy_past && rb == 0;
    const f16* pk_base = past_k + bk * g.past_stride * D;
    const f16* pv_base = past_v + bk * g.past_stride * D;
    // the new tokens, indexed by key t >= past_len
    const bool in_pres = new_in_present(past_len, g);
    const f16* kn_base = in_pres ? pres_k + bk * g.present_len * D : kn + (bk * g.S - past_len) * D;
    const f16* vn_base = in_pres ? pres_v + bk * g.present_len * D : vn + (bk * g.S - past_len) * D;
    f16* prk = pres_k + bk * g.present_len * D;
    f16* prv = pres_v + bk * g.present_len * D;

    u32x4 kreg[KIT];
    u32x4 vreg[VIT][4];

    // Blocks of up to 64 keys, none across past_len (the keys' source changes there): block
    // [kb, block_end(kb)).
    auto block_end = [&](int64_t kb) {
        const int64_t stop = kb < past_len ? std::min(past_len, k_stop) : k_stop;
        return std::min<int64_t>(kb + kBN, stop);
    };
    // One block into registers.  K: 16 bytes per item, items of a key consecutive; V: 8 dims of 4
    // keys per item.  Buffer loads from the block's own (uniform) base, whose bound makes keys past
    // its end zeros.  (Picking source and bound per lane put every load behind a branch of its
    // own, and the wait for each cost 2,600 of a block's 8,400 cycles.)
    auto load = [&](int64_t kb) {
        const bool in_past = kb < past_len;
        const uint32_t bytes = (uint32_t)(block_end(kb) - kb) * (D * 2);
        const auto rk = buffer_of((in_past ? pk_base : kn_base) + kb * D, bytes);
        const auto rv = buffer_of((in_past ? pv_base : vn_base) + kb * D, bytes);
#pragma unroll
        for (int it = 0; it < KIT; ++it) kreg[it] = buffer_load16(rk, (uint32_t)(tid + NT * it) * 16, 0);
#pragma unroll
        for (int it = 0; it < VIT; ++it) {
            const int c = tid + NT * it;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                vreg[it][q] = buffer_load16(
                    rv, (uint32_t)((4 * (c & 15) + q) * D + 8 * (c >> 4)) * 2, 0);
        }
    };

    auto store = [&](int64_t kb) {
#pragma unroll
        for (int it = 0; it < KIT; ++it) {
            const int c = tid + NT * it;
            if (KCH % NT == 0 || c < KCH) {
                const int kk = c / CPR;
                *reinterpret_cast<u32x4*>(&Ks[lds_row(kk) * KP + 8 * (c % CPR)]) = kreg[it];
            }
        }
#pragma unroll
        for (int it = 0; it < VIT; ++it) {
            const int c = tid + NT * it;
            if (VITEMS % NT == 0 || c < VITEMS) {
                const int kg = c & 15;
                const int dc = c >> 4;
                const f16x8 v0 = __builtin_bit_cast(f16x8, vreg[it][0]);
                const f16x8 v1 = __builtin_bit_cast(f16x8, vreg[it][1]);
                const f16x8 v2 = __builtin_bit_cast(f16x8, vreg[it][2]);
                const f16x8 v3 = __builtin_bit_cast(f16x8, vreg[it][3]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const h4 col = {v0[e], v1[e], v2[e], v3[e]};
                    *reinterpret_cast<h4*>(&Vt[(8 * dc + e) * kVP + 4 * kg]) = col;
                }
            }
        }
        if (copy && kb < past_len) {                     // uniform: past tokens into present
            const int64_t kend = block_end(kb);
#pragma unroll
            for (int it = 0; it < KIT; ++it) {
                const int c = tid + NT * it;
                const int64_t t = kb + c / CPR;
                if (c < KCH && t < kend)
                    *reinterpret_cast<u32x4*>(prk + t * D + 8 * (c % CPR)) = kreg[it];
            }
#pragma unroll
            for (int it = 0; it < VIT; ++it) {
                const int c = tid + NT * it;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int64_t t = kb + 4 * (c & 15) + q;
                    if (c < VITEMS && t < kend)
                        *reinterpret_cast<u32x4*>(prv + t * D + 8 * (c >> 4)) = vreg[it][q];
                }
            }
        }
    };

    auto compute = [&](int64_t kb) {
        const int64_t kend = block_end(kb);
        // S^T tiles: c2 = 32-key half, a = 16-key MFMA tile.  Lane (j, grp) ends up with the
        // scores of query j and keys kb + 32 c2 + 8 grp + 4 a + i.
        f32x4 sc[2][2];
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                sc[c2][a] = f32x4{0.f, 0.f, 0.f, 0.f};
                const f16* krow = &Ks[(32 * c2 + 16 * a + j) * KP];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    f16x8 kf;
                    if constexpr (TAIL) {
                        if (ks + 1 < KS) {
                            kf = *reinterpret_cast<const f16x8*>(krow + 32 * ks + 8 * grp);
                        } else {                         // dims past D are zero in K as well
                            kf = *reinterpret_cast<const f16x8*>(krow + 32 * ks + 8 * (grp & 1));
                            kf = grp < 2 ? kf : f16x8{};
                        }
                    } else {
                        kf = *reinterpret_cast<const f16x8*>(krow + 32 * ks + 8 * grp);
                    }
#pragma unroll
                    for (int hl = 0; hl < 2; ++hl)
                        sc[c2][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            kf, qf[hl][ks], sc[c2][a], 0, 0, 0);
                }
            }
        f16x8 pb[2], pl[2];                              // P = pb + pl to 2^-22
        // uniform: the block crosses the diagonal, or is short
        if (kb + kBN - 1 > tp_lo || kend - kb < kBN) {
            // first masked key of the lane, counted from its first key of the block
            const int cut = (int)std::min<int64_t>(tp + 1 - kb, kend - kb) - 8 * grp;
#pragma unroll
            for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (32 * c2 + 4 * a + i >= cut) sc[c2][a][i] = -INFINITY;
        }
        float mloc = -INFINITY;
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int i = 0; i < 4; ++i) mloc = fmaxf(mloc, sc[c2][a][i]);
        mloc *= g.scale_log2;                            // positive: a masked score stays -inf
        mloc = fmaxf(mloc, __shfl_xor(mloc, 16));
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
        const float m_new = fmaxf(m_run, mloc);
        // most blocks after the first few raise no row's maximum: nothing to rescale
        if (__any(m_new != m_run)) {
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
        }
        float l = 0.f;
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                float p[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(
                        sc[c2][i >> 2][(i & 3) + e], g.scale_log2, -m_new));
                    l += p[e];
                }
                const f16x2 hi = {(f16)p[0], (f16)p[1]};
                const f16x2 lo = {(f16)minus_half<0>(p[0], hi), (f16)minus_half<1>(p[1], hi)};
                pb[c2][i] = hi.x;
                pb[c2][i + 1] = hi.y;
                pl[c2][i] = lo.x;
                pl[c2][i + 1] = lo.y;
            }
        l_run += l;
        // O^T += V^T P^T over keys kb + 32 c2 + 8 grp .. + 7.
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const f16x8 vf =
                    *reinterpret_cast<const f16x8*>(&Vt[(16 * dt + j) * kVP + 32 * c2 + 8 * grp]);
                oacc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pb[c2], oacc[dt], 0, 0, 0);
                oacc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl[c2], oacc[dt], 0, 0, 0);
            }
    };

    load(k_begin);
    for (int64_t kb = k_begin; kb < k_stop;) {
        const int64_t next = block_end(kb);
        if (kb != k_begin) __syncthreads();              // the previous block is consumed
        store(kb);
        __syncthreads();
        if (next < k_stop) load(next);
        if (wave_active && kb <= tp_hi) compute(kb);
        kb = next;
    }

    float l = l_run;
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (!rvalid) return;
    if (g.splits == 1) {
        const int64_t s = r / g.G;
        const int h = (int)(bk % g.nkv) * g.G + (int)(r % g.G);
        f16* o = out + (((int64_t)b * g.S + s) * g.nq + h) * D + 4 * grp;
        const float inv = 1.f / l;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const f32x4 x = oacc[dt];
            const h4 v = {(f16)(x[0] * inv), (f16)(x[1] * inv), (f16)(x[2] * inv),
                          (f16)(x[3] * inv)};
            *reinterpret_cast<h4*>(o + 16 * dt) = v;
        }
        return;
    }
    const int64_t bks = g.work / ((int64_t)g.splits * g.row_blocks);
    const int64_t prow = ((int64_t)split * bks + bk) * g.R + r;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        *reinterpret_cast<f32x4*>(part_o + prow * D + 16 * dt + 4 * grp) = oacc[dt];
    if (grp == 0) {
        part_ml[2 * prow] = m_run;
        part_ml[2 * prow + 1] = l;
    }
}

// Workgroup: one row (batch x KV head x query row).  Lane s of every wavefront holds split s's
// maximum and sum (at most 64 splits); the threads add the splits' rows, 4 dims each, in groups
// that take every (256 / (D / 4))-th split, and the groups are added through LDS in order.  (One
// thread walking all the splits of its dims took 6.7 us at 8 splits of 256 rows.)
__global__ void __launch_bounds__(256)
gqa_combine(const float* __restrict__ part_o, const float* __restrict__ part_ml,
            f16* __restrict__ out, int64_t rows, int D, GqaDims g) {
    __shared__ __align__(16) f32x4 red[256];
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int quads = D >> 2;
    const int groups = 256 / quads;                      // 4 .. 64 (D <= 256)
    const int grp = threadIdx.x / quads;
    const int q = threadIdx.x - grp * quads;
    float m = kMasked, l = 0.f;
    if (lane < g.splits) {
        m = part_ml[2 * ((int64_t)lane * rows + row)];
        l = part_ml[2 * ((int64_t)lane * rows + row) + 1];
    }
    const float top = wave_max64(m);
    const float wgt = lane < g.splits ? __builtin_amdgcn_exp2f(m - top) : 0.f;
    const float sum = group_sum(wgt * l, 64);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // every lane takes part in the shuffles; splits past the last weigh nothing
    for (int sp0 = 0; sp0 < g.splits; sp0 += groups) {
        const int sp = sp0 + grp;
        const float ws = __shfl(wgt, sp & 63);
        if (grp < groups && sp < g.splits)
            acc += ws * *reinterpret_cast<const f32x4*>(part_o + ((int64_t)sp * rows + row) * D + 4 * q);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (grp != 0) return;
    for (int k = 1; k < groups; ++k) acc += red[k * quads + q];
    const float inv = 1.f / sum;
    const int64_t bk = row / g.R;
    const int64_t r = row % g.R;
    const int b = (int)(bk / g.nkv);
    const int h = (int)(bk % g.nkv) * g.G + (int)(r % g.G);
    const int64_t s = r / g.G;
    const h4 v = {(f16)(acc[0] * inv), (f16)(acc[1] * inv), (f16)(acc[2] * inv),
                  (f16)(acc[3] * inv)};
    *reinterpret_cast<h4*>(out + (((int64_t)b * g.S + s) * g.nq + h) * D + 4 * q) = v;
}

bool gqa_supported(int head_dim) { return head_dim >= 16 && head_dim <= 256 && head_dim % 16 == 0; }

GqaPlan gqa_plan(const GqaArgs& a) {
    GqaPlan p{};
    const int64_t G = a.nq / a.nkv;
    const int64_t R = a.seq * G;
    const int64_t bk = a.batch * a.nkv;
    p.waves = R > 16 ? 4 : 1;
    const int64_t block = 16 * p.waves;
    p.row_blocks = (R + block - 1) / block;
    const int64_t base = bk * p.row_blocks;
    const int64_t t_max = a.past_stride + a.seq;        // bound on keys per query
    p.splits = 1;
    p.chunk = (t_max + kBN - 1) / kBN * kBN;
    // Keys are split until the workgroups fill the chip: about 1024 one-wavefront ones (decode),
    // 512 of four wavefronts; at least one (four wavefronts: two) 64-key blocks each.
    const int64_t fill = p.waves == 1 ? 1024 : 512;
    const int64_t least = p.waves == 1 ? kBN : 2 * kBN;
    if (base < fill && t_max > least) {
        const int64_t want = (fill + base - 1) / base;
        int64_t chunk = (t_max + want - 1) / want;
        chunk = std::max<int64_t>(least, (chunk + kBN - 1) / kBN * kBN);
        const int64_t splits = std::min<int64_t>((t_max + chunk - 1) / chunk, kMaxSplits);
        chunk = std::max<int64_t>(chunk, ((t_max + splits - 1) / splits + kBN - 1) / kBN * kBN);
        p.splits = (int)((t_max + chunk - 1) / chunk);
        p.chunk = chunk;
    }
    return p;
}

static size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t gqa_workspace_bytes(const GqaArgs& a) {
    const GqaPlan p = gqa_plan(a);
    const size_t q = (size_t)a.batch * a.nq * a.seq * a.d;
    const size_t kv = (size_t)a.batch * a.nkv * a.seq * a.d;
    size_t n = al256(q * 4) + 2 * al256(kv * 2);     // rotated Q as fp16 high and low parts
    if (p.splits > 1) n += al256((size_t)p.splits * q * 4) + al256((size_t)p.splits * (q / a.d) * 8);
    return n;
}

template <int D, int W>
static void attend_go(const GqaDims& g, const f16* qr, const void* pk, const void* pv,
                      const f16* kn, const f16* vn, const int32_t* seqlens, void* out, void* prk,
                      void* prv, float* po, float* pml, hipStream_t st) {
    hipLaunchKernelGGL((gqa_attend<D, W>), dim3((unsigned)g.work), dim3(64 * W), 0, st, qr,
                       static_cast<const f16*>(pk), static_cast<const f16*>(pv), kn, vn, seqlens,
                       static_cast<f16*>(out), static_cast<f16*>(prk), static_cast<f16*>(prv), po,
                       pml, g);
}

template <int D>
static void attend_w(const GqaPlan& p, const GqaDims& g, const f16* qr, const void* pk,
                     const void* pv, const f16* kn, const f16* vn, const int32_t* seqlens,
                     void* out, void* prk, void* prv, float* po, float* pml, hipStream_t st) {
    if (p.waves == 1)
        return attend_go<D, 1>(g, qr, pk, pv, kn, vn, seqlens, out, prk, prv, po, pml, st);
    attend_go<D, 4>(g, qr, pk, pv, kn, vn, seqlens, out, prk, prv, po, pml, st);
}

hipError_t launch_gqa(const GqaArgs& a, const void* qkv, const void* past_k, const void* past_v,
                      const int32_t* seqlens, const void* cos_cache, const void* sin_cache,
                      void* out, void* pres_k, void* pres_v, void* workspace, hipStream_t st) {
    if (!gqa_supported(a.d) || a.nkv <= 0 || a.nq % a.nkv) return hipErrorInvalidValue;
    if (a.batch == 0 || a.seq == 0) return hipSuccess;
    const GqaPlan p = gqa_plan(a);
    GqaDims g{};
    g.S = a.seq;
    g.G = a.nq / a.nkv;
    g.R = a.seq * g.G;
    g.past_stride = a.past_stride;
    g.present_len = a.present_len;
    g.max_seq = a.max_seq;
    g.chunk = p.chunk;
    g.nq = a.nq;
    g.nkv = a.nkv;
    g.rh = a.rot / 2;
    g.rot = a.rot;
    g.row_blocks = (int)p.row_blocks;
    g.splits = p.splits;
    g.copy_past = a.copy_past ? 1 : 0;
    g.work = a.batch * a.nkv * p.row_blocks * p.splits;
    // Scores are scaled as their maximum is subtracted (one FMA): the factor has to be positive.
    const float sl = a.scale * 1.4426950408889634f;
    const bool tiny = std::fabs(sl) < 1e-20f;
    g.scale_log2 = tiny ? 1.f : std::fabs(sl);
    g.q_factor = tiny ? sl : std::copysign(1.f, sl);
    g.q_elems = (int64_t)((size_t)a.batch * a.nq * a.seq * a.d);

    const size_t q = (size_t)a.batch * a.nq * a.seq * a.d;
    const size_t kv = (size_t)a.batch * a.nkv * a.seq * a.d;
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    f16* qr = reinterpret_cast<f16*>(ws);
    ws += al256(q * 4);
    f16* kn = reinterpret_cast<f16*>(ws);
    ws += al256(kv * 2);
    f16* vn = reinterpret_cast<f16*>(ws);
    ws += al256(kv * 2);
    float* po = nullptr;
    float* pml = nullptr;
    if (p.splits > 1) {
        po = reinterpret_cast<float*>(ws);
        ws += al256((size_t)p.splits * q * 4);
        pml = reinterpret_cast<float*>(ws);
    }

    const int heads = a.nq + 2 * a.nkv;
    const dim3 pgrid((unsigned)(a.batch * a.seq), (unsigned)((heads * (a.d / 8) + 255) / 256));
    auto prep = [&](auto kern) {
        hipLaunchKernelGGL(kern, pgrid, dim3(256), 0, st, static_cast<const f16*>(qkv), seqlens,
                           static_cast<const f16*>(cos_cache), static_cast<const f16*>(sin_cache),
                           qr, kn, vn, static_cast<f16*>(pres_k), static_cast<f16*>(pres_v), a.d,
                           g);
    };
    // chunked cos/sin loads also need their bases on 16 bytes
    const bool vec = g.rh % 8 == 0 && reinterpret_cast<uintptr_t>(cos_cache) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(sin_cache) % 16 == 0;
    if (vec) prep(gqa_prep<true>);
    else prep(gqa_prep<false>);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;

    switch (a.d) {
#define MNB_GQA_D(DD) \
    case DD: attend_w<DD>(p, g, qr, past_k, past_v, kn, vn, seqlens, out, pres_k, pres_v, po, pml, st); break;
        MNB_GQA_D(16) MNB_GQA_D(32) MNB_GQA_D(48) MNB_GQA_D(64) MNB_GQA_D(80) MNB_GQA_D(96)
        MNB_GQA_D(112) MNB_GQA_D(128) MNB_GQA_D(144) MNB_GQA_D(160) MNB_GQA_D(176)
        MNB_GQA_D(192) MNB_GQA_D(208) MNB_GQA_D(224) MNB_GQA_D(240) MNB_GQA_D(256)
#undef MNB_GQA_D
        default: return hipErrorInvalidValue;
    }
    e = hipGetLastError();
    if (e != hipSuccess || p.splits == 1) return e;
    const int64_t rows = a.batch * a.nkv * g.R;
    hipLaunchKernelGGL(gqa_combine, dim3((unsigned)rows), dim3(256), 0, st, po, pml,
                       static_cast<f16*>(out), rows, a.d, g);
    return hipGetLastError();
}

}  // namespace mnb
