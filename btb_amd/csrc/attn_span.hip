// Attention of a pass of several rows over long key spans, on the matrix cores: a workgroup walks its span in batches
// of 128 keys with an online softmax. attn_mfma.hip's kernel is the straight-line form of one batch (spans of 128 keys,
// 2 or 4 query heads a kv head); this one takes any span of whole batches and 1, 2, 4 or 8 query heads a kv head, so a
// long cache is cut into as many spans as fill the chip and not into one per 128 keys, whose partial states (520 bytes
// a (row, head, span), written and read back) come to outweigh the keys.
//
// A workgroup: one kv head, one span, up to 64 of the pass's (row, head) pairs; wider passes are more workgroups (the
// z axis), which read the same keys out of the last-level cache. Four waves; the products' layout is attn_mfma.hip's:
// scores S^T = K Q^T with wave w on keys 32 w .. + 31 of the batch, outputs O^T = V^T P^T with wave w on dims 32 w ..
// + 31, weights rounded to bf16 and their sum made of the rounded ones. Between batches a pair's maximum moves in every
// lane that holds the pair, so the rescaling needs no exchange; the sums stay a lane's own until the span ends.
//
// The next batch's K is asked for as soon as the scores are made and its V as soon as this one's lies in LDS, into the
// registers just freed: a batch's arithmetic (about 1 us for 64 pairs) hides the next one's trip. Two barriers a batch:
// the maxima, which are also the sign that the last batch's V and weights have been read, and the weights.
//
// Bound: HBM for the keys (one read of the span), then the vector ALUs' softmax: 10 instructions a score against
// a quarter of an MFMA.

#include "btb_attn.hpp"
#include "btb_common.hpp"
#include "btb_tuning.hpp"

#include "../../include/btb_hip.h"

namespace btb {

constexpr int AS_D = 128;
constexpr int AS_KEYS = 128;  // keys a batch
constexpr int AS_VROW = 272;  // bytes a V row takes in LDS: 256 + 16, so the eight rows a fragment read touches differ in bank
constexpr int AS_PROW = 80;   // bytes a pair's 32 weights of a step take: 64 + 16, sixteen pairs in sixteen bank groups

__host__ __device__ constexpr size_t as_lds_bytes(int NQT) {
    const size_t NQ = 16 * (size_t)NQT;
    return (size_t)AS_KEYS * AS_VROW + 4 * NQ * sizeof(float) + 4 * NQ * AS_PROW;
}

__device__ __forceinline__ float as_xor16(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(((int)(threadIdx.x & 63) ^ 16) << 2, __builtin_bit_cast(int, v)));
}

// NQT tiles of 16 (row, head) pairs a workgroup: pair r is row t_base + r / G, head r % G, G = 1 << gs. TBL: the cache
// has a row map. Every load stays on a slot one of the workgroup's rows may see, so the cache's capacity need not be
// known and what lies past the rows is never read.
template <int NQT, bool TBL>
__global__ void __launch_bounds__(256, 2) attn_span_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V,
    const int32_t* __restrict__ n0p, const int32_t* __restrict__ par, int T, int Hq, int Hk, int gs, long long hs,
    long long rs, float scale_log2, float* __restrict__ part_m, float* __restrict__ part_l, float* __restrict__ part_acc,
    int span, int win, const int32_t* __restrict__ tbl) {
    constexpr int D = AS_D, NQ = 16 * NQT;
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t* v_lds = lds;                                             // [128 keys][AS_VROW]
    float* red = reinterpret_cast<float*>(lds + AS_KEYS * AS_VROW);   // [4 waves][NQ]: maxima, at the end the sums
    uint8_t* p_lds = reinterpret_cast<uint8_t*>(red + 4 * NQ);        // [4 steps of 32 keys][NQ pairs][AS_PROW]
    const int g = blockIdx.x, sp = blockIdx.y, S = gridDim.y, G = 1 << gs;
    const int TPW = NQ >> gs, t_base = blockIdx.z * TPW;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int c = lane & 15, a = lane >> 4;
    const float ninf = bits_f32(0xff800000u);
    const int parent = tree_parent(par, T);
    const int n0 = *n0p;
    const int k_begin = sp * span;
    // the keys any of the workgroup's rows may see end at n_max (a chain's last row, or the whole pass for a tree)
    const int n_max = par != nullptr ? n0 + T : n0 + min(T, t_base + TPW);
    const int k_lim = min(n_max, k_begin + span);
    const int last = max(k_lim - 1, 0);

    uint4 qreg[NQT][4];
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
        const int r = qt * 16 + c, t = min(t_base + (r >> gs), T - 1), j = r & (G - 1);
        const uint16_t* qr = q + ((size_t)t * Hq + (size_t)g * G + j) * D + a * 8;
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) qreg[qt][ds] = *reinterpret_cast<const uint4*>(qr + ds * 32);
    }
    const uint16_t* Kg = K + (size_t)g * hs + a * 8;
    const uint16_t* Vg = V + (size_t)g * hs + (tid & 15) * 8;
    auto slot_of = [&](int key) {
        const int s = min(key, last);  // past the end: the last key again, not used
        return TBL ? tbl[s] : s;
    };
    uint4 kreg[2][4], vreg[8];
    auto request_k = [&](int kb) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint16_t* kr = Kg + (size_t)slot_of(kb + 32 * wv + 16 * h + c) * rs;
#pragma unroll
            for (int ds = 0; ds < 4; ++ds) kreg[h][ds] = *reinterpret_cast<const uint4*>(kr + ds * 32);
        }
    };
    auto request_v = [&](int kb) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            vreg[i] = *reinterpret_cast<const uint4*>(Vg + (size_t)slot_of(kb + (tid >> 4) + 16 * i) * rs);
    };

    f32x4 ot[2][NQT];      // O^T tile [dt][qt], lane: pair c of tile qt, dims 32 wv + 16 dt + 4 a .. + 3
    float m[NQT], l[NQT];  // pair c's running maximum (the same in its lanes of every wave), the lane's share of its sum
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
        m[qt] = ninf;
        l[qt] = 0.f;
        ot[0][qt] = ot[1][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (k_begin < k_lim) {
        request_k(k_begin);
        request_v(k_begin);
    }
    const uint32_t rows = tree_rows(parent, T);  // while the first batch travels
    for (int kb = k_begin; kb < k_lim; kb += AS_KEYS) {
        // scores: S^T tile [h][qt], lane: pair c of tile qt against keys kb + 32 wv + 16 h + 4 a .. + 3
        f32x4 st[2][NQT];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int qt = 0; qt < NQT; ++qt) {
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < 4; ++ds)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kreg[h][ds]),
                                                                  __builtin_bit_cast(bf16x8, qreg[qt][ds]), acc, 0, 0, 0);
                st[h][qt] = acc;
            }
        const bool more = kb + AS_KEYS < k_lim;
        if (more) request_k(kb + AS_KEYS);
        // scaled, masked where a row may not see a key (a batch wholly in the cache, without a window, needs no mask)
        if (kb + AS_KEYS <= n0 && win == 0) {
#pragma unroll
            for (int qt = 0; qt < NQT; ++qt)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st[h][qt][i] *= scale_log2;
        } else {
#pragma unroll
            for (int qt = 0; qt < NQT; ++qt) {
                const int t = t_base + ((qt * 16 + c) >> gs);
                const RowView rv = row_view_of(rows, par, min(t, T - 1), T, n0, win);
                const int k_end = t < T ? min(rv.n, k_lim) : 0;
                const int tb = rv.tree_base >= 0 ? rv.tree_base : 0x7FFFFFFF;  // the first of the pass's own slots, if a tree
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = kb + 32 * wv + 16 * h + 4 * a + i;
                        const uint32_t named = (rv.tree_mask >> min(max(key - tb, 0), 31)) & 1u;
                        const bool inside = key >= tb ? named != 0u : key >= rv.k_first;
                        const bool live = (key < k_end) & inside;
                        st[h][qt][i] = live ? st[h][qt][i] * scale_log2 : ninf;
                    }
            }
        }
#pragma unroll
        for (int qt = 0; qt < NQT; ++qt) {
            float b = ninf;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) b = fmaxf(b, st[h][qt][i]);
            b = fmaxf(b, as_xor16(b));
            b = fmaxf(b, xor32(b));
            if (a == 0) red[wv * NQ + qt * 16 + c] = b;
        }
        __syncthreads();
        // V into LDS, keys past the end as zeros (weight 0 times whatever bits lie there must not make a NaN)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int kl = (tid >> 4) + 16 * i;
            *reinterpret_cast<uint4*>(v_lds + kl * AS_VROW + (tid & 15) * 16) =
                kb + kl < k_lim ? vreg[i] : make_uint4(0u, 0u, 0u, 0u);
        }
        if (more) request_v(kb + AS_KEYS);
        // the pairs' maxima move; weights, rounded to bf16, P^T into LDS
#pragma unroll
        for (int qt = 0; qt < NQT; ++qt) {
            const int r = qt * 16 + c;
            const float mn = fmaxf(fmaxf(m[qt], fmaxf(red[r], red[NQ + r])), fmaxf(red[2 * NQ + r], red[3 * NQ + r]));
            // nothing seen yet: the state is as it was (zeros) and no difference of infinities is formed
            const float corr = m[qt] == ninf ? 0.f : __builtin_amdgcn_exp2f(m[qt] - mn);
            m[qt] = mn;
            float sum = 0.f;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t pw[2];
#pragma unroll
                for (int i2 = 0; i2 < 2; ++i2) {
                    const float s0 = st[h][qt][2 * i2], s1 = st[h][qt][2 * i2 + 1];
                    const float p0 = s0 == ninf ? 0.f : __builtin_amdgcn_exp2f(s0 - mn);
                    const float p1 = s1 == ninf ? 0.f : __builtin_amdgcn_exp2f(s1 - mn);
                    pw[i2] = f32x2_bf16(p0, p1);
                    sum += bf16lo_f32(pw[i2]);
                    sum += bf16hi_f32(pw[i2]);
                }
                // step wv (the wave's 32 keys), pair r, slots 16 h + 4 a .. + 3
                *reinterpret_cast<uint2*>(p_lds + (wv * NQ + r) * AS_PROW + (16 * h + 4 * a) * 2) = make_uint2(pw[0], pw[1]);
            }
            l[qt] = fmaf(l[qt], corr, sum);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) ot[dt][qt][i] *= corr;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            uint4 pfrag[NQT];
#pragma unroll
            for (int qt = 0; qt < NQT; ++qt)
                pfrag[qt] = *reinterpret_cast<const uint4*>(p_lds + (ks * NQ + qt * 16 + c) * AS_PROW + a * 16);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) {
                // V^T fragment: dim 32 wv + 16 dt + c, keys 32 ks + 8 a .. + 7
                const uint8_t* col = v_lds + (32 * ks + 8 * a) * AS_VROW + (32 * wv + 16 * dt + c) * 2;
                uint32_t vw[4];
#pragma unroll
                for (int e2 = 0; e2 < 4; ++e2) {
                    const uint32_t lo = *reinterpret_cast<const uint16_t*>(col + (2 * e2) * AS_VROW);
                    const uint32_t hi = *reinterpret_cast<const uint16_t*>(col + (2 * e2 + 1) * AS_VROW);
                    vw[e2] = lo | (hi << 16);
                }
                const bf16x8 vfrag = __builtin_bit_cast(bf16x8, make_uint4(vw[0], vw[1], vw[2], vw[3]));
#pragma unroll
                for (int qt = 0; qt < NQT; ++qt)
                    ot[dt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vfrag, __builtin_bit_cast(bf16x8, pfrag[qt]),
                                                                         ot[dt][qt], 0, 0, 0);
            }
        }
    }
    // the span's state out: the sums meet across the pair's lanes and the waves
    __syncthreads();  // the last batch's maxima have been read
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
        float s = l[qt];
        s += as_xor16(s);
        s += xor32(s);
        if (a == 0) red[wv * NQ + qt * 16 + c] = s;
    }
    __syncthreads();
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
        const int r = qt * 16 + c, t = t_base + (r >> gs), j = r & (G - 1);
        if (t < T) {
            const size_t o = ((((size_t)t * Hk + g) * S + sp) << gs) + j;
            if (wv == 0 && a == 0) {
                part_m[o] = m[qt];
                part_l[o] = ((red[r] + red[NQ + r]) + red[2 * NQ + r]) + red[3 * NQ + r];
            }
            float* dst = part_acc + o * D + 32 * wv + 4 * a;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
                *reinterpret_cast<float4*>(dst + 16 * dt) =
                    make_float4(ot[dt][qt][0], ot[dt][qt][1], ot[dt][qt][2], ot[dt][qt][3]);
        }
    }
}

template <int NQT>
static void launch_span(const void* q, const void* K, const void* V, const int32_t* n0, const int32_t* par, int T, int Hq,
                        int Hk, int gs, long long hs, long long rs, float scale_log2, float* part_m, float* part_l,
                        float* part_acc, int S, int span, int win, const int32_t* tbl, hipStream_t st) {
    const int TPW = (16 * NQT) >> gs;
    const dim3 grid((unsigned)Hk, (unsigned)S, (unsigned)((T + TPW - 1) / TPW));
    static_assert(as_lds_bytes(NQT) <= 64 * 1024, "within what a workgroup gets without asking for more");
#define SPAN(TBL)                                                                                                   \
    hipLaunchKernelGGL((attn_span_kernel<NQT, TBL>), grid, dim3(256), as_lds_bytes(NQT), st,                        \
                       static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(K),                            \
                       static_cast<const uint16_t*>(V), n0, par, T, Hq, Hk, gs, hs, rs, scale_log2, part_m, part_l, \
                       part_acc, span, win, tbl)
    if (tbl != nullptr) SPAN(true);
    else SPAN(false);
#undef SPAN
}

// whether a pass takes this kernel: several rows, 1, 2, 4 or 8 query heads a kv head
bool attn_span_fits(size_t T, size_t G) {
    return T >= 2 && (G == 1 || G == 2 || G == 4 || G == 8) && tuning("attn_mfma") != 0;
}

// the partial states of every (row, head, span), for the merge
int32_t attn_decode_span(const void* q, const void* K, const void* V, const int32_t* n0, const int32_t* par, size_t T,
                         size_t Hq, size_t Hk, long long hs, long long rs, float scale_log2, float* part_m, float* part_l,
                         float* part_acc, size_t S, int span, int win, const int32_t* tbl, hipStream_t st) {
    const size_t G = Hq / Hk, pairs = T * G;  // pairs of one kv head
    const int gs = G == 1 ? 0 : G == 2 ? 1 : G == 4 ? 2 : 3;
#define AS(NN) \
    launch_span<NN>(q, K, V, n0, par, (int)T, (int)Hq, (int)Hk, gs, hs, rs, scale_log2, part_m, part_l, part_acc, (int)S, \
                    span, win, tbl, st)
    if (pairs <= 16) AS(1);
    else if (pairs <= 32) AS(2);
    else AS(4);
#undef AS
    return hip_status(hipGetLastError(), "attn_decode_span launch");
}

}  // namespace btb
