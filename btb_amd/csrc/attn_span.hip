// Attention of a pass of several rows over long key spans, on the matrix cores: a workgroup walks its span in batches
// of 128 keys with an online softmax. attn_mfma.hip's kernel is the straight-line form of one batch (spans of 128 keys,
// 2 or 4 query heads a kv head); this one takes any span of whole batches and 1, 2, 4 or 8 query heads a kv head, so a
// long cache is cut into as many spans as fill the chip and not into one per 128 keys, whose partial states (520 bytes
// a (row, head, span), written and read back) come to outweigh the keys.
//
// A workgroup: one kv head, one span, up to 32 of the pass's (row, head) pairs; wider passes are more workgroups (the
// z axis), which read the same keys out of the last-level cache. Four waves; the products' layout is attn_mfma.hip's:
// scores S^T = K Q^T with wave w on keys 32 w .. + 31 of the batch, outputs O^T = V^T P^T with wave w on dims 32 w ..
// + 31. Between batches a pair's maximum moves in every lane that holds the pair, so the rescaling needs no exchange; the
// sums stay a lane's own until the span ends.
//
// A weight goes to the matrix cores as two bf16 terms, its rounding and what the rounding left (2^-17 of it stays out),
// one product each into the same sum. A weight rounded once is not enough here: the vector kernels take a weight against
// the maximum of its own stream, eight keys a batch, so the heaviest of them are 1 and exact, and against f64 their
// outputs lie 1.8e-3 to 2.2e-3 off (relative 2-norm, normal q and k, 100 to 32000 keys) where weights taken against a whole
// batch's maximum and rounded once lie 2.1e-3 to 2.2e-3 off; with two terms 1.66e-3, what rounding the outputs to bf16
// alone makes. The second product costs 3 to 8 %: 8 rows x 32 / 8 heads over 6125 keys, with the fold, 15.2 -> 16.4 us
// (the vector kernel 32.8).
// Two terms of unlike sign, or a zero, must not meet an infinite value: a workgroup that ends with an output that is not
// finite walks its span once more with such values taken out of the product and added by their whole weight, to the rows
// that see their keys and to no other - what a later row of the pass holds never reaches an earlier one.
//
// The next batch's K is asked for as soon as the scores are made and its V as soon as this one's lies in LDS, into the
// registers just freed: a batch's arithmetic (2.0 us for 16 pairs, 2.5 for 32) hides the next one's trip. Two barriers a batch:
// the maxima, which are also the sign that the last batch's V and weights have been read, and the weights.
//
// Bound: a batch's chain of phases - scores, maxima, weights, outputs, a barrier between - at one or two workgroups a CU;
// one row x 32 / 8 heads over 32000 keys reads its 131 MB in 26.5 us with the fold, 4.9 TB/s.
//
// ONE, the one-row step: the spans are cut from the keys the cache holds and not from its capacity, so that a large cache
// with few keys in it is spread over the workgroups as a full one is (35200 slots, 704 keys: 19.5 -> 10.0 us; full ones
// as before). Its keys are asked for when *n0 is there; the row's own words travel meanwhile.

#include "btb_attn.hpp"
#include "btb_common.hpp"
#include "btb_head_tile.hpp"
#include "btb_tuning.hpp"

#include <type_traits>

#include "../../include/btb_hip.h"

namespace btb {

constexpr int AS_KEYS = 128;  // keys a batch
constexpr int AS_VROW = 272;  // bytes a V row takes in LDS: 256 + 16, so the eight rows a fragment read touches differ in bank
constexpr int AS_PROW = 144;  // bytes a pair's 32 weights of a step take: 64 a term and 16, so that pairs differ in bank
constexpr int AS_HROW = 272;  // bytes a prepared q, k or v row takes in LDS: as a V row

// own: the pass's own rows kept in LDS (their k, then their v), none where q is given
__host__ __device__ constexpr size_t as_lds_bytes(int NQT, int own) {
    const size_t NQ = 16 * (size_t)NQT;
    return (size_t)AS_KEYS * AS_VROW + 4 * NQ * sizeof(float) + 4 * sizeof(int) + 4 * NQ * AS_PROW +
           2 * (size_t)own * AS_HROW;
}

// eight bf16 values with those that are not finite as zeros
__device__ __forceinline__ uint32_t finite2(uint32_t w) {
    if ((w & 0x7F80u) == 0x7F80u) w &= 0xFFFF0000u;
    if ((w & 0x7F800000u) == 0x7F800000u) w &= 0x0000FFFFu;
    return w;
}
__device__ __forceinline__ uint4 finite8(const uint4& v) {
    return make_uint4(finite2(v.x), finite2(v.y), finite2(v.z), finite2(v.w));
}

// whether a row sees the key of this slot, below `lim`; branch-free
__device__ __forceinline__ bool sees(const RowView& v, int key, int lim) {
    const int tb = v.tree_base >= 0 ? v.tree_base : 0x7FFFFFFF;  // the first of the pass's own slots, if a tree
    const uint32_t named = (v.tree_mask >> min(max(key - tb, 0), 31)) & 1u;
    const bool inside = key >= tb ? named != 0u : key >= v.k_first;
    return (key < min(v.n, lim)) & inside;
}

// NQT tiles of 16 (row, head) pairs a workgroup: pair r is row t_base + r / G, head r % G, G = 1 << gs. TBL: the cache
// has a row map. Every load stays on a slot one of the workgroup's rows may see, so the cache's capacity need not be
// known and what lies past the rows is never read.
// QKV: the rows come as the fused qkv rows, before the q / k norm and rope. A workgroup prepares the q heads of its own
// rows, a tile of 16 a wave, while the first batch's K travels (but for ONE its addresses wait for nothing: they stay
// within the cache's capacity); where its span holds some of the pass's own slots *n0 .. *n0 + T - 1 it prepares the
// pass's k heads too, takes those keys and their values from LDS, and the last of the z axis - whose rows see all of them -
// writes them into the cache. T <= 32. The arithmetic is norm_rope_kv_kernel's, then this kernel's.
template <int NQT, bool TBL, bool QKV, bool ONE = false>
__global__ void __launch_bounds__(256, 2) attn_span_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V,
    const int32_t* __restrict__ n0p, const int32_t* __restrict__ par, int T, int Hq, int Hk, int gs, long long hs,
    long long rs, float scale_log2, float* __restrict__ part_m, float* __restrict__ part_l, float* __restrict__ part_acc,
    int span, int win, const int32_t* __restrict__ tbl, int cap, AmQkv x) {
    constexpr int D = AD, NQ = 16 * NQT;
    static_assert(!(QKV && TBL), "the fused rows go with a cache without a row map");
    static_assert(!ONE || (QKV && NQT == 1), "one row comes as its fused row");
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t* v_lds = lds;                                             // [128 keys][AS_VROW]
    float* red = reinterpret_cast<float*>(lds + AS_KEYS * AS_VROW);   // [4 waves][NQ]: maxima, at the end the sums
    int* odd = reinterpret_cast<int*>(red + 4 * NQ);                  // [4 waves]: an output of the wave is not finite
    uint8_t* p_lds = reinterpret_cast<uint8_t*>(odd + 4);             // [4 steps of 32 keys][NQ pairs][AS_PROW]
    uint8_t* q_lds = p_lds;                                           // QKV, before the first weights: [NQ][AS_HROW]
    uint8_t* kn_lds = p_lds + 4 * NQ * AS_PROW;                       // QKV: the pass's own k rows, then their v rows
    uint8_t* vn_lds = kn_lds + T * AS_HROW;
    static_assert(NQ * AS_HROW <= 4 * NQ * AS_PROW, "the prepared q rows lie where the weights will");
    const int g = blockIdx.x, sp = blockIdx.y, S = gridDim.y, G = 1 << gs;
    const int TPW = NQ >> gs, t_base = blockIdx.z * TPW;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, a = lane >> 4;
    const float ninf = bits_f32(0xff800000u);
    const int parent = tree_parent(par, T);
    int k_begin = sp * span;
    const uint16_t* Kg = K + (size_t)g * hs + a * 8;
    const uint16_t* Vg = V + (size_t)g * hs + (tid & 15) * 8;
    uint4 kreg[2][4], vreg[8];
    // keys past `last` are the last again, not used
    auto request_k = [&](int kb, int last) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int s = min(kb + 32 * wv + 16 * h + c, last);
            const uint16_t* kr = Kg + (size_t)(TBL ? tbl[s] : s) * rs;
#pragma unroll
            for (int ds = 0; ds < 4; ++ds) kreg[h][ds] = *reinterpret_cast<const uint4*>(kr + ds * 32);
        }
    };
    auto request_v = [&](int kb, int last) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int s = min(kb + (tid >> 4) + 16 * i, last);
            vreg[i] = *reinterpret_cast<const uint4*>(Vg + (size_t)(TBL ? tbl[s] : s) * rs);
        }
    };
    const int in_cap = min(k_begin + span, cap) - 1;
    // QKV: the heads to prepare come as tiles of 16 - the workgroup's q heads, then the pass's k heads -, a tile a wave. What
    // does not wait for *n0 is asked for first, a k tile's words whether or not this span turns out to hold the pass's rows.
    constexpr int MAX_TASKS = NQT + 2;
    static_assert(MAX_TASKS <= 4, "a tile a wave");
    const bool k_tile = wv >= NQT;
    const int task_row = k_tile ? (wv - NQT) * 16 + c : t_base + ((wv * 16 + c) >> gs);  // unclamped
    const uint16_t* qkv_row = x.qkv + (size_t)min(task_row, T - 1) * (Hq + 2 * Hk) * D;
    const uint16_t* wn = k_tile ? x.wk : x.wq;
    HeadTile task;
    if constexpr (QKV) {
        const uint16_t* src = qkv_row + (size_t)(k_tile ? Hq + g : g * G + ((wv * 16 + c) & (G - 1))) * D;
        if (wv < NQT || (wv - NQT) * 16 < T) tile_request(task, src, wn, a);
        if constexpr (!ONE) request_k(k_begin, in_cap);
    }
    const int n0 = *n0p;
    if constexpr (ONE) {  // the spans of the keys there are
        span = ((n0 + S) / S + AS_KEYS - 1) / AS_KEYS * AS_KEYS;
        k_begin = sp * span;
    }
    // the keys any of the workgroup's rows may see end at n_max (a chain's last row, or the whole pass for a tree)
    const int n_max = par != nullptr ? n0 + T : n0 + min(T, t_base + TPW);
    const int k_lim = min(n_max, k_begin + span);
    const int last = max(QKV ? min(k_lim - 1, cap - 1) : k_lim - 1, 0);
    const bool own_here = QKV && k_begin < n0 + T && n0 < k_begin + span;  // some of the pass's own slots lie in this span
    // Under a window the walk starts with the first batch that any of the workgroup's rows sees
    TreeRows rows;
    int k_walk = k_begin;
    if (!QKV && win > 0) {  // uniform
        rows = tree_rows(parent, T, win);
        int first = n0 + t_base + 1;
        if (par != nullptr) {
            const int r = lane & 31;
            first = r >= t_base && r < min(T, t_base + TPW) ? n0 + rows.path : n0 + T;
#pragma unroll
            for (int d = 1; d < 32; d <<= 1) first = min(first, lane_value(first, lane ^ d));
        }
        first = min(max(first - win, 0), n0);  // (the pass's own slots are all seen, each by its row)
        k_walk += max(first - k_begin, 0) / AS_KEYS * AS_KEYS;
    }
    const bool any = k_walk < k_lim;

    uint4 qreg[NQT][4];
    if constexpr (QKV) {
        if (any) {
            if constexpr (ONE) request_k(k_begin, last);
            const bool mine = wv < NQT || (own_here && (wv - NQT) * 16 < T);  // uniform in the wave
            if (mine) {
                const int t = min(task_row, T - 1);
                cs_sn_request(task, x.cos_t, x.sin_t, n0 + (x.depth != nullptr ? x.depth[t] : t), a);
                if (k_tile) {
                    const uint16_t* vsrc = qkv_row + (size_t)(Hq + Hk + g) * D + a * 8;
#pragma unroll
                    for (int ds = 0; ds < 4; ++ds) task.vrow[ds] = *reinterpret_cast<const uint4*>(vsrc + ds * 32);
                }
            }
            request_v(k_begin, last);
            if (mine) {
                float v[4][8];
                tile_norm(task, wn != nullptr, x.eps, x.centered, v);
                uint4 out[4];
                tile_rope(v, task, out);
                if (!k_tile) {
#pragma unroll
                    for (int ds = 0; ds < 4; ++ds)
                        *reinterpret_cast<uint4*>(q_lds + (wv * 16 + c) * AS_HROW + ds * 64 + a * 16) = out[ds];
                } else if (task_row < T) {
                    const int slot = n0 + task_row;
#pragma unroll
                    for (int ds = 0; ds < 4; ++ds) {
                        *reinterpret_cast<uint4*>(kn_lds + task_row * AS_HROW + ds * 64 + a * 16) = out[ds];
                        *reinterpret_cast<uint4*>(vn_lds + task_row * AS_HROW + ds * 64 + a * 16) = task.vrow[ds];
                    }
                    // (a slot at or past the cache's capacity is not written: the caller has let the cache overflow)
                    if (blockIdx.z == gridDim.z - 1 && slot >= k_begin && slot < min(k_begin + span, cap)) {
                        uint16_t* kc = x.Kw + (size_t)g * hs + (size_t)slot * rs + a * 8;
                        uint16_t* vc = x.Vw + (size_t)g * hs + (size_t)slot * rs + a * 8;
#pragma unroll
                        for (int ds = 0; ds < 4; ++ds) {
                            *reinterpret_cast<uint4*>(kc + ds * 32) = out[ds];
                            *reinterpret_cast<uint4*>(vc + ds * 32) = task.vrow[ds];
                        }
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int qt = 0; qt < NQT; ++qt)
#pragma unroll
                for (int ds = 0; ds < 4; ++ds)
                    qreg[qt][ds] = *reinterpret_cast<const uint4*>(q_lds + (qt * 16 + c) * AS_HROW + ds * 64 + a * 16);
        }
    } else {
#pragma unroll
        for (int qt = 0; qt < NQT; ++qt) {
            const int r = qt * 16 + c, t = min(t_base + (r >> gs), T - 1), j = r & (G - 1);
            const uint16_t* qr = q + ((size_t)t * Hq + (size_t)g * G + j) * D + a * 8;
#pragma unroll
            for (int ds = 0; ds < 4; ++ds) qreg[qt][ds] = *reinterpret_cast<const uint4*>(qr + ds * 32);
        }
        if (any) {
            request_k(k_walk, last);
            request_v(k_walk, last);
        }
    }

    f32x4 ot[2][NQT];      // O^T tile [dt][qt], lane: pair c of tile qt, dims 32 wv + 16 dt + 4 a .. + 3
    float m[NQT], l[NQT];  // pair c's running maximum (the same in its lanes of every wave), the lane's share of its sum
    if (QKV || win <= 0) rows = tree_rows(parent, T, 0);  // while the first batch travels
    // one batch of keys; CAREFUL: values that are not finite are taken out of the product and added by their whole weight
    auto batch = [&](auto mode, int kb) {
        constexpr bool CAREFUL = decltype(mode)::value;
        if constexpr (CAREFUL) {
            request_k(kb, last);
            request_v(kb, last);
        }
        const bool own = own_here && kb < n0 + T && n0 < kb + AS_KEYS;
        if constexpr (QKV) {
            if (own) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int tr = kb + 32 * wv + 16 * h + c - n0;  // which of the pass's rows this key is, if any
                    const uint8_t* kn = kn_lds + min(max(tr, 0), T - 1) * AS_HROW + a * 16;
#pragma unroll
                    for (int ds = 0; ds < 4; ++ds) {
                        const uint4 v = *reinterpret_cast<const uint4*>(kn + ds * 64);
                        if (tr >= 0 && tr < T) kreg[h][ds] = v;
                    }
                }
            }
        }
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
        const bool more = !CAREFUL && kb + AS_KEYS < k_lim;
        if (more) request_k(kb + AS_KEYS, last);
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
                const RowView rv = row_view_of(rows, par != nullptr, min(t, T - 1), T, n0, win);
                const int lim = t < T ? k_lim : 0;
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const bool live = sees(rv, kb + 32 * wv + 16 * h + 4 * a + i, lim);
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
            b = fmaxf(b, xor_lanes16(b));
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
        if constexpr (QKV) {
            if (own) {  // the rows of the pass among them, by the threads that have just written their places
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int key = kb + (tid >> 4) + 16 * i, tr = key - n0;
                    if (tr >= 0 && tr < T && key < k_lim)
                        *reinterpret_cast<uint4*>(v_lds + (key - kb) * AS_VROW + (tid & 15) * 16) =
                            *reinterpret_cast<const uint4*>(vn_lds + tr * AS_HROW + (tid & 15) * 16);
                }
            }
        }
        if (more) request_v(kb + AS_KEYS, last);
        // the pairs' maxima move; weights in two terms, P^T into LDS
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
                uint32_t pw[2], pw2[2];
#pragma unroll
                for (int i2 = 0; i2 < 2; ++i2) {
                    const float s0 = st[h][qt][2 * i2], s1 = st[h][qt][2 * i2 + 1];
                    const float p0 = s0 == ninf ? 0.f : __builtin_amdgcn_exp2f(s0 - mn);
                    const float p1 = s1 == ninf ? 0.f : __builtin_amdgcn_exp2f(s1 - mn);
                    pw[i2] = f32x2_bf16(p0, p1);
                    pw2[i2] = f32x2_bf16(p0 - bf16lo_f32(pw[i2]), p1 - bf16hi_f32(pw[i2]));
                    sum += p0;
                    sum += p1;
                }
                // step wv (the wave's 32 keys), pair r, slots 16 h + 4 a .. + 3
                const int at = (wv * NQ + r) * AS_PROW + (16 * h + 4 * a) * 2;
                *reinterpret_cast<uint2*>(p_lds + at) = make_uint2(pw[0], pw[1]);
                *reinterpret_cast<uint2*>(p_lds + at + 64) = make_uint2(pw2[0], pw2[1]);
            }
            l[qt] = fmaf(l[qt], corr, sum);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) ot[dt][qt][i] *= corr;
        }
        __syncthreads();
        if constexpr (CAREFUL) {
            RowView see[NQT];
#pragma unroll
            for (int qt = 0; qt < NQT; ++qt)
                see[qt] = row_view_of(rows, par != nullptr, min(t_base + ((qt * 16 + c) >> gs), T - 1), T, n0, win);
#pragma unroll 1
            for (int key = 0; key < AS_KEYS; ++key)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t v =
                            *reinterpret_cast<const uint16_t*>(v_lds + key * AS_VROW + (32 * wv + 16 * dt + 4 * a + i) * 2);
                        if ((v & 0x7F80u) != 0x7F80u) continue;
#pragma unroll
                        for (int qt = 0; qt < NQT; ++qt) {
                            if (!sees(see[qt], kb + key, k_lim)) continue;
                            const uint32_t p = *reinterpret_cast<const uint16_t*>(
                                p_lds + ((key >> 5) * NQ + qt * 16 + c) * AS_PROW + (key & 31) * 2);
                            ot[dt][qt][i] = fmaf(bits_f32(p << 16), bits_f32(v << 16), ot[dt][qt][i]);
                        }
                    }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint4* v = reinterpret_cast<uint4*>(v_lds + ((tid >> 4) + 16 * i) * AS_VROW + (tid & 15) * 16);
                *v = finite8(*v);
            }
            __syncthreads();
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            bf16x8 vfrag[2];
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
                vfrag[dt] = __builtin_bit_cast(bf16x8, make_uint4(vw[0], vw[1], vw[2], vw[3]));
            }
#pragma unroll
            for (int term = 1; term >= 0; --term) {  // the weights' second terms, then their first
                const uint8_t* pt = p_lds + (ks * NQ + c) * AS_PROW + term * 64 + a * 16;
                bf16x8 pfrag[NQT];
#pragma unroll
                for (int qt = 0; qt < NQT; ++qt)
                    pfrag[qt] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(pt + qt * 16 * AS_PROW));
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int qt = 0; qt < NQT; ++qt)
                        ot[dt][qt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vfrag[dt], pfrag[qt], ot[dt][qt], 0, 0, 0);
            }
        }
    };
    auto walk = [&](auto mode) {
#pragma unroll
        for (int qt = 0; qt < NQT; ++qt) {
            m[qt] = ninf;
            l[qt] = 0.f;
            ot[0][qt] = ot[1][qt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int kb = k_walk; kb < k_lim; kb += AS_KEYS) batch(mode, kb);
    };
    walk(std::false_type{});
    bool strange = false;
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt)
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) strange = strange || !(fabsf(ot[dt][qt][i]) < __builtin_inff());
    const bool strange_here = __ballot(strange) != 0;
    if (lane == 0) odd[wv] = strange_here ? 1 : 0;
    __syncthreads();  // the last batch's maxima have been read
    if ((odd[0] | odd[1] | odd[2] | odd[3]) != 0) {  // the same in all four waves
        walk(std::true_type{});
        __syncthreads();
    }
    // the span's state out: the sums meet across the pair's lanes and the waves
#pragma unroll
    for (int qt = 0; qt < NQT; ++qt) {
        float s = l[qt];
        s += xor_lanes16(s);
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

template <int NQT, bool TBL, bool QKV, bool ONE = false>
static int32_t launch_span(const void* q, const void* K, const void* V, const int32_t* n0, const int32_t* par, size_t T,
                           size_t Hq, size_t Hk, int gs, long long hs, long long rs, float scale_log2, float* part_m,
                           float* part_l, float* part_acc, size_t S, int span, int win, const int32_t* tbl, int cap,
                           const AmQkv& x, hipStream_t st) {
    const size_t TPW = (16 * NQT) >> gs;
    const dim3 grid((unsigned)Hk, (unsigned)S, (unsigned)((T + TPW - 1) / TPW));
    auto kern = attn_span_kernel<NQT, TBL, QKV, ONE>;
    const size_t lds = as_lds_bytes(NQT, QKV ? (int)T : 0);
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return hip_status(e, "hipFuncSetAttribute");
    }
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(K),
                       static_cast<const uint16_t*>(V), n0, par, (int)T, (int)Hq, (int)Hk, gs, hs, rs, scale_log2, part_m,
                       part_l, part_acc, span, win, tbl, cap, x);
    return hip_status(hipGetLastError(), "attn_span launch");
}

static int group_shift(size_t G) { return G == 1 ? 0 : G == 2 ? 1 : G == 4 ? 2 : G == 8 ? 3 : -1; }

// Tiles of 16 pairs a workgroup takes: two, one where the pass has no more or where workgroups of one do not outnumber the
// CUs - a batch is 2.0 us for one tile, 2.5 for two. (8 rows x 32 / 8 heads over 14000 keys, one tile / two: 16 spans, 256
// workgroups of one, 22.6 / 26.4 us; 21 spans, 336 workgroups of one, 27.0 / 22.5. Four tiles want 360 registers, a
// workgroup a CU, and lose everywhere: 32 rows over 14000 keys, 16 spans, 64.2 / 40.2 / 43.7.) The bits are the same.
static int tiles_of(size_t T, size_t Hk, int gs, size_t S) {
    const size_t rows = 16u >> gs;
    return T <= rows || Hk * S * ((T + rows - 1) / rows) <= (size_t)device_info().cus ? 1 : 2;
}

// whether a pass takes this kernel: several rows, 1, 2, 4 or 8 query heads a kv head
bool attn_span_fits(size_t T, size_t G) { return T >= 2 && group_shift(G) >= 0 && tuning("attn_mfma") != 0; }

// the partial states of every (row, head, span), for the merge
int32_t attn_decode_span(const void* q, const void* K, const void* V, const int32_t* n0, const int32_t* par, size_t T,
                         size_t Hq, size_t Hk, long long hs, long long rs, float scale_log2, float* part_m, float* part_l,
                         float* part_acc, size_t S, int span, int win, const int32_t* tbl, hipStream_t st) {
    const int gs = group_shift(Hq / Hk), tiles = tiles_of(T, Hk, gs, S);
#define AS(NN, TBL)                                                                                                      \
    return launch_span<NN, TBL, false>(q, K, V, n0, par, T, Hq, Hk, gs, hs, rs, scale_log2, part_m, part_l, part_acc, S, \
                                       span, win, tbl, 0, AmQkv{}, st)
    if (tbl != nullptr) {
        if (tiles == 1) AS(1, true);
        AS(2, true);
    }
    if (tiles == 1) AS(1, false);
    AS(2, false);
#undef AS
}

// the same states from the fused qkv rows; the new K / V rows land in the cache on the way. T <= 32
int32_t attn_decode_span_qkv(const AmQkv& x, const int32_t* n0, const int32_t* par, size_t T, size_t Hq, size_t Hk,
                             long long hs, long long rs, float scale_log2, float* part_m, float* part_l, float* part_acc,
                             size_t S, int span, size_t cap, hipStream_t st) {
    const int gs = group_shift(Hq / Hk), tiles = tiles_of(T, Hk, gs, S), capi = (int)(cap < 0x7FFFFFFFu ? cap : 0x7FFFFFFFu);
#define AS(...)                                                                                                         \
    return launch_span<__VA_ARGS__>(nullptr, x.Kw, x.Vw, n0, par, T, Hq, Hk, gs, hs, rs, scale_log2, part_m, part_l, \
                                        part_acc, S, span, 0, nullptr, capi, x, st)
    if (T == 1) AS(1, false, true, true);
    if (tiles == 1) AS(1, false, true);
    AS(2, false, true);
#undef AS
}

}  // namespace btb
