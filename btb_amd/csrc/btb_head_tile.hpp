// Sixteen attention heads at a time in the layout the matrix cores take an operand in: their norm and rope, for the
// kernels that start from a pass's fused qkv rows (attn_mfma.hip, attn_span.hip).
#pragma once

#include "btb_attn.hpp"
#include "btb_common.hpp"

namespace btb {

__device__ __forceinline__ float xor_lanes16(float v) {  // the value of lane l ^ 16
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(((int)(threadIdx.x & 63) ^ 16) << 2, __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float xor_lanes32(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(((int)(threadIdx.x & 63) ^ 32) << 2, __builtin_bit_cast(int, v)));
}

// A tile of 16 heads (q heads of a pass's rows, or the rows' k heads) prepared - RMSNorm, rope - in the layout the
// matrix cores take an operand in: lane (c, a) holds head c's dims 32 ds + 8 a .. + 7 for ds = 0 .. 3. Under rope the
// partner of a dim, 64 dims away, is chunk ds ^ 2 of the same lane. The sum of squares folds in the order of
// head_finish's (a lane l there holds dims 2 l, 2 l + 1 and the lanes fold by group_sum<64>: l ^ 1, ^ 2, ^ 4 .. ^ 32;
// here l = 16 ds + 4 a + e / 2), so the bits that come out are head_finish's.
struct HeadTile {
    uint4 raw[4], wn[4], cs[4], sn[4];
    uint4 vrow[4];  // with a k tile: the rows' v, as they come
};
__device__ __forceinline__ void tile_request(HeadTile& h, const uint16_t* src, const uint16_t* wn, int a) {
    const uint16_t* wsrc = wn != nullptr ? wn : src;  // no weight: any words, unused
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
        h.raw[ds] = *reinterpret_cast<const uint4*>(src + ds * 32 + a * 8);
        h.wn[ds] = *reinterpret_cast<const uint4*>(wsrc + ds * 32 + a * 8);
    }
}
__device__ __forceinline__ void cs_sn_request(HeadTile& h, const uint16_t* cos_t, const uint16_t* sin_t, int pos, int a) {
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
        h.cs[ds] = *reinterpret_cast<const uint4*>(cos_t + (size_t)pos * AD + ds * 32 + a * 8);
        h.sn[ds] = *reinterpret_cast<const uint4*>(sin_t + (size_t)pos * AD + ds * 32 + a * 8);
    }
}
__device__ __forceinline__ float bf16_of(const uint4& q, int e) {  // element e of eight
    const uint32_t w = e < 2 ? q.x : e < 4 ? q.y : e < 6 ? q.z : q.w;
    return (e & 1) ? bf16hi_f32(w) : bf16lo_f32(w);
}
__device__ __forceinline__ void tile_norm(const HeadTile& h, bool has_wn, float eps, int centered, float (&v)[4][8]) {
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[ds][e] = bf16_of(h.raw[ds], e);
    if (has_wn) {
        float t[4];
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) {
            float sq[4];
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2)
                sq[e2] = fmaf(v[ds][2 * e2 + 1], v[ds][2 * e2 + 1], fmaf(v[ds][2 * e2], v[ds][2 * e2], 0.f));
            t[ds] = (sq[0] + sq[1]) + (sq[2] + sq[3]);  // l ^ 1, then l ^ 2
        }
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) t[ds] += xor_lanes16(t[ds]);  // l ^ 4
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) t[ds] += xor_lanes32(t[ds]);  // l ^ 8
        const float ss = (t[0] + t[1]) + (t[2] + t[3]);              // l ^ 16, then l ^ 32
        const float rstd = rsqrtf(ss / (float)AD + eps);
#pragma unroll
        for (int ds = 0; ds < 4; ++ds)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float w = bf16_of(h.wn[ds], e);
                v[ds][e] = bfround(v[ds][e] * rstd * (centered ? 1.f + w : w));
            }
    }
}
__device__ __forceinline__ void tile_rope(const float (&v)[4][8], const HeadTile& h, uint4 (&out)[4]) {
#pragma unroll
    for (int ds = 0; ds < 4; ++ds) {
        const float sgn = ds < 2 ? -1.f : 1.f;
        uint32_t w[4];
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2) {
            float o[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int e = 2 * e2 + i;
                const float qc = bfround(v[ds][e] * bf16_of(h.cs[ds], e));
                o[i] = fmaf(sgn * v[ds ^ 2][e], bf16_of(h.sn[ds], e), qc);
            }
            w[e2] = f32x2_bf16(o[0], o[1]);
        }
        out[ds] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// What a variant that starts from the pass's fused qkv rows [T, (Hq + 2 Hk) 128] needs on top: the q / k norm
// weights (or none), the rope tables, the rows' depths (a tree) or none (a chain: row t stands at *n0 + t), the cache
// to write the new rows into.
struct AmQkv {
    const uint16_t* qkv;
    const uint16_t* wq;
    const uint16_t* wk;
    const uint16_t* cos_t;
    const uint16_t* sin_t;
    const int32_t* depth;
    uint16_t* Kw;
    uint16_t* Vw;
    float eps;
    int centered;
};
}  // namespace btb
