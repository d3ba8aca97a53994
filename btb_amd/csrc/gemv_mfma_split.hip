// Eight to thirty-two rows of x against a bf16 matrix, the columns split over workgroups.
//
// gemv_mfma_lds gives a workgroup whole rows of the matrix, so every workgroup reads all of x: 32 rows of 9728 values are
// 622 KB a CU where the CU's share of a [2560 x 9728] matrix is 195 KB, and a CU takes in 25 to 30 bytes a nanosecond
// whatever they are. Here the eight slices of a row that the eight waves of that kernel sum are eight workgroups' instead: a
// workgroup keeps its slice of x in LDS (78 KB of those 622, laid out as the matrix cores want it, shared by its waves),
// each of its waves takes whole tiles of sixteen rows over that slice, and the slices' f32 sums meet in a second, small
// launch, in slice order. The slices, the order of the products inside one and the order of the sum are that kernel's, so
// every output has its bits, at any number of rows of x. A workgroup's slice is its number mod 8, so a slice of x is read
// into one die's L2. 32 rows of x, before / after, MI355X: [2560 x 9728] 29.4 -> 16.1 us (3.1 TB/s of weights), [5120 x 7168]
// 38.2 -> 20.3, [16384 x 10240] 165 -> 66 (5.1 TB/s); where it pays is split_pays in gemv.hip.
//
// [workspace] float4 [slice][tile][tile of x rows][lane]: a lane's four consecutive outputs of one row of x, as the matrix
// cores leave them.

#include "btb_common.hpp"
#include "btb_tuning.hpp"

#include "../../include/btb_hip.h"

namespace btb {

constexpr int SPLIT_SLICES = 8;
constexpr int SPLIT_WAVES = 8;
constexpr int SPLIT_SB = 8;                              // steps a sub-block: 512 bytes of each of a tile's rows
constexpr int SPLIT_STRIDE = SPLIT_SB * 64 + 16;         // a slab row: 4 banks past a multiple of 64
constexpr int SPLIT_SLAB = 16 * SPLIT_STRIDE;

// MT: tiles of sixteen rows of x. NSB: sub-blocks a slice holds (its last may be shorter). All of a tile's sub-blocks are in
// flight at once - 40 KB a wave at five - since most waves have a tile or two.
template <int MT, int NSB>
__global__ void __launch_bounds__(SPLIT_WAVES * WAVE) mfma_split_kernel(const uint8_t* __restrict__ w,
                                                                        const uint4* __restrict__ x, f32x4* __restrict__ part,
                                                                        int R, int C, int M, int spw, int groups) {
    extern __shared__ __align__(16) uint8_t lds[];  // the slice of x [step][tile of x rows][lane] x 16 bytes, then the slabs
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int li = lane & 15, lg = lane >> 4;
    const int nsteps = C / 32;
    const int slice = (int)blockIdx.x % SPLIT_SLICES, grp = (int)blockIdx.x / SPLIT_SLICES;
    const int s0 = slice * spw;
    const int n = min(spw, nsteps - s0);  // the slice's steps; none: its sums are zeros, which the fold knows
    if (n <= 0) return;
    uint4* xl = reinterpret_cast<uint4*>(lds);
    uint8_t* slab = lds + (size_t)spw * MT * 1024 + wv * SPLIT_SLAB;
    const int ntiles = (R + 15) / 16;
    const size_t rowbytes = (size_t)C * 2;
    auto tile_of = [&](int k) { return (k * SPLIT_WAVES + wv) * groups + grp; };
    auto row_of = [&](int tile) { return min(tile * 16, R - 16); };  // the last tile of a ragged matrix overlaps its neighbour

    // x: eight rows by 128 bytes a load instruction. A piece past the slice's end is its last piece again, written to that
    // piece's place again; a row past M is the last row again, whose sums nobody reads.
    constexpr int XL = (MT * 2 * NSB * SPLIT_SB / 2 + SPLIT_WAVES - 1) / SPLIT_WAVES;
    u32x4 xv[XL];
    int xo[XL];
#pragma unroll
    for (int q = 0; q < XL; ++q) {
        const int idx = wv + SPLIT_WAVES * q;
        const int row = (idx % (MT * 2)) * 8 + (lane >> 3);
        const int piece = min(idx / (MT * 2) * 8 + (lane & 7), n * 4 - 1);
        xv[q] = *reinterpret_cast<const u32x4*>(x + (size_t)min(row, M - 1) * (C / 8) + (size_t)s0 * 4 + piece);
        xo[q] = ((piece >> 2) * MT + (row >> 4)) * WAVE + (piece & 3) * 16 + (row & 15);
    }
    auto x_to_lds = [&] {
#pragma unroll
        for (int q = 0; q < XL; ++q) reinterpret_cast<u32x4*>(xl)[xo[q]] = xv[q];
    };

    // a load instruction covers two rows' 512 bytes of a sub-block
    const uint32_t lane_row = lane >> 5, lane_byte = (lane & 31) * 16;
    const uint32_t loff = lane_row * SPLIT_STRIDE + lane_byte;
    u32x4 raw[NSB][8];
    auto request = [&](int tile, int sb, u32x4 (&r)[8]) {
        // bytes past the slice's end are its last sixteen again (and meet no product)
        const uint32_t byte = min((uint32_t)(sb * SPLIT_SB * 64) + lane_byte, (uint32_t)(n * 64 - 16));
        const uint8_t* base = w + (size_t)row_of(tile) * rowbytes + (size_t)s0 * 64;
        const uint32_t goff = lane_row * (uint32_t)rowbytes + byte;
#pragma unroll
        for (int q = 0; q < 8; ++q)
            r[q] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(base + (size_t)(2 * q) * rowbytes + goff));
    };
    if (tile_of(0) >= ntiles) {  // uniform: the wave has no tile, only its part of x to bring in
        x_to_lds();
        __syncthreads();
        return;
    }
    __builtin_amdgcn_sched_barrier(0);  // x ahead of the weights: loads come back in order
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) request(tile_of(0), sb, raw[sb]);
    __builtin_amdgcn_sched_barrier(0);
    x_to_lds();
    __syncthreads();
    for (int k = 0; tile_of(k) < ntiles; ++k) {
        const int tile = tile_of(k), next = tile_of(k + 1);
        const bool more = next < ntiles;
        f32x4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int sb = 0; sb < NSB; ++sb) {
#pragma unroll
            for (int q = 0; q < 8; ++q) *reinterpret_cast<u32x4*>(slab + q * 2 * SPLIT_STRIDE + loff) = raw[sb][q];
            if (more) request(next, sb, raw[sb]);
#pragma unroll
            for (int t = 0; t < SPLIT_SB; ++t) {
                const int i = sb * SPLIT_SB + t;
                if (i < n) {  // uniform
                    const bf16x8 a = *reinterpret_cast<const bf16x8*>(slab + li * SPLIT_STRIDE + t * 64 + lg * 16);
#pragma unroll
                    for (int m = 0; m < MT; ++m)
                        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            a, *reinterpret_cast<const bf16x8*>(xl + (i * MT + m) * WAVE + lane), acc[m], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) part[(((size_t)slice * ntiles + tile) * MT + m) * WAVE + lane] = acc[m];
    }
}

// the slices' sums added up in slice order; a thread a lane's four outputs
template <int MT>
__global__ void __launch_bounds__(WAVE) mfma_split_fold_kernel(const f32x4* __restrict__ part, uint16_t* __restrict__ y, int R,
                                                               int M, int live) {
    const int ntiles = (R + 15) / 16;
    const int tile = (int)blockIdx.x / MT, t = (int)blockIdx.x % MT, lane = threadIdx.x;
    f32x4 p[SPLIT_SLICES];
#pragma unroll
    for (int s = 0; s < SPLIT_SLICES; ++s)  // a slice without columns (the last ones of a short row) adds zero
        p[s] = part[(((size_t)min(s, live - 1) * ntiles + tile) * MT + t) * WAVE + lane];
    f32x4 sum = p[0];
#pragma unroll
    for (int s = 1; s < SPLIT_SLICES; ++s) {
        const bool on = s < live;
        sum.x += on ? p[s].x : 0.f;
        sum.y += on ? p[s].y : 0.f;
        sum.z += on ? p[s].z : 0.f;
        sum.w += on ? p[s].w : 0.f;
    }
    const int m = t * 16 + (lane & 15), own = tile * 16, row = min(own, R - 16) + (lane >> 4) * 4;
    if (m < M) {
        uint16_t* o = y + (size_t)m * R + row;
        if (row + 0 >= own) o[0] = f32_bf16(sum.x);
        if (row + 1 >= own) o[1] = f32_bf16(sum.y);
        if (row + 2 >= own) o[2] = f32_bf16(sum.z);
        if (row + 3 >= own) o[3] = f32_bf16(sum.w);
    }
}

static int split_steps(int C) { return (C / 32 + SPLIT_SLICES - 1) / SPLIT_SLICES; }

// floats of workspace a pass of up to 32 rows takes
size_t mfma_split_floats(size_t R, size_t M) {
    return (size_t)SPLIT_SLICES * ((R + 15) / 16) * (M > 16 ? 2 : 1) * WAVE * 4;
}

// the shapes the kernel can take: rows whose slices gemv_mfma_lds cuts eight ways, and whose slice of x and slabs fit LDS
bool mfma_split_fits(size_t R, size_t C) {
    return R >= 16 && C % 32 == 0 && C > 1280 && C <= 10240 && device_info().lds_bytes >= 160 * 1024;
}

template <int MT, int NSB>
static int32_t launch_split(const void* w, const void* x, void* y, int R, int C, int M, float* ws, hipStream_t st) {
    const int spw = split_steps(C), ntiles = (R + 15) / 16;
    const size_t lds = (size_t)spw * MT * 1024 + SPLIT_WAVES * SPLIT_SLAB;
    auto kern = mfma_split_kernel<MT, NSB>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return hip_status(e, "hipFuncSetAttribute");
    // a workgroup a CU; fewer where the tiles are few
    int groups = device_info().cus / SPLIT_SLICES;
    if (groups > ntiles) groups = ntiles;
    f32x4* part = reinterpret_cast<f32x4*>(ws);
    hipLaunchKernelGGL(kern, dim3(SPLIT_SLICES * groups), dim3(SPLIT_WAVES * WAVE), lds, st, static_cast<const uint8_t*>(w),
                       static_cast<const uint4*>(x), part, R, C, M, spw, groups);
    const int live = (C / 32 + spw - 1) / spw;
    hipLaunchKernelGGL(mfma_split_fold_kernel<MT>, dim3(ntiles * MT), dim3(WAVE), 0, st, part, static_cast<uint16_t*>(y), R, M,
                       live);
    return hip_status(hipGetLastError(), "gemv_mfma_split launch");
}

// up to 32 rows of x
int32_t gemv_mfma_split_bf16(const void* w, const void* x, void* y, int R, int C, int M, float* ws, hipStream_t st) {
    const int nsb = (split_steps(C) + SPLIT_SB - 1) / SPLIT_SB;
#define BTB_SPLIT(N_)                                                                        \
    case N_:                                                                                 \
        return M > 16 ? launch_split<2, N_>(w, x, y, R, C, M, ws, st) : launch_split<1, N_>(w, x, y, R, C, M, ws, st)
    switch (nsb) {
        BTB_SPLIT(1);
        BTB_SPLIT(2);
        BTB_SPLIT(3);
        BTB_SPLIT(4);
        BTB_SPLIT(5);
        default:
            return ERR_DOMAIN;
    }
#undef BTB_SPLIT
}

}  // namespace btb
