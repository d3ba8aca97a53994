// bf16 verify widths (M = 5..32 rows of x) over rows of up to 4096 columns, any multiple of 8: two tiles of weights in flight a
// wave.
//
// The decomposition is gemv_mfma_lds's - KS waves a workgroup, a wave a fixed slice of the columns whose x fragments it holds
// for the whole kernel, tiles of sixteen rows, the waves' partial tiles folded through LDS in wave order - and so are the
// slices, the order of the products and the order of the sum: every output has that kernel's bits. What differs is how the
// weights come in. There a wave has one sub-block of eight steps in flight, two trips to memory a tile for rows of 2560 columns,
// the second a quarter full: 64 and then 16 KB a CU where the memory's latency under load asks for 160. Here a wave's whole
// slice of a tile is one run of 16-byte pieces dealt out to the lanes (any slice length fills its load instructions), and
// the next two tiles are always on their way.

#include "btb_common.hpp"
#include "btb_formats.hpp"
#include "btb_stream.hpp"
#include "btb_tuning.hpp"

#include "../../include/btb_hip.h"

namespace btb {

// SPW: the steps (32 columns) a wave's slice holds at most. TR: the rows of a tile that are rows of the matrix; the others are
// not read, and what the matrix cores make of them is not written. RAG: R is no multiple of TR (and at least that): the last
// tile starts TR rows before the end and writes the rows no other tile has. GLU: W is I gate rows over I up rows, a tile
// eight of each (the same outputs'), y their fold [M, I]; RAG there: I is no multiple of eight. XN: x is not given but made, the
// residual add and RMSNorm of xa (every workgroup makes the pass's rows, add_rmsnorm_kernel's bits).
template <int KS, int MT, int SPW, int TR, bool RAG, bool GLU, bool XN>
__device__ __forceinline__ void mfma_ahead(const uint8_t* __restrict__ w, const uint4* __restrict__ x, uint16_t* __restrict__ y,
                                           int R, int C, int M, const XArgs& xa) {
    constexpr int PIECES = SPW * 4;                      // 16-byte pieces a slice has of a row
    constexpr int NLD = (TR * PIECES + WAVE - 1) / WAVE;  // load instructions a wave's share of a tile takes
    constexpr int STRIDE = SPW * 64 + 16;                // a slab row: 4 banks past a multiple of 32
    constexpr int SLAB = 16 * STRIDE;
    static_assert(!GLU || TR == 16, "a folded tile is eight gate rows over eight up rows");
    extern __shared__ __align__(16) uint8_t lds[];  // KS slabs, then two sets of KS * MT partial tiles; XN: the made rows first
    const int lane = threadIdx.x & (WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int li = lane & 15, lg = lane >> 4;
    uint8_t* slab = lds + wv * SLAB;
    f32x4* part = reinterpret_cast<f32x4*>(lds + KS * SLAB);
    const int nsteps = (C + 31) / 32, spw = (nsteps + KS - 1) / KS, s0 = wv * spw;
    const int n = max(min(s0 + spw, nsteps) - s0, 0);  // this wave's steps; none: it adds zeros
    const uint32_t rowbytes = (uint32_t)C * 2;
    const int ntiles = RAG ? (R + TR - 1) / TR : R / TR;
    const int grid = (int)gridDim.x, first = (int)blockIdx.x;
    const int turns = (ntiles - first + grid - 1) / grid;

    const int sn = n > 0 ? s0 : 0, last = max(n, 1) - 1;  // a wave without steps reads (and leaves) the first slice's
    // the slice's bytes of a row; C no multiple of 32: the last step is short, x and the weights past its end are zeros
    const uint32_t valid = min((uint32_t)(last + 1) * 64, rowbytes - (uint32_t)sn * 64);
    const bool ragged = valid % 64 != 0;  // uniform
    uint4 xb[MT][SPW];
    if constexpr (XN) {
        static_assert(MT == 1, "sixteen rows in the making");
        const int stride = C * 2 + 16;
        // A wave makes a row by itself: four sums a lane, each that of a lane of one of the four waves that add_rmsnorm_kernel
        // gives a row, over the same words in the same order. (Rows and weights at any 2-byte place, as in stage_x.)
        // Several rows' words are asked for at once where the rows are short: two waves that made eight rows of 520 values one
        // after the other took 6 us of a launch of 13.
        constexpr int WORDS = (KS * SPW * 32 + 1023) / 1024;  // 4-element words a lane has of each of the four
        constexpr int ROWS = WORDS == 1 ? 4 : WORDS == 2 ? 2 : 1;
        const int n4 = C / 4;
        const bool has_y = xa.y != nullptr, writer = first == 0 && xa.h_out != nullptr;
        const uint2* ws = reinterpret_cast<const uint2*>(xa.norm_w);
        auto word = [&](int v, int q) { return q * 256 + v * 64 + lane; };
        for (int m0 = wv; m0 < M; m0 += KS * ROWS) {
            uint2 hv[ROWS][4][WORDS], yv[ROWS][4][WORDS];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {  // past the pass's rows its last again, made and left like the first time
                const int m = min(m0 + r * KS, M - 1);
                size_t hrow = (size_t)m;
                if (xa.ids != nullptr) hrow = (size_t)min(max(xa.ids[m], 0), xa.vocab - 1);
                const uint2* hs = reinterpret_cast<const uint2*>(xa.x + hrow * C);
                const uint2* ys = has_y ? reinterpret_cast<const uint2*>(xa.y + (size_t)m * C) : hs;
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int q = 0; q < WORDS; ++q) {
                        hv[r][v][q] = hs[min(word(v, q), n4 - 1)];
                        yv[r][v][q] = ys[min(word(v, q), n4 - 1)];
                    }
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const int m = min(m0 + r * KS, M - 1);
                float sums[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float ss = 0.f;
#pragma unroll
                    for (int q = 0; q < WORDS; ++q) {
                        const int i = word(v, q);
                        const uint2 hw = hv[r][v][q], yw = yv[r][v][q];
                        float f[4] = {bf16lo_f32(hw.x), bf16hi_f32(hw.x), bf16lo_f32(hw.y), bf16hi_f32(hw.y)};
                        const float g[4] = {bf16lo_f32(yw.x), bf16hi_f32(yw.x), bf16lo_f32(yw.y), bf16hi_f32(yw.y)};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float sum = bfround(f[e] + g[e]);
                            f[e] = has_y ? sum : f[e];
                            const float sq = fmaf(f[e], f[e], ss);
                            ss = i < n4 ? sq : ss;
                        }
                        hv[r][v][q] = make_uint2(f32x2_bf16(f[0], f[1]), f32x2_bf16(f[2], f[3]));  // exact: bf16 values
                        if (writer && i < n4) reinterpret_cast<uint2*>(xa.h_out + (size_t)m * C)[i] = hv[r][v][q];
                    }
                    sums[v] = wave_sum(ss);
                }
                const float rstd = rsqrtf((((sums[0] + sums[1]) + sums[2]) + sums[3]) / (float)C + xa.eps);
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int q = 0; q < WORDS; ++q) {
                        const int i = word(v, q);
                        const uint2 hw = hv[r][v][q], nw = ws[min(i, n4 - 1)];
                        const float f[4] = {bf16lo_f32(hw.x), bf16hi_f32(hw.x), bf16lo_f32(hw.y), bf16hi_f32(hw.y)};
                        const float g[4] = {bf16lo_f32(nw.x), bf16hi_f32(nw.x), bf16lo_f32(nw.y), bf16hi_f32(nw.y)};
                        float o[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = f[e] * rstd * (xa.centered ? 1.f + g[e] : g[e]);
                        if (i < n4)
                            *reinterpret_cast<uint2*>(lds + (size_t)m * stride + (size_t)i * 8) =
                                make_uint2(f32x2_bf16(o[0], o[1]), f32x2_bf16(o[2], o[3]));
                    }
            }
        }
        __syncthreads();
        const uint8_t* xr = lds + (size_t)min(li, M - 1) * stride + (size_t)sn * 64;
#pragma unroll
        for (int i = 0; i < SPW; ++i)
            xb[0][i] = *reinterpret_cast<const uint4*>(xr + min(min(i, last) * 4 + lg, (int)valid / 16 - 1) * 16);
        __syncthreads();  // the rows have been read: the slabs may take their place
    }
#pragma unroll
    for (int t = 0; t < (XN ? 0 : MT); ++t) {
        const uint4* xr = x + (size_t)min(t * 16 + li, M - 1) * (C / 8) + (size_t)sn * 4;
#pragma unroll
        for (int i = 0; i < SPW; ++i) xb[t][i] = xr[min(min(i, last) * 4 + lg, (int)valid / 16 - 1)];
    }

    // where the lane's pieces of a tile lie: in the matrix past the tile's first byte of the slice, and in the slab. Pieces
    // past the tile are its last one again, bytes past the slice's end its last sixteen again (they meet no product)
    constexpr bool WHOLE = WAVE % PIECES == 0;  // a load covers whole rows of the slice: one offset a lane for all of them
    constexpr int NOFF = WHOLE ? 1 : NLD;
    uint32_t goff[NOFF], loff[NOFF];
#pragma unroll
    for (int q = 0; q < NOFF; ++q) {
        const int p = WHOLE ? lane : min(q * WAVE + lane, TR * PIECES - 1);
        const uint32_t row = (uint32_t)p / PIECES, byte = (uint32_t)p % PIECES * 16;
        goff[q] = (row + (GLU && !WHOLE && row >= 8 ? (uint32_t)R / 2 - 8 : 0)) * rowbytes + min(byte, valid - 16);
        loff[q] = row * STRIDE + byte;
    }
    constexpr int RPL = WAVE / PIECES;  // WHOLE: rows a load covers
    static_assert(!WHOLE || TR % RPL == 0, "a tile is whole loads");
    constexpr int OUT = GLU ? 8 : TR;  // outputs a tile
    const int outs = GLU ? R / 2 : R;
    auto row_of = [&](int tile) { return RAG ? min(tile * OUT, outs - OUT) : tile * OUT; };
    uint32_t past = 0;  // the loads whose piece lies past a short last step's end
    if (ragged) {
#pragma unroll
        for (int q = 0; q < NLD; ++q)
            if ((uint32_t)min(q * WAVE + lane, TR * PIECES - 1) % PIECES * 16 >= valid) past |= 1u << q;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int i = 0; i < SPW; ++i)
                if (i * 64 + lg * 16 >= (int)valid) xb[t][i] = make_uint4(0, 0, 0, 0);
    }
    uint4 raw[2][NLD];
    // The loads of the workgroup's k-th tile. Past its last one they are issued all the same, of one piece a wave: loads under
    // a condition are loads the compiler cannot count, and it then waits for every one in flight.
    auto request = [&](int k, uint4 (&r)[NLD]) {
        const bool live = k < turns;
        const uint8_t* base = w + (size_t)row_of(live ? first + k * grid : first) * rowbytes + (size_t)sn * 64;
        // (a row is no bytes past the last tile, not a choice a load: of those the compiler made a branch each in the fold)
        const uint32_t pitch = live ? rowbytes : 0;
#pragma unroll
        for (int q = 0; q < NLD; ++q) {
            const uint32_t rows = WHOLE ? (uint32_t)(q * RPL) + (GLU && q * RPL >= 8 ? (uint32_t)R / 2 - 8 : 0u) : 0u;
            const uint8_t* at = base + (size_t)rows * pitch;
            r[q] = load_stream16(reinterpret_cast<const uint4*>(at + (live ? goff[WHOLE ? 0 : q] : 0u)));
        }
    };
    __builtin_amdgcn_sched_barrier(0);  // x ahead of the weights: loads come back in order
    request(0, raw[0]);
    __builtin_amdgcn_sched_barrier(0);
    request(1, raw[1]);
    __builtin_amdgcn_sched_barrier(0);

    auto turn = [&](int k, uint4 (&r)[NLD]) {
        const int tile = first + k * grid;
        if (ragged) {
#pragma unroll
            for (int q = 0; q < NLD; ++q)
                if (past >> q & 1) r[q] = make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < NLD; ++q) *reinterpret_cast<uint4*>(slab + (WHOLE ? loff[0] + q * RPL * STRIDE : loff[q])) = r[q];
        __builtin_amdgcn_sched_barrier(0);
        request(k + 2, r);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto product = [&](int i) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(slab + li * STRIDE + i * 64 + lg * 16);
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, xb[t][i]), acc[t], 0, 0, 0);
        };
        if (n == SPW) {
#pragma unroll
            for (int i = 0; i < SPW; ++i) product(i);
        } else {
#pragma unroll
            for (int i = 0; i < SPW; ++i)
                if (i < n) product(i);  // uniform
        }
        // the KS partial tiles, folded in wave order; two sets of partials alternate so one barrier a tile suffices
        f32x4* mine = part + (size_t)(k & 1) * KS * MT * WAVE;
#pragma unroll
        for (int t = 0; t < MT; ++t) mine[(wv * MT + t) * WAVE + lane] = acc[t];
        __syncthreads();
        if (wv < MT) {
            f32x4 s = mine[wv * WAVE + lane];
#pragma unroll
            for (int q = 1; q < KS; ++q) {
                const f32x4 o = mine[(q * MT + wv) * WAVE + lane];
                s.x += o.x;
                s.y += o.y;
                s.z += o.z;
                s.w += o.w;
            }
            const int m = wv * 16 + li;
            if constexpr (GLU) {
                // lanes of row groups 0, 1 hold gate sums, the lanes 32 further on the up sums of the same outputs
                const f32x4 up = f32x4{xor32(s.x), xor32(s.y), xor32(s.z), xor32(s.w)};
                if (m < M && lg < 2) {
                    // the arithmetic of the stand-alone fold over the two rounded outputs (silu_pair)
                    auto fold = [](float g, float u) {
                        const float gb = bfround(g), ub = bfround(u);
                        return f32_bf16(bfround(gb / (1.f + expf(-gb))) * ub);
                    };
                    // (the four outputs under one condition where no tiles overlap: one store)
                    const int row = row_of(tile) + lg * 4, own = tile * OUT;
                    uint16_t* o = y + (size_t)m * outs + row;
                    if (!RAG || row + 0 >= own) o[0] = fold(s.x, up.x);
                    if (!RAG || row + 1 >= own) o[1] = fold(s.y, up.y);
                    if (!RAG || row + 2 >= own) o[2] = fold(s.z, up.z);
                    if (!RAG || row + 3 >= own) o[3] = fold(s.w, up.w);
                }
            } else {
                const int in_tile = lg * 4, row = row_of(tile) + in_tile;
                const int own = RAG ? tile * TR : 0;  // the tile's own rows begin here
                if (m < M) {
                    uint16_t* o = y + (size_t)m * R + row;
                    if (in_tile + 0 < TR && row + 0 >= own) o[0] = f32_bf16(s.x);
                    if (in_tile + 1 < TR && row + 1 >= own) o[1] = f32_bf16(s.y);
                    if (in_tile + 2 < TR && row + 2 >= own) o[2] = f32_bf16(s.z);
                    if (in_tile + 3 < TR && row + 3 >= own) o[3] = f32_bf16(s.w);
                }
            }
        }
    };
    // (the odd last turn stands alone: leaving from the middle of the loop is, to the compiler, a way round it on which the
    // first buffer's loads are the newest, and it waits for everything)
    int k = 0;
    for (; k + 1 < turns; k += 2) {
        turn(k, raw[0]);
        turn(k + 1, raw[1]);
    }
    if (k < turns) turn(k, raw[0]);
}
// Two kernels: with the norm's arguments among them a launch's own lie on a second line of 64 bytes, another trip before the first
// load: 0.1 us of every launch ([6144 x 2560] 8 rows 8.95 -> 9.05 in a pass, the pass of 36 layers 2570 -> 2587).
template <int KS, int MT, int SPW, int TR, bool RAG, bool GLU>
__global__ void __launch_bounds__(KS * 64) mfma_ahead_kernel(const uint8_t* __restrict__ w, const uint4* __restrict__ x,
                                                             uint16_t* __restrict__ y, int R, int C, int M) {
    mfma_ahead<KS, MT, SPW, TR, RAG, GLU, false>(w, x, y, R, C, M, XArgs{});
}
template <int KS, int SPW, bool GLU>
__global__ void __launch_bounds__(KS * 64) mfma_ahead_norm_kernel(const uint8_t* __restrict__ w, uint16_t* __restrict__ y, int R,
                                                                  int C, int M, XArgs xa) {
    mfma_ahead<KS, 1, SPW, 16, true, GLU, true>(w, nullptr, y, R, C, M, xa);
}

template <int KS, int MT, int SPW, int TR, bool RAG, bool GLU, bool XN = false>
static int32_t launch_ahead(const void* w, const void* x, void* y, int R, int C, int M, int cap, hipStream_t st,
                            const XArgs& xa = XArgs{}) {
    constexpr int SLAB = 16 * (SPW * 64 + 16);
    size_t lds = (size_t)KS * SLAB + 2 * (size_t)KS * MT * WAVE * sizeof(f32x4);
    if (XN && 16 * ((size_t)C * 2 + 16) > lds) lds = 16 * ((size_t)C * 2 + 16);  // the made rows, before the slabs
    auto kern = [] {
        if constexpr (XN)
            return mfma_ahead_norm_kernel<KS, SPW, GLU>;
        else
            return mfma_ahead_kernel<KS, MT, SPW, TR, RAG, GLU>;
    }();
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return hip_status(e, "hipFuncSetAttribute");
    }
    const int ntiles = RAG ? (R + TR - 1) / TR : R / TR;
    // whole turns of the grid over the tiles: the smallest grid that walks them in ceil(ntiles / cap) turns
    const int turns = (ntiles + cap - 1) / cap, grid = (ntiles + turns - 1) / turns;
    if constexpr (XN)
        hipLaunchKernelGGL(kern, dim3(grid), dim3(KS * 64), lds, st, static_cast<const uint8_t*>(w), static_cast<uint16_t*>(y), R, C, M,
                           xa);
    else
        hipLaunchKernelGGL(kern, dim3(grid), dim3(KS * 64), lds, st, static_cast<const uint8_t*>(w), static_cast<const uint4*>(x),
                           static_cast<uint16_t*>(y), R, C, M);
    return hip_status(hipGetLastError(), "gemv_mfma_ahead launch");
}

template <int KS, int MT, int SPW>
static int32_t run_ahead(const void* w, const void* x, void* y, int R, int C, int M, bool glu, hipStream_t st) {
    // Eight waves a CU are what two tiles in flight leave registers for; a launch of one turn at twelve takes those (us at 8 rows,
    // eight / twelve waves: [9728 x 1024] 7.4 / 6.3, [40000 x 1024] 15.9 / 17.5). Not workgroups of two waves that hold more than
    // one short slice of x: the registers or the LDS of six of them a CU are not there, and the last ones begin when others end
    // (1000 shapes of 256 to 640 columns whose tiles are four to six a CU, twelve / eight, medians: slices of eight steps and one tile
    // of x rows 1 / 1.07, two 1 / 0.88; of ten steps 1 / 0.99 and 1 / 0.89). Four waves of any slice: 1 / 1.03 to 1 / 1.18.
    constexpr bool TWELVE = KS == 4 || (KS == 2 && MT == 1 && SPW == 8);
    int per_cu = tuning("mfma_wgs_per_cu");
    if (per_cu <= 0) per_cu = TWELVE && R <= 16 * (12 / KS) * device_info().cus ? 12 / KS : 8 / KS;
    const int cap = device_info().cus * per_cu;
    if (glu) {
        if (R % 16 != 0) return launch_ahead<KS, MT, SPW, 16, true, true>(w, x, y, R, C, M, cap, st);
        return launch_ahead<KS, MT, SPW, 16, false, true>(w, x, y, R, C, M, cap, st);
    }
    if (R % 16 != 0 && R % 12 != 0 && R % 10 != 0) return launch_ahead<KS, MT, SPW, 16, true, false>(w, x, y, R, C, M, cap, st);
    if constexpr (KS == 8) {
        if (tuning("mfma_tile_rows") != 0) {
            auto rows_of = [&](int t) { return (long)(((R + t - 1) / t + cap - 1) / cap) * t; };
            int tr = 16;
            if (R % 12 == 0 && rows_of(12) * 8 <= rows_of(16) * 7) tr = 12;
            if (R % 10 == 0 && rows_of(10) * 8 <= rows_of(16) * 7 && rows_of(10) < rows_of(tr)) tr = 10;
            if (tr == 12) return launch_ahead<KS, MT, SPW, 12, false, false>(w, x, y, R, C, M, cap, st);
            if (tr == 10) return launch_ahead<KS, MT, SPW, 10, false, false>(w, x, y, R, C, M, cap, st);
        }
    }
    if (R % 16 != 0) return launch_ahead<KS, MT, SPW, 16, true, false>(w, x, y, R, C, M, cap, st);
    return launch_ahead<KS, MT, SPW, 16, false, false>(w, x, y, R, C, M, cap, st);
}

// Which shapes. Measured on MI355X, us a launch, gemv_mfma_lds / this at 8, 16, 17, 32 rows of x: [19456 x 2560] with the fold
// 20.6 / 18.9, 21.7 / 19.7, 22.5 / 20.7, 24.4 / 22.1 (4.5 TB/s); [151936 x 2560] 131.8 / 125.5, 144.7 / 132.0, 148.5 / 135.0,
// 163.9 / 144.2; [6144 x 2560] 9.2 / 8.9, 10.5 / 9.5, 10.9 / 10.2, 13.0 / 11.9; [1024 x 1280] 4.7 / 3.8, 4.9 / 4.0, 5.6 / 4.5,
// 6.4 / 5.1; [40000 x 1024] 18.9 / 15.9, 20.0 / 16.5, 22.6 / 17.0, 25.3 / 19.4; [512 x 512] 3.3 / 2.7, 3.4 / 2.8, 3.8 / 3.0,
// 3.9 / 3.2. Past 2560 columns that kernel has two full sub-blocks a tile and the x fragments of a second tile of x rows do not
// fit beside two tiles of weights: up to 16 rows of x, and where the CUs go round once ([2560 x 4096] at 8 rows 7.9 / 7.2,
// [2048 x 3072] 6.7 / 6.0; but [24576 x 4096] 35.8 / 36.5, [8192 x 3072] 12.1 / 12.4), with slices of twelve steps or all of sixteen
// ([4096 x 3584], fourteen, at 5 / 8 / 16 rows 8.45 / 8.56, 8.73 / 8.85, 9.55 / 9.79).
bool mfma_ahead_fits(int R, int C, int M, bool glu) {
    const int nsteps = C / 32, cus = device_info().cus;
    if (tuning("mfma_ahead") == 0 || R < 16 || C % 32 != 0 || nsteps > 128 || (glu && R % 16 != 0)) return false;
    if (glu && (uint64_t)R * C >= 1ull << 31) return false;  // a gate row's up row within 32 bits
    if (tuning("mfma_ahead") > 0) return nsteps <= 80 ? M <= 32 : M <= 16;
    if (nsteps > 80) return M <= 16 && R <= 16 * cus && (nsteps <= 96 || nsteps > 120);
    // Slices of the kernel's eight steps or fewer. What it gains by two tiles in flight it gains in long launches and, with two or
    // four waves a workgroup, in those of at most half a turn of eight waves a CU. In between nothing of the second tile is
    // ahead, and a slice of four to seven steps still loads and stores all eight. 6600 shapes, medians of the time against
    // gemv_mfma_lds's by turns (to half a turn, to two, more), one tile of x rows / two: short slices of two waves 0.92 / 0.89, 1.03 /
    // 1.03, 1.00 / 0.86, of four 0.98 / 0.98, 1.04 / 1.05, 0.95 / 0.85, of eight 1.03 / 1.06, 1.04 / 1.06, 0.88 / 0.91; whole ones 0.97 /
    // 0.95, 0.99 / 0.97, 0.92 / 0.86 (nine and ten steps 0.90 / 0.95, 0.94 / 0.95, 0.89 / 0.82). With the fold 0.03 to 0.06
    // more: two waves' short slices then pay to a quarter of a turn, and slices of nine steps not between one turn and two ([18816 x
    // 544] 5 rows 7.4 / 8.2).
    const int ks = nsteps <= 20 ? 2 : nsteps <= 40 ? 4 : 8, steps = (nsteps + ks - 1) / ks;
    const int64_t waves = (int64_t)((R + 15) / 16) * ks;
    if (M > 32) return false;
    if (steps > 8) return !(glu && steps == 9 && M <= 16 && waves > 8 * cus && waves <= 16 * cus);
    if (waves > 16 * cus) return M > 16 || ks != 2 || steps == 8;
    if (steps == 8) return !glu || ks == 2;
    return glu ? ks == 2 && waves <= 2 * cus : ks < 8 && waves <= 4 * cus;
}
// Rows of a multiple of 8 columns but not of 32, which the other matrix-core kernels do not take and which went through passes
// of four rows on the vector units: from five rows of x on, in passes of 32 rows, or of 16 past 2560 columns. us at 5 / 8 / 16 / 32
// rows, those passes / here: [512 x 520] 4.5 / 3.2, 5.2 / 3.3, 10.0 / 3.4, 19.5 / 3.9; [2560 x 2056] 9.0 / 5.4, 9.8 / 5.5, 18.8 / 5.9,
// 37.7 / 7.5; [5003 x 3000] 16.1 / 11.3, 17.3 / 11.5, 32.3 / 11.7, 63.8 / 23.0; [40000 x 3000] 84 / 43, 85 / 44, 168 / 45, 318 / 87
// (5.5 TB/s); [512 x 4088] 7.1 / 6.5, 8.6 / 6.7, 16.6 / 7.7, 32.8 / 14.8. The gate / up fold and the add + norm go with it, or their
// sums would be in another order than the matvec's: at 5 / 8 / 16 rows the fold [2560 x 520] 7.4 / 4.5, 8.7 / 4.5, 16.6 / 4.5,
// [8192 x 2056] 17.7 / 11.3, 19.1 / 11.3, 37.8 / 12.0; the norm [2560 x 520] 8.9 / 8.2, 11.4 / 8.2, 22.3 / 12.1, [1000 x 1016] 8.7 /
// 9.0, 11.3 / 9.0, 21.9 / 9.2, [8192 x 2056] 22.0 / 14.4, 28.5 / 14.8, 55.3 / 18.9, [512 x 4088] 14.6 / 12.8, 22.6 / 13.1, 44.8 / 19.8.
bool mfma_ahead_ragged_fits(int R, int C) {
    return R >= 16 && C % 32 != 0 && C % 8 == 0 && C >= 64 && C <= 4096 &&
           (uint64_t)R * C < 1ull << 31;  // a gate row's up row within 32 bits
}
// the waves a tile by row length as gemv_mfma_lds has them (two, four or eight), the slice's size close above its steps
int32_t gemv_mfma_ahead_bf16(const void* w, const void* x, void* y, int R, int C, int M, bool glu, hipStream_t st) {
    const int nsteps = (C + 31) / 32;
#define BTB_AHEAD(KS_, SPW_) \
    return M <= 16 ? run_ahead<KS_, 1, SPW_>(w, x, y, R, C, M, glu, st) : run_ahead<KS_, 2, SPW_>(w, x, y, R, C, M, glu, st)
    if (nsteps <= 16) BTB_AHEAD(2, 8);
    if (nsteps <= 20) BTB_AHEAD(2, 10);
    if (nsteps <= 32) BTB_AHEAD(4, 8);
    if (nsteps <= 40) BTB_AHEAD(4, 10);
    if (nsteps <= 64) BTB_AHEAD(8, 8);
    if (nsteps <= 80) BTB_AHEAD(8, 10);
#undef BTB_AHEAD
    if (nsteps <= 96) return run_ahead<8, 1, 12>(w, x, y, R, C, M, glu, st);
    return run_ahead<8, 1, 16>(w, x, y, R, C, M, glu, st);
}

// ... with x made by the residual add and RMSNorm, for the ragged rows (mfma_ahead_ragged_fits): up to sixteen rows of the
// residual stream
template <int KS, int SPW>
static int32_t run_ahead_norm(const void* w, const XArgs& xa, void* y, int R, int C, int M, bool glu, hipStream_t st) {
    const int cap = device_info().cus * (8 / KS);
    if (glu) return launch_ahead<KS, 1, SPW, 16, true, true, true>(w, nullptr, y, R, C, M, cap, st, xa);
    return launch_ahead<KS, 1, SPW, 16, true, false, true>(w, nullptr, y, R, C, M, cap, st, xa);
}
int32_t gemv_mfma_ahead_norm_bf16(const void* w, const XArgs& xa, void* y, int R, int C, int M, bool glu, hipStream_t st) {
    const int nsteps = (C + 31) / 32;
    if (nsteps <= 16) return run_ahead_norm<2, 8>(w, xa, y, R, C, M, glu, st);
    if (nsteps <= 20) return run_ahead_norm<2, 10>(w, xa, y, R, C, M, glu, st);
    if (nsteps <= 32) return run_ahead_norm<4, 8>(w, xa, y, R, C, M, glu, st);
    if (nsteps <= 40) return run_ahead_norm<4, 10>(w, xa, y, R, C, M, glu, st);
    if (nsteps <= 64) return run_ahead_norm<8, 8>(w, xa, y, R, C, M, glu, st);
    if (nsteps <= 80) return run_ahead_norm<8, 10>(w, xa, y, R, C, M, glu, st);
    if (nsteps <= 96) return run_ahead_norm<8, 12>(w, xa, y, R, C, M, glu, st);
    return run_ahead_norm<8, 16>(w, xa, y, R, C, M, glu, st);
}

}  // namespace btb
