// A bf16 tensor into its 12-bit form on the GPU (the reference packs in torch: btb/pack12.py:48-67): the bytes that
// `pack12.pack_bf16` writes, in five launches where that is thirty-odd passes over the tensor.
//
//   1. p12_clear_kernel, p12_hist_kernel   how often each high byte occurs (reads 2 B a weight)
//   2. p12_table_kernel   the table: the 15 most frequent high bytes, equal counts by ascending byte value; with it the
//                         pair table, the byte -> code map and the number of escapes (n less what the table covers)
//   3. p12_encode_kernel  low bytes and codes (2 B read, 1.5 B written a weight), escapes counted a chunk of 2048
//                         and listed a workgroup of sixteen chunks as they are met
//   4. p12_emit_kernel    the workgroups' lists end to end, and every row's first entry; a workgroup whose list was too
//                         long to keep is read out of its codes (0.5 B a weight)
//
// The list's length has to be known on the host before the list can be allocated. It is known after the table's launch, so
// the host waits for that one (an event) while the encoder is already queued behind it.
//
// Bound: HBM, 2 + 2 + 1.5 B a weight; the second read of a tensor that fits the 256 MB last-level cache comes out
// of that. [19456 x 2560] packed, with its rows' words, and widened back: 1456 us with the packing in torch, 103 in these
// launches with every list read out of the codes (15 us of it), 92 with the lists kept (4).

#include "btb_common.hpp"
#include "btb_formats.hpp"
#include "btb_tuning.hpp"

#include "../../include/btb_hip.h"

namespace btb {

constexpr int P12_CHUNK = 2048;          // weights a wave encodes at a time: four 16-byte loads a lane
constexpr int P12_BLOCK = 16;            // chunks a workgroup: four waves, four chunks each
constexpr int P12_WAVE_LIST = 64;        // escapes a wave of the encoder lists (its four chunks of a matrix of weights hold two)
constexpr int P12_LIST = 4 * P12_WAVE_LIST;
constexpr uint32_t P12_LISTED = 0x80000000u;  // of a workgroup's count: the list holds its escapes
constexpr int P12_COPIES = 32;           // copies of each LDS counter, one a lane of a half wave: no two lanes meet
// words of the workspace: the counters, the byte -> code map, then a count a workgroup of chunks, a count a chunk and a
// list a workgroup: low byte | high byte << 8 | place among the workgroup's weights << 16
constexpr int P12_HIST = 0, P12_CODES = 256, P12_BLOCKS = 256 + 64;
static size_t p12_chunks(size_t n) { return (n + P12_CHUNK - 1) / P12_CHUNK; }
static size_t p12_blocks(size_t n) { return (p12_chunks(n) + P12_BLOCK - 1) / P12_BLOCK; }

__global__ void __launch_bounds__(256) p12_clear_kernel(uint32_t* __restrict__ hist) { hist[threadIdx.x] = 0; }

// Every lane of a half wave adds into its own copy of the counter, so the LDS unit serves an add without a conflict
// however few distinct bytes there are (a trained or random matrix has about ten); one counter a byte would serialise
// on them. A workgroup's non-zero sums go to memory as one atomic add each. [19456 x 2560]: 27 us for 99.6 MB, bound by
// the LDS unit's adds - one to eight workgroups a CU and 64 copies instead of 32 all take 27 - 29 us.
__global__ void __launch_bounds__(512) p12_hist_kernel(const uint4* __restrict__ t, size_t n, uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[256 * P12_COPIES];
    const int tid = threadIdx.x;
    for (int i = tid; i < 256 * P12_COPIES; i += 512) cnt[i] = 0;
    __syncthreads();
    const uint32_t copy = tid & (P12_COPIES - 1);
    auto add = [&](uint32_t w) {  // the two high bytes of a dword
        atomicAdd(&cnt[((w >> 8) & 255u) * P12_COPIES + copy], 1u);
        atomicAdd(&cnt[(w >> 24) * P12_COPIES + copy], 1u);
    };
    const size_t units = n / 8, step = (size_t)gridDim.x * 512;
    size_t u = (size_t)blockIdx.x * 512 + tid;
    for (; u + 3 * step < units; u += 4 * step) {
        uint4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = t[u + k * step];
#pragma unroll
        for (int k = 0; k < 4; ++k) add(v[k].x), add(v[k].y), add(v[k].z), add(v[k].w);
    }
    for (; u < units; u += step) {
        const uint4 v = t[u];
        add(v.x), add(v.y), add(v.z), add(v.w);
    }
    if (blockIdx.x == 0 && tid == 0) {
        const uint16_t* s = reinterpret_cast<const uint16_t*>(t);
        for (size_t i = units * 8; i < n; ++i) atomicAdd(&cnt[(uint32_t)(s[i] >> 8) * P12_COPIES + copy], 1u);
    }
    __syncthreads();
    if (tid < 256) {
        uint32_t s = 0;
#pragma unroll 8
        for (int k = 0; k < P12_COPIES; ++k) s += cnt[tid * P12_COPIES + ((k + tid) & (P12_COPIES - 1))];
        if (s != 0) atomicAdd(&hist[tid], s);
    }
}

// One workgroup: a byte's rank is how many bytes come before it by (count descending, byte ascending). Only the bytes
// that occur are compared - about thirty of a matrix of weights -, gathered first in ascending order.
__global__ void __launch_bounds__(256) p12_table_kernel(const uint32_t* __restrict__ hist, uint32_t n,
                                                        uint8_t* __restrict__ table, uint16_t* __restrict__ pairs,
                                                        uint8_t* __restrict__ codes, int32_t* __restrict__ total) {
    __shared__ __align__(16) uint2 live[256];  // (count, byte), count 0 past the last
    __shared__ uint32_t in_wave[4], tab[16], covered[16];
    const uint32_t b = threadIdx.x, lane = b & 63, wave = b >> 6;
    const uint32_t mine = hist[b];
    const uint64_t m = __ballot(mine != 0);
    if (lane == 0) in_wave[wave] = (uint32_t)__popcll(m);
    if (b < 16) tab[b] = 0, covered[b] = 0;
    live[b] = make_uint2(0, 0);
    __syncthreads();
    uint32_t at = (uint32_t)__popcll(m & ((1ull << lane) - 1));
    for (uint32_t w = 0; w < wave; ++w) at += in_wave[w];
    const uint32_t n_live = in_wave[0] + in_wave[1] + in_wave[2] + in_wave[3];
    if (mine != 0) live[at] = make_uint2(mine, b);
    __syncthreads();
    uint32_t rank = 0;
    for (uint32_t o = 0; o < n_live; o += 4) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint2 c = live[o + k];
            rank += c.x > mine || (c.x == mine && c.y < b) ? 1 : 0;
        }
    }
    const bool in = mine != 0 && rank < 15;
    if (in) tab[rank] = b, covered[rank] = mine;
    codes[b] = (uint8_t)(in ? rank : 15);
    __syncthreads();
    if (b < 16) table[b] = (uint8_t)tab[b];
    pairs[b] = (uint16_t)(tab[b & 15u] | (tab[b >> 4] << 8));  // slot 15 holds 0
    if (b == 0) {
        uint32_t s = 0;
        for (int k = 0; k < 15; ++k) s += covered[k];
        *total = (int32_t)(n - s);
    }
}

// the marks of the escape code (15) among a dword's eight codes: bit 4 i of code i
__device__ __forceinline__ uint32_t escape_marks(uint32_t codes) {
    const uint32_t a = codes & (codes >> 1);
    return a & (a >> 2) & 0x11111111u;
}

// A wave takes chunks of 2048 weights, four 16-byte loads a lane; codes by one LDS read a weight (a map of 64 words: the
// few bytes that occur are broadcasts). 28 us for [19456 x 2560]: 174 MB at 6.2 TB/s.
__global__ void __launch_bounds__(256) p12_encode_kernel(const uint4* __restrict__ t, size_t n,
                                                         const uint32_t* __restrict__ code_map, uint2* __restrict__ lo,
                                                         uint32_t* __restrict__ hi4, uint32_t* __restrict__ block_counts,
                                                         uint32_t* __restrict__ counts, uint32_t* __restrict__ lists) {
    __shared__ uint32_t map32[64];
    __shared__ uint32_t sums[4];
    __shared__ uint32_t found[4][P12_WAVE_LIST];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t units = n / 8;
    if (tid < 64) map32[tid] = code_map[tid];
    __syncthreads();
    const uint8_t* map = reinterpret_cast<const uint8_t*>(map32);
    const size_t chunks = (n + P12_CHUNK - 1) / P12_CHUNK;
    uint32_t wave_total = 0;
    for (int k = 0; k < P12_BLOCK / 4; ++k) {
        const size_t chunk = (size_t)blockIdx.x * P12_BLOCK + wave * (P12_BLOCK / 4) + k;
        if (chunk >= chunks) break;
        const size_t u0 = chunk * (P12_CHUNK / 8) + lane;
        uint4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = units > 0 ? t[min(u0 + 64 * j, units - 1)] : make_uint4(0, 0, 0, 0);
        uint32_t total = 0;  // the chunk's escapes, the same in every lane
        const uint32_t place0 = (uint32_t)(wave * (P12_BLOCK / 4) + k) * P12_CHUNK;  // the chunk among the workgroup's weights
        auto list = [&](uint32_t at, uint32_t place, uint32_t weight) {
            if (at < P12_WAVE_LIST) found[wave][at] = weight | (place << 16);
        };
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const size_t u = u0 + 64 * j;
            const uint32_t h0 = __builtin_amdgcn_perm(v[j].y, v[j].x, 0x07050301u);  // the high bytes, four a dword
            const uint32_t h1 = __builtin_amdgcn_perm(v[j].w, v[j].z, 0x07050301u);
            uint32_t c = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                c |= (uint32_t)map[(h0 >> (8 * e)) & 255u] << (4 * e);
                c |= (uint32_t)map[(h1 >> (8 * e)) & 255u] << (4 * e + 16);
            }
            const uint32_t marks = u < units ? escape_marks(c) : 0u;
            if (u < units) {
                lo[u] = make_uint2(__builtin_amdgcn_perm(v[j].y, v[j].x, 0x06040200u),
                                   __builtin_amdgcn_perm(v[j].w, v[j].z, 0x06040200u));
                hi4[u] = c;
            }
            if (__ballot(marks != 0) != 0) {  // rare: the lanes' escapes in ascending order
                const uint32_t m = (uint32_t)__popc(marks);  // 0 .. 8 a lane: four bits, a ballot each
                uint32_t before = 0, all = 0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint64_t w = __ballot((m >> b) & 1u);
                    before += (uint32_t)__popcll(w & ((1ull << lane) - 1)) << b;
                    all += (uint32_t)__popcll(w) << b;
                }
                uint32_t at = wave_total + total + before;
                for (uint32_t left = marks; left != 0; left &= left - 1, ++at) {
                    const uint32_t e = (uint32_t)(__ffs((int)left) - 1) / 4;
                    const uint32_t lo2 = e & 2 ? v[j].y : v[j].x, hi2 = e & 2 ? v[j].w : v[j].z;
                    const uint32_t pair = e & 4 ? hi2 : lo2;
                    list(at, place0 + (uint32_t)(64 * j + lane) * 8 + e, e & 1 ? pair >> 16 : pair & 0xFFFFu);
                }
                total += all;
            }
        }
        // the tail (n % 8 weights) belongs to the last chunk: its first lane takes it, a code byte a pair
        if (chunk == chunks - 1 && units * 8 < n) {
            uint32_t tail = 0;
            if (lane == 0) {
                const uint16_t* s = reinterpret_cast<const uint16_t*>(t);
                uint8_t* lo8 = reinterpret_cast<uint8_t*>(lo);
                uint8_t* hi8 = reinterpret_cast<uint8_t*>(hi4);
                for (size_t i = units * 8; i < n; i += 2) {
                    uint32_t c = 0;
                    for (size_t e = i; e < min(i + 2, n); ++e) {
                        lo8[e] = (uint8_t)s[e];
                        const uint32_t m = map[s[e] >> 8];
                        c |= m << (4 * (e - i));
                        if (m == 15u) list(wave_total + total + tail++, place0 + (uint32_t)(e - chunk * P12_CHUNK), s[e]);
                    }
                    hi8[i / 2] = (uint8_t)c;
                }
            }
            total += __builtin_amdgcn_readfirstlane(tail);
        }
        if (lane == 0) counts[chunk] = total;
        wave_total += total;
    }
    if (lane == 0) sums[wave] = wave_total;
    __syncthreads();
    const bool listed = max(max(sums[0], sums[1]), max(sums[2], sums[3])) <= P12_WAVE_LIST;
    uint32_t first = 0;
    for (int w = 0; w < wave; ++w) first += sums[w];
    if (listed && lane < (int)wave_total) lists[(size_t)blockIdx.x * P12_LIST + first + lane] = found[wave][lane];
    if (tid == 0) block_counts[blockIdx.x] = (sums[0] + sums[1] + sums[2] + sums[3]) | (listed ? P12_LISTED : 0u);
}

// The escape list. A workgroup takes the chunks one of the encoding workgroups took; where its part of the list begins is the
// sum of those workgroups' counts before it. Where the encoder kept its escapes they are copied, and a row's first entry
// (row_ptr, for the rows whose first weight lies here) is a search among them: [19456 x 2560] 15 us -> 4. Else they come
// out of the codes, a chain of three trips to memory - codes, the escapes' weights, the stores.
__global__ void __launch_bounds__(256) p12_emit_kernel(const uint16_t* __restrict__ t, const uint8_t* __restrict__ hi4,
                                                       size_t n, const uint32_t* __restrict__ block_counts,
                                                       const uint32_t* __restrict__ counts,
                                                       const uint32_t* __restrict__ lists, size_t n_esc,
                                                       int32_t* __restrict__ esc_idx, uint8_t* __restrict__ esc_val,
                                                       size_t cols, size_t rows, int32_t* __restrict__ row_ptr) {
    __shared__ uint32_t part[4];
    __shared__ uint32_t kept[P12_LIST];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t chunks = (n + P12_CHUNK - 1) / P12_CHUNK;
    const uint32_t here_all = block_counts[blockIdx.x];
    const uint32_t entry = lists[(size_t)blockIdx.x * P12_LIST + tid];  // past the count: whatever lies there, unused
    uint32_t s = 0;
#pragma unroll 4
    for (size_t i = tid; i < blockIdx.x; i += 256) s += block_counts[i] & ~P12_LISTED;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s += __shfl_xor(s, d, WAVE);
    if (lane == 0) part[wave] = s;
    if (here_all & P12_LISTED) {  // uniform
        const uint32_t count = here_all & ~P12_LISTED;
        kept[tid] = entry >> 16;
        __syncthreads();
        const uint32_t base = part[0] + part[1] + part[2] + part[3];
        const size_t b0 = (size_t)blockIdx.x * P12_BLOCK * P12_CHUNK, b1 = min(b0 + (size_t)P12_BLOCK * P12_CHUNK, n);
        if (tid < (int)count && base + tid < n_esc) {
            esc_idx[base + tid] = (int32_t)(b0 + (entry >> 16));
            esc_val[base + tid] = (uint8_t)(entry >> 8);
        }
        const uint32_t r0 = ((uint32_t)b0 + (uint32_t)cols - 1) / (uint32_t)cols;  // below 2^32: n and cols are below 2^31
        for (size_t r = r0 + (size_t)tid; r < rows && r * cols < b1; r += 256) {
            const uint32_t o = (uint32_t)(r * cols - b0);  // the row's first weight among the workgroup's
            uint32_t below = 0, above = count;
            while (below < above) {
                const uint32_t mid = (below + above) / 2;
                if (kept[mid] < o)
                    below = mid + 1;
                else
                    above = mid;
            }
            row_ptr[r] = (int32_t)(base + below);
        }
        if (rows != 0 && b1 == n && tid == 0) row_ptr[rows] = (int32_t)n_esc;
        return;
    }
    const size_t mine = (size_t)blockIdx.x * P12_BLOCK + (size_t)wave * (P12_BLOCK / 4);
    // everything that does not depend on anything is asked for first: the wave's codes, the counts
    uint32_t marks[P12_BLOCK / 4][4];
#pragma unroll
    for (int k = 0; k < P12_BLOCK / 4; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const size_t i = (mine + k) * P12_CHUNK + (size_t)(64 * j + lane) * 8;  // the lane's eight weights of a stretch
            marks[k][j] = i + 8 <= n ? escape_marks(*reinterpret_cast<const uint32_t*>(hi4 + i / 2)) : 0;
        }
    const size_t c16 = (size_t)blockIdx.x * P12_BLOCK + (lane & (P12_BLOCK - 1));
    const uint32_t count16 = c16 < chunks ? counts[c16] : 0;  // lane l: the count of the workgroup's chunk l % 16
    __syncthreads();
    uint32_t base = part[0] + part[1] + part[2] + part[3];
    for (int c = 0; c < wave * (P12_BLOCK / 4); ++c) base += __builtin_amdgcn_readlane(count16, c);
#pragma unroll
    for (int k = 0; k < P12_BLOCK / 4; ++k) {
        const size_t chunk = mine + k;
        if (chunk >= chunks) break;
        const size_t c0 = chunk * P12_CHUNK, c1 = min(c0 + P12_CHUNK, n);
        const uint32_t here = __builtin_amdgcn_readlane(count16, wave * (P12_BLOCK / 4) + k);
        if (here != 0) {
            if (c1 == n) {  // the tail (n % 8 weights)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const size_t i = c0 + (size_t)(64 * j + lane) * 8;
                    if (i < n && i + 8 > n)
                        for (size_t e = i; e < n; ++e)
                            if (((hi4[e / 2] >> (4 * (e & 1))) & 15u) == 15u) marks[k][j] |= 1u << (4 * (e - i));
                }
            }
            uint32_t at = base;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t m = (uint32_t)__popc(marks[k][j]);  // 0 .. 8 a lane: four bits, a ballot each
                if (__ballot(m != 0) == 0) continue;
                uint32_t before = 0, all = 0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint64_t v = __ballot((m >> b) & 1u);
                    before += (uint32_t)__popcll(v & ((1ull << lane) - 1)) << b;
                    all += (uint32_t)__popcll(v) << b;
                }
                uint32_t o = at + before;
                for (uint32_t left = marks[k][j]; left != 0; left &= left - 1, ++o) {
                    const size_t i = c0 + (size_t)(64 * j + lane) * 8 + (__ffs((int)left) - 1) / 4;
                    if (o < n_esc) {
                        esc_idx[o] = (int32_t)i;
                        esc_val[o] = (uint8_t)(t[i] >> 8);
                    }
                }
                at += all;
            }
        }
        const uint32_t r0 = ((uint32_t)c0 + (uint32_t)cols - 1) / (uint32_t)cols;  // below 2^32: n and cols are below 2^31
        for (size_t r = r0; r < rows && r * cols < c1; ++r) {
            const int o = (int)(r * cols - c0);  // the row's first weight within the chunk
            uint32_t below = 0;
            if (here != 0) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k8 = min(max(o - (64 * j + lane) * 8, 0), 8);
                    below += (uint32_t)__popc(k8 == 8 ? marks[k][j] : marks[k][j] & ((1u << (4 * k8)) - 1));
                }
#pragma unroll
                for (int d = 32; d > 0; d >>= 1) below += __shfl_xor(below, d, WAVE);
            }
            if (lane == 0) row_ptr[r] = (int32_t)(base + below);
        }
        if (rows != 0 && chunk == chunks - 1 && lane == 0) row_ptr[rows] = (int32_t)n_esc;
        base += here;
    }
}

}  // namespace btb

using namespace btb;

extern "C" {

size_t btb_hip_p12_pack_words(size_t n) { return P12_BLOCKS + p12_blocks(n) * (1 + P12_LIST) + p12_chunks(n); }

int32_t btb_hip_p12_pack(const void* t, size_t n, void* lo, void* hi4, void* table, void* pairs, void* work,
                         int32_t* host_total, void* stream) {
    if (t == nullptr || lo == nullptr || hi4 == nullptr || table == nullptr || pairs == nullptr || work == nullptr ||
        host_total == nullptr)
        return ERR_NULL;
    if (n == 0 || n > 0x7FFFFFFFull) return ERR_DOMAIN;
    auto al = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
    if (!al(t, 16) || !al(lo, 8) || !al(hi4, 4) || !al(pairs, 2) || !al(work, 4) || !al(host_total, 4)) return ERR_DOMAIN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint32_t* w = static_cast<uint32_t*>(work);
    hipEvent_t ready;
    hipError_t e = hipEventCreateWithFlags(&ready, hipEventDisableTiming);
    if (e != hipSuccess) return hip_status(e, "p12_pack event");
    hipLaunchKernelGGL(p12_clear_kernel, dim3(1), dim3(256), 0, st, w + P12_HIST);
    // one workgroup of eight waves a CU at most, four loads a lane in flight (two: 28.2 against 27.0 us)
    const size_t want = (n / 8 + 4 * 512 - 1) / (4 * 512);
    const size_t hg = (size_t)device_info().cus;
    const unsigned hist_grid = (unsigned)(want < 1 ? 1 : want < hg ? want : hg);
    hipLaunchKernelGGL(p12_hist_kernel, dim3(hist_grid), dim3(512), 0, st, static_cast<const uint4*>(t), n, w + P12_HIST);
    hipLaunchKernelGGL(p12_table_kernel, dim3(1), dim3(256), 0, st, w + P12_HIST, (uint32_t)n,
                       static_cast<uint8_t*>(table), static_cast<uint16_t*>(pairs),
                       reinterpret_cast<uint8_t*>(w + P12_CODES), host_total);
    e = hipEventRecord(ready, st);
    const size_t blocks = p12_blocks(n);
    hipLaunchKernelGGL(p12_encode_kernel, dim3((unsigned)blocks), dim3(256), 0, st, static_cast<const uint4*>(t), n,
                       w + P12_CODES, static_cast<uint2*>(lo), static_cast<uint32_t*>(hi4),
                       w + P12_BLOCKS, w + P12_BLOCKS + blocks, w + P12_BLOCKS + blocks + p12_chunks(n));
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipEventSynchronize(ready);
    (void)hipEventDestroy(ready);
    return hip_status(e, "p12_pack");
}

int32_t btb_hip_p12_emit(const void* t, const void* hi4, size_t n, const void* work, size_t n_esc, void* esc_idx,
                         void* esc_val, size_t rows, size_t cols, void* row_ptr, void* stream) {
    if (t == nullptr || hi4 == nullptr || work == nullptr) return ERR_NULL;
    if (n_esc > 0 && (esc_idx == nullptr || esc_val == nullptr)) return ERR_NULL;
    if (n == 0 || n > 0x7FFFFFFFull || n_esc > n) return ERR_DOMAIN;
    if (row_ptr != nullptr && (rows == 0 || cols == 0 || rows > n || cols > n || rows * cols != n)) return ERR_DOMAIN;
    auto al = [](const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
    if (!al(t, 2) || !al(hi4, 4) || !al(work, 4) || !al(esc_idx, 4) || !al(row_ptr, 4)) return ERR_DOMAIN;
    if (n_esc == 0 && row_ptr == nullptr) return OK;
    const size_t blocks = p12_blocks(n);
    hipLaunchKernelGGL(p12_emit_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(t), static_cast<const uint8_t*>(hi4), n,
                       static_cast<const uint32_t*>(work) + P12_BLOCKS,
                       static_cast<const uint32_t*>(work) + P12_BLOCKS + blocks,
                       static_cast<const uint32_t*>(work) + P12_BLOCKS + blocks + p12_chunks(n), n_esc,
                       static_cast<int32_t*>(esc_idx),
                       static_cast<uint8_t*>(esc_val), row_ptr != nullptr ? cols : 1, row_ptr != nullptr ? rows : 0,
                       static_cast<int32_t*>(row_ptr));
    return hip_status(hipGetLastError(), "p12_emit launch");
}

}  // extern "C"
