// device_sort.h -- stable LSD radix sort of (uint32 key, uint32 value)
// pairs for the commit-time device kernels (bvh_device.hip,
// mesh_device.hip).  8-bit passes over the key bits in use.  A workgroup
// owns a tile of kSortTile pairs, each of its waves a contiguous quarter:
//   hist      digit counts of every tile, [digit][tile]
//   scan      one workgroup per digit: exclusive prefix over the tiles, and
//             the digit's total
//   scatter   a pair's place = pairs of smaller digits (scan of the totals)
//             + of its digit in earlier tiles, earlier waves, earlier rounds
//             of its wave and lower lanes; the last from 8 ballots
// so equal keys keep their input order.  A pass moves a few megabytes at
// commit-time sizes and is bound by its three launches, each a single wave of
// workgroups: the Morton codes of 200 K triangles and their 600 K corners, 7
// passes in all, take 0.11 ms (MI355X).  One lane walking 256 pairs in order
// with the scan in one workgroup, always four passes, took 9.25 ms.
#ifndef OMV_DEVICE_SORT_H
#define OMV_DEVICE_SORT_H

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

namespace {

constexpr int kSortBlock = 256;                        // = digits of a pass
constexpr int kSortWaves = kSortBlock / 64;
constexpr int kSortRounds = 4;                         // pairs per lane
constexpr int kSortTile = kSortBlock * kSortRounds;

// exclusive prefix of x over the workgroup; `all` becomes the sum
__device__ inline uint32_t sortBlockScan(uint32_t x, uint32_t* waveSum, uint32_t& all) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = x;
    for (int s = 1; s < 64; s <<= 1) {
        const uint32_t y = __shfl_up(inc, s);
        if (lane >= s) inc += y;
    }
    __syncthreads();   // waveSum may still be read from the scan before
    if (lane == 63) waveSum[wave] = inc;
    __syncthreads();
    uint32_t before = 0;
    all = 0;
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t s = waveSum[w];
        if (w < wave) before += s;
        all += s;
    }
    return before + inc - x;
}

__global__ __launch_bounds__(kSortBlock) void sortHist(const uint32_t* __restrict__ key, uint32_t n, int shift, uint32_t ntiles,
                                                       uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[kSortBlock];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t i = blockIdx.x * kSortTile + r * kSortBlock + threadIdx.x;
        if (i < n) atomicAdd(&cnt[(key[i] >> shift) & 0xFFu], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(kSortBlock) void sortScan(uint32_t* __restrict__ hist, uint32_t ntiles, uint32_t* __restrict__ total) {
    __shared__ uint32_t waveSum[kSortWaves];
    uint32_t* a = hist + (size_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (uint32_t t0 = 0; t0 < ntiles; t0 += kSortBlock) {
        const uint32_t t = t0 + threadIdx.x;
        uint32_t all;
        const uint32_t before = sortBlockScan(t < ntiles ? a[t] : 0u, waveSum, all);
        if (t < ntiles) a[t] = carry + before;
        carry += all;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

__global__ __launch_bounds__(kSortBlock) void sortScatter(const uint32_t* __restrict__ key, const uint32_t* __restrict__ val, uint32_t n,
                                                          int shift, uint32_t ntiles, const uint32_t* __restrict__ hist,
                                                          const uint32_t* __restrict__ total, uint32_t* __restrict__ keyOut,
                                                          uint32_t* __restrict__ valOut) {
    __shared__ uint32_t cnt[kSortWaves][kSortBlock], waveSum[kSortWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int w = 0; w < kSortWaves; ++w) cnt[w][threadIdx.x] = 0;
    __syncthreads();
    const uint32_t i0 = blockIdx.x * kSortTile + wave * (kSortTile / kSortWaves) + lane;
    uint32_t k[kSortRounds], v[kSortRounds], rank[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t i = i0 + 64 * r;
        k[r] = i < n ? key[i] : 0u;
        v[r] = i < n ? val[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const bool valid = i0 + 64 * r < n;
        const uint32_t d = (k[r] >> shift) & 0xFFu;
        uint64_t same = __ballot(valid);   // lanes of this digit
        for (int b = 0; b < 8; ++b) {
            const uint64_t ones = __ballot((d >> b) & 1u);
            same &= ((d >> b) & 1u) ? ones : ~ones;
        }
        const uint32_t lower = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        const uint32_t base = cnt[wave][d];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && lower == 0) cnt[wave][d] = base + (uint32_t)__popcll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        rank[r] = base + lower;
    }
    __syncthreads();
    uint32_t all;
    uint32_t run = sortBlockScan(total[threadIdx.x], waveSum, all) + hist[(size_t)threadIdx.x * ntiles + blockIdx.x];
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t c = cnt[w][threadIdx.x];
        cnt[w][threadIdx.x] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
        if (i0 + 64 * r < n) {
            const uint32_t o = cnt[wave][(k[r] >> shift) & 0xFFu] + rank[r];
            keyOut[o] = k[r];
            valOut[o] = v[r];
        }
}

inline uint32_t sortTiles(uint32_t n) { return (n + kSortTile - 1) / kSortTile; }
inline uint64_t sortHistWords(uint32_t n) { return 256ull * sortTiles(n) + 256; }

// Sorts (key, val) by the low `bits` bits of the keys (the others are zero),
// with (key2, val2) and hist (sortHistWords(n) words) as work space.  The
// pointers change places so that (key, val) hold the result.
inline hipError_t sortPairs32(uint32_t*& key, uint32_t*& val, uint32_t*& key2, uint32_t*& val2, uint32_t* hist, uint32_t n, int bits,
                              hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const uint32_t nt = sortTiles(n);
    uint32_t* total = hist + 256ull * nt;
    for (int shift = 0; shift < bits; shift += 8) {
        sortHist<<<nt, kSortBlock, 0, stream>>>(key, n, shift, nt, hist);
        sortScan<<<256, kSortBlock, 0, stream>>>(hist, nt, total);
        sortScatter<<<nt, kSortBlock, 0, stream>>>(key, val, n, shift, nt, hist, total, key2, val2);
        std::swap(key, key2);
        std::swap(val, val2);
    }
    return hipGetLastError();
}

}  // namespace

#endif
