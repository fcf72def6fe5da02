// kernels_order.hip - the order in which the sorted conv takes a rulebook's rows.
//
// The sorted conv (kernels_conv_sorted.hip) multiplies, per block of rows,
// every offset at which any of its rows has a neighbour.  Rows with equal or
// similar neighbour masks are therefore put next to each other: on voxelised
// surfaces the masks repeat (a few thousand different ones), and 256-row
// blocks in mask order have a neighbour for 0.65-0.93 of the row-offsets they
// multiply, against 0.4-0.6 in raster order.
//
// The sort is one bucket pass over a 14-bit key: the Gray-code rank of the
// mask's 8 corner and 6 face bits (neighbouring buckets differ in one bit, so
// blocks that span two stay full; edges follow from corners and faces on
// surfaces: 0.80 against 0.82 for a full 26-bit sort on the R = 256 shells).
// The order within a bucket follows the atomics; a row's result does not
// depend on which rows share its block, so the outputs do not either.
#include "tsh_internal.h"

namespace tsh {
namespace {

constexpr int kOrderBits = 14;
constexpr int kOrderBins = 1 << kOrderBits;
constexpr int kThreads = 1024;
constexpr int kRowsPerThread = 4;
constexpr int kRowsPerBlock = kThreads * kRowsPerThread;

// Most significant bit first: corners, then faces.
__device__ __forceinline__ uint32_t order_key(uint32_t m) {
    constexpr int bits[kOrderBits] = {0, 2, 6, 8, 18, 20, 24, 26, 4, 10, 12, 14, 16, 22};
    uint32_t k = 0;
#pragma unroll
    for (int j = 0; j < kOrderBits; ++j) k = (k << 1) | ((m >> bits[j]) & 1u);
    // Rank of the code word k in the Gray sequence.
    k ^= k >> 1;
    k ^= k >> 2;
    k ^= k >> 4;
    k ^= k >> 8;
    return k;
}

__global__ void __launch_bounds__(kThreads) k_order_clear(int32_t * __restrict__ bins) {
    bins[blockIdx.x * kThreads + threadIdx.x] = 0;
}

// Block histograms hold two 16-bit counts per word (a block has at most 4096
// rows): 32 KB, half the words to clear and to look through.
constexpr int kHistWords = kOrderBins / 2;

// Bucket sizes: an LDS histogram per block, one add per bucket it has.
__global__ void __launch_bounds__(kThreads) k_order_count(const uint32_t * __restrict__ mask, int64_t n,
                                                          int64_t window, int32_t * __restrict__ bins) {
    __shared__ uint32_t s_hist[kHistWords];
    const int t = threadIdx.x;
    const int64_t row0 = (int64_t) blockIdx.x * kRowsPerBlock;
    for (int b = t; b < kHistWords; b += kThreads) s_hist[b] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRowsPerThread; ++j) {
        const int64_t i = row0 + j * kThreads + t;
        if (i < n) {
            const uint32_t k = order_key(mask[i]);
            atomicAdd(&s_hist[k >> 1], 1u << (16 * (k & 1u)));
        }
    }
    __syncthreads();
    int32_t * out = bins + row0 / window * kOrderBins;
    for (int b = t; b < kHistWords; b += kThreads) {
        const uint32_t c = s_hist[b];
        if ((c & 0xffffu) != 0) atomicAdd(&out[2 * b], (int32_t) (c & 0xffffu));
        if ((c >> 16) != 0) atomicAdd(&out[2 * b + 1], (int32_t) (c >> 16));
    }
}

// Bucket starts (exclusive scan in place, one block per window).
__global__ void __launch_bounds__(kThreads) k_order_scan(int32_t * __restrict__ all, int64_t window) {
    int32_t * bins = all + (int64_t) blockIdx.x * kOrderBins;
    constexpr int kPer = kOrderBins / kThreads;
    __shared__ int32_t s_wave[kThreads / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int32_t v[kPer], sum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        v[j] = bins[t * kPer + j];
        sum += v[j];
    }
    int32_t incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int32_t o = __shfl_up(incl, d);
        if (lane >= d) incl += o;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    int32_t at = incl - sum + (int32_t) (blockIdx.x * window);
    for (int w = 0; w < wave; ++w) at += s_wave[w];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        bins[t * kPer + j] = at;
        at += v[j];
    }
}

// Places: a row's rank in its block's part of the bucket comes from LDS, the
// part's start from one add per block and bucket.
__global__ void __launch_bounds__(kThreads) k_order_place(const uint32_t * __restrict__ mask, int64_t n,
                                                          int64_t window, int32_t * __restrict__ bins,
                                                          int32_t * __restrict__ perm) {
    __shared__ uint32_t s_hist[kHistWords];
    __shared__ int32_t s_start[kOrderBins];
    const int t = threadIdx.x;
    const int64_t row0 = (int64_t) blockIdx.x * kRowsPerBlock;
    for (int b = t; b < kHistWords; b += kThreads) s_hist[b] = 0;
    __syncthreads();
    uint32_t key[kRowsPerThread], rank[kRowsPerThread];
#pragma unroll
    for (int j = 0; j < kRowsPerThread; ++j) {
        const int64_t i = row0 + j * kThreads + t;
        key[j] = i < n ? order_key(mask[i]) : 0u;
        const uint32_t sh = 16 * (key[j] & 1u);
        rank[j] = i < n ? (atomicAdd(&s_hist[key[j] >> 1], 1u << sh) >> sh) & 0xffffu : 0u;
    }
    __syncthreads();
    int32_t * at = bins + row0 / window * kOrderBins;
    for (int b = t; b < kHistWords; b += kThreads) {
        const uint32_t c = s_hist[b];
        if ((c & 0xffffu) != 0) s_start[2 * b] = atomicAdd(&at[2 * b], (int32_t) (c & 0xffffu));
        if ((c >> 16) != 0) s_start[2 * b + 1] = atomicAdd(&at[2 * b + 1], (int32_t) (c >> 16));
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRowsPerThread; ++j) {
        const int64_t i = row0 + j * kThreads + t;
        if (i < n) perm[s_start[key[j]] + (int32_t) rank[j]] = (int32_t) i;
    }
}

}  // namespace

size_t order_bins_bytes(int64_t n, int64_t window) {
    return (size_t) ((n + window - 1) / window) * kOrderBins * sizeof(int32_t);
}

hipError_t launch_order(const uint32_t * mask, int64_t n, int64_t window, int32_t * bins, int32_t * perm,
                        hipStream_t s) {
    const unsigned blocks = (unsigned) ((n + kRowsPerBlock - 1) / kRowsPerBlock);
    const unsigned windows = (unsigned) ((n + window - 1) / window);
    if (window % kRowsPerBlock != 0) return hipErrorInvalidValue;
    k_order_clear<<<windows * (kOrderBins / kThreads), kThreads, 0, s>>>(bins);
    k_order_count<<<blocks, kThreads, 0, s>>>(mask, n, window, bins);
    k_order_scan<<<windows, kThreads, 0, s>>>(bins, window);
    k_order_place<<<blocks, kThreads, 0, s>>>(mask, n, window, bins, perm);
    return hipGetLastError();
}

}  // namespace tsh
