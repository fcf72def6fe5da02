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
// Each block of rows counts its buckets in LDS, a second kernel turns every
// bucket's counts into starts over the blocks, and no count goes through a
// global atomic: adding the block histograms up in global memory and drawing
// each block's starts with adds that return took 0.097 ms for 1,263,630 rows
// of random children (nearly every row a bucket of its own there) and 0.090
// for 3,788,747 surface rows, latency of the adds; now 0.055 and 0.075, half of
// it the scattered places.
#include "tsh_internal.h"

namespace tsh {
namespace {

constexpr int kOrderBits = 14;
constexpr int kOrderBins = 1 << kOrderBits;
constexpr int kThreads = 1024;
constexpr int kRowsPerThread = 4;
constexpr int kRowsPerBlock = kThreads * kRowsPerThread;
constexpr int kColThreads = 256;
constexpr int kPlaceThreads = 256;

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

// Block histograms hold two 16-bit counts per word (a block has at most 4096
// rows): 32 KB, half the words to clear and to look through.
constexpr int kHistWords = kOrderBins / 2;

// A block's bucket sizes, and each row's rank in its block's part of a bucket.
__global__ void __launch_bounds__(kThreads) k_order_count(const uint32_t * __restrict__ mask, int64_t n,
                                                          int32_t * __restrict__ counts,
                                                          uint16_t * __restrict__ rank) {
    __shared__ uint32_t s_hist[kHistWords];
    const int t = threadIdx.x;
    const int64_t row0 = (int64_t) blockIdx.x * kRowsPerBlock;
    for (int b = t; b < kHistWords; b += kThreads) s_hist[b] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRowsPerThread; ++j) {
        const int64_t i = row0 + j * kThreads + t;
        if (i < n) {
            const uint32_t k = order_key(mask[i]), sh = 16 * (k & 1u);
            rank[i] = (uint16_t) (atomicAdd(&s_hist[k >> 1], 1u << sh) >> sh);
        }
    }
    __syncthreads();
    int2 * out = (int2 *) (counts + (int64_t) blockIdx.x * kOrderBins);
    for (int b = t; b < kHistWords; b += kThreads) {
        const uint32_t c = s_hist[b];
        out[b] = int2{(int32_t) (c & 0xffffu), (int32_t) (c >> 16)};
    }
}

// Per window and bucket: the blocks' counts become starts within the bucket
// (in place), their sum the bucket's size.
__global__ void __launch_bounds__(kColThreads) k_order_columns(int32_t * __restrict__ counts, int64_t blocks,
                                                               int64_t per_window, int32_t * __restrict__ bins) {
    constexpr int kCols = kOrderBins / kColThreads, kAhead = 8;
    const int64_t w = blockIdx.x / kCols;
    const int bin = (int) (blockIdx.x % kCols) * kColThreads + threadIdx.x;
    const int64_t b1 = (w + 1) * per_window < blocks ? (w + 1) * per_window : blocks;
    int32_t at = 0;
    for (int64_t b = w * per_window; b < b1; b += kAhead) {
        int32_t c[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) c[j] = b + j < b1 ? counts[(b + j) * kOrderBins + bin] : 0;
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            if (b + j < b1) counts[(b + j) * kOrderBins + bin] = at;
            at += c[j];
        }
    }
    bins[w * kOrderBins + bin] = at;
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

// Places: the bucket's start, the block's part of it, the row's rank there.
__global__ void __launch_bounds__(kPlaceThreads) k_order_place(const uint32_t * __restrict__ mask, int64_t n,
                                                               int64_t window, const int32_t * __restrict__ bins,
                                                               const int32_t * __restrict__ counts,
                                                               const uint16_t * __restrict__ rank,
                                                               int32_t * __restrict__ perm) {
    const int64_t row0 = (int64_t) blockIdx.x * (kPlaceThreads * kRowsPerThread);
    const int32_t * start = bins + row0 / window * kOrderBins;
    const int32_t * part = counts + row0 / kRowsPerBlock * kOrderBins;
#pragma unroll
    for (int j = 0; j < kRowsPerThread; ++j) {
        const int64_t i = row0 + j * kPlaceThreads + threadIdx.x;
        if (i < n) {
            const uint32_t k = order_key(mask[i]);
            perm[start[k] + part[k] + (int32_t) rank[i]] = (int32_t) i;
        }
    }
}

int64_t order_blocks(int64_t n) { return (n + kRowsPerBlock - 1) / kRowsPerBlock; }

}  // namespace

// Bucket starts of each window, bucket counts of each block, ranks.
size_t order_bins_bytes(int64_t n, int64_t window) {
    return (size_t) ((n + window - 1) / window + order_blocks(n)) * kOrderBins * sizeof(int32_t) +
           (size_t) n * sizeof(uint16_t);
}

hipError_t launch_order(const uint32_t * mask, int64_t n, int64_t window, int32_t * bins, int32_t * perm,
                        hipStream_t s) {
    static_assert(kRowsPerBlock % (kPlaceThreads * kRowsPerThread) == 0, "a place block lies in one count block");
    if (window <= 0 || window % kRowsPerBlock != 0) return hipErrorInvalidValue;
    const int64_t blocks = order_blocks(n), windows = (n + window - 1) / window;
    int32_t * counts = bins + windows * kOrderBins;
    uint16_t * rank = (uint16_t *) (counts + blocks * kOrderBins);
    k_order_count<<<(unsigned) blocks, kThreads, 0, s>>>(mask, n, counts, rank);
    k_order_columns<<<(unsigned) (windows * (kOrderBins / kColThreads)), kColThreads, 0, s>>>(
        counts, blocks, window / kRowsPerBlock, bins);
    k_order_scan<<<(unsigned) windows, kThreads, 0, s>>>(bins, window);
    const int64_t places = (n + kPlaceThreads * kRowsPerThread - 1) / (kPlaceThreads * kRowsPerThread);
    k_order_place<<<(unsigned) places, kPlaceThreads, 0, s>>>(mask, n, window, bins, counts, rank, perm);
    return hipGetLastError();
}

}  // namespace tsh
