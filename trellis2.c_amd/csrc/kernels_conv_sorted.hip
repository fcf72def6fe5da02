// kernels_conv_sorted.hip - output-stationary MFMA conv over rows in mask order.
#include <type_traits>

#include "tsh_internal.h"
#include "mfma_ring.h"

namespace tsh {
namespace {

// A block owns BM rows (places in the rulebook's mask order) x BN output
// channels and keeps their fp32 sums in registers over all offsets: an
// implicit GEMM over (offset with a neighbour in the block, input channel).
// Rows with like masks share blocks, so 0.65-0.93 of the row-offsets a block
// multiplies have a neighbour on voxelised surfaces (0.55 where the children
// of a subdivision are random; the choice of a shape below does not look at
// it), which costs less than compacting the valid pairs: no unit lists, no tile
// sums in LDS, no scatter.  Not so on voxels scattered at random in few
// channels (300,000 at 20 %: 64 -> 16 54 us, compacted 54, 128 -> 32 100 and
// 92; from 128 -> 128 on it is the faster one).
//
// RW x CW wavefronts hold BM / RW rows x BN / CW channels each.  Each K step
// (32 input channels of one offset) brings BM gathered rows' 64 bytes and
// BN x 64 bytes of weights straight into one of SLOTS LDS slots
// (buffer_load ... lds, no registers on the way); a row without a neighbour
// reads past the buffer's end, which the hardware answers with zeros.  The
// loads run SLOTS steps ahead of their MFMAs.  Plain blocks read a step's
// fragments from LDS one step ahead, so its MFMAs wait for nothing but the
// one barrier.  Ping-pong blocks (PP: 224 or 256 x 256, one per CU) let wavefronts
// 0-3 (one per SIMD) and 4-7 take turns, half a step apart: one half reads
// fragments and issues loads while the other half multiplies (256 -> 256 on
// 300,000 rows: 0.74 -> 0.61 ms, MFMAs alone 0.46, loads and LDS alone 0.48).
//
// LDS layout of 16 rows x 64 bytes (one load instruction): row i at 64 i,
// its 16-byte chunk c at place c ^ (i >= 8 ? 2 : 0): four neighbouring lanes
// fetch one row's 64 contiguous bytes, and the fragment reads (lane i + 16 c:
// row i, chunk c) are free of bank conflicts (240 B per clock and CU,
// measured; 125 without the swizzle).
//
// What bounds it: the gathers and weights arrive at 20-24 B per clock and CU
// (L2 misses to the last-level cache, 5.5-5.8 TB/s; 45 when all rows hit the
// L2).  In 224 x 256 and 256 x 256 blocks the matrix cores are busy 80 % of
// the cycles (512 -> 512 on 328,123 rows: 1.02 PFLOP/s of valid pairs, 1.49
// with the absent ones), in 128-channel ones 36-55 %, 64-channel ones 21 %.
// Measured against the compacted schedule (ms, conv alone): 128 -> 128 on
// 419,341 rows 0.60 -> 0.31; 256 -> 1024 on 350,000 5.1 -> 2.7; 512 -> 512 on
// 79,523 1.11 -> 0.71; 1024 -> 1024 on 18,216 1.12 -> 0.77; 256 -> 256 on
// 5,003 0.100 -> 0.036; 64 -> 64 on 3,788,747 1.11 -> 0.85; 256 -> 128 on
// 1,259,866 random children 1.71 -> 1.56.
template <int DT, int BM, int BN, int RW, int CW, int SLOTS, bool PP = false>
__global__ void __launch_bounds__(64 * RW * CW, RW * CW == 8 ? 2 : 1)
    k_conv_sorted(const typename Store<DT>::T * __restrict__ x, const int32_t * __restrict__ table,
                  const int32_t * __restrict__ perm, const typename Store<DT>::T * __restrict__ w16,
                  const float * __restrict__ bias,
                  typename Store<DT>::T * __restrict__ y, int64_t n, int ci, int co, int group, ConvEpilogue epi) {
    using T = typename Store<DT>::T;
    using V = typename Mfma<DT>::V;
    constexpr int NW = RW * CW, NTHR = 64 * NW;
    constexpr int QB = BM / RW / 16;   // row blocks per wavefront
    constexpr int NT = BN / CW / 16;   // column tiles per wavefront
    using R = RingShape<BM, BN, RW, CW>;
    // Loads of a step, the block's and a wavefront's: of A, of the weights.
    constexpr int AL = R::AL, NA = R::NA, WL = R::WL, NB = R::NB, SLOT = R::SLOT;
    constexpr int OUT = BM * BN * 2;
    constexpr int RING = SLOTS * SLOT > OUT ? SLOTS * SLOT : OUT;
    __shared__ __attribute__((aligned(1024))) unsigned char s_ring[RING];
    __shared__ __attribute__((aligned(16))) int32_t s_nbr[BM * kMapRow];
    __shared__ int32_t s_perm[BM];
    __shared__ uint32_t s_or[NW];

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rw = wave % RW, cw = wave / RW;
    const int l16 = lane & 15, lg = lane >> 4;

    // Blocks b, b + 8, ... run on one XCD.  With 2, 4 or 8 column blocks each
    // XCD keeps to one of them (its weights in that XCD's L2), and the row
    // blocks, whose cost rises and falls along the mask order, are dealt to
    // the XCDs in turn.  (A contiguous eighth of the rows per XCD, in windows
    // of 2^15 rows, was slower: 64 -> 64 on 3,788,747 rows with its map 1.33
    // -> 1.41 ms, 512 -> 512 on 327,689 2.73 -> 2.81.)
    const int64_t row_tiles = (n + BM - 1) / BM;
    const int col_tiles = co / BN;
    int64_t tile;
    int colb;
    if (col_tiles == 2 || col_tiles == 4 || col_tiles == 8) {
        const int per = 8 / col_tiles;
        const int64_t b = blockIdx.x;
        colb = (int) (b % 8) / per;
        tile = b / 8 * per + (b % 8) % per;
        if (tile >= row_tiles) return;
    } else {
        tile = blockIdx.x % row_tiles;
        colb = (int) (blockIdx.x / row_tiles);
    }
    const int64_t row0 = tile * BM;
    const int col0 = colb * BN;
    const int rows = (int) ((n - row0) < BM ? (n - row0) : BM);
    const int ci8 = ci >> 3;
    const int KS = ci >> 5;

    // The rows at this block's places and their neighbours (a table row is
    // seven 16-byte pieces, the last holding the mask).
    for (int r = t; r < BM; r += NTHR) s_perm[r] = r < rows ? (perm != nullptr ? perm[row0 + r] : (int32_t) row0 + r) : -1;
    __syncthreads();
    uint32_t m = 0;
    for (int e = t; e < BM * 7; e += NTHR) {
        const int r = e / 7, c = e - r * 7;
        const int32_t row = s_perm[r];
        int4 v = c == 6 ? int4{-1, -1, -1, 0} : int4{-1, -1, -1, -1};
        if (row >= 0) v = *(const int4 *) (table + (int64_t) row * kMapRow + c * 4);
        *(int4 *) (s_nbr + e * 4) = v;
        if (c == 6) m |= (uint32_t) v.w;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) m |= (uint32_t) __shfl_xor((int) m, d);
    if (lane == 0) s_or[wave] = m;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) any |= s_or[w];
    any = (uint32_t) __builtin_amdgcn_readfirstlane((int) any);
    const int steps = __popc(any) * KS;

    // ---- loads ----------------------------------------------------------
    const uint32_t xbytes = (uint32_t) (n * ci * (int64_t) sizeof(T));
    const uint32_t wbytes = (uint32_t) (27ll * ci * co * (int64_t) sizeof(T));
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void *) x, 0, (int) xbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc((void *) w16, 0, (int) wbytes, 0x00020000);
    const uint32_t ring = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) unsigned char *) s_ring;
    constexpr uint32_t kAbsent = 0x80000000u;
    // A load j: row block (wave * NA + j) % AL, row lane / 4 of it, chunk place lane % 4.
    auto ablock = [&](int j) { return (wave * NA + j) % AL; };
    const uint32_t achunk = (uint32_t) (((lane & 3) ^ (((lane >> 5) & 1) << 1)) * 16);
    uint32_t av[NA];
    int32_t nsrc[NA];
    uint32_t wv[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int e = (wave * NB + j) % WL * 64 + lane;  // granule: chunk e / BN, column e % BN
        wv[j] = (uint32_t) ((e / BN * co + col0 + e % BN) * 16);
    }
    uint32_t left = any;   // offsets whose rows are not fetched yet
    int ik = 0, is = 0;    // offset and K step of the next load
    auto fetch_src = [&]() {
        // Sources at the next offset (read a whole offset before their use).
        const int k = left != 0 ? __builtin_ctz(left) : 0;
#pragma unroll
        for (int j = 0; j < NA; ++j) nsrc[j] = s_nbr[(ablock(j) * 16 + (lane >> 2)) * kMapRow + k];
    };
    auto next_offset = [&]() {
        const bool end = left == 0;
        ik = end ? ik : __builtin_ctz(left);
#pragma unroll
        for (int j = 0; j < NA; ++j)
            av[j] = (end || nsrc[j] < 0) ? kAbsent : (uint32_t) nsrc[j] * (uint32_t) (ci * 2) + achunk;
        left &= left - 1;
        fetch_src();
    };
    uint32_t islot = ring;
    auto load = [&](int j) {
        if (j < NA) {
            dma_b128(xres, islot + (uint32_t) ablock(j) * 1024u, av[j], (uint32_t) is * 64u);
        } else {
            dma_b128(wres, islot + (uint32_t) (BM * 64 + (wave * NB + j - NA) % WL * 1024), wv[j - NA],
                     (uint32_t) ((ik * ci8 + is * 4) * co) * 16u);
        }
    };
    auto advance = [&]() {
        islot = islot == ring + (SLOTS - 1) * SLOT ? ring : islot + SLOT;
        if (++is == KS) {
            is = 0;
            next_offset();
        }
    };

    f32x4 acc[QB][NT];
    fetch_src();
    next_offset();
    ring_multiply<DT, BM, BN, RW, CW, SLOTS, PP>(s_ring, steps, load, advance, acc);

    // ---- epilogue: bias, one rounding, the tile through LDS ----------------
    // Packed column p of a group of 16 g columns holds channel (p % 16) g +
    // p / 16 of it.  Chunk c (8 channels) of row r is staged at c ^ (r & SWZ).
    constexpr int CHUNKS = BN / 8;
    constexpr int PASSES = BM * CHUNKS / NTHR;
    constexpr int SWZ = CHUNKS < 8 ? CHUNKS - 1 : 7;
    static_assert(PASSES >= 1 && NTHR % CHUNKS == 0, "whole rows per pass");
    T * s_out = (T *) s_ring;
    int ch[NT];
    float bv[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int pc = cw * NT * 16 + nt * 16, gs = 16 * group;
        ch[nt] = pc / gs * gs + l16 * group + pc % gs / 16;
        bv[nt] = bias != nullptr ? bias[col0 + ch[nt]] : 0.0f;
    }
    lds_barrier();
#pragma unroll
    for (int q = 0; q < QB; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = (rw * QB + q) * 16 + lg * 4 + i;
#pragma unroll
            for (int nt = 0; nt < NT; nt += 2) {
                if constexpr (NT == 1) {
                    s_out[r * BN + ((ch[0] >> 3) ^ (r & SWZ)) * 8 + (ch[0] & 7)] = round_to_store<DT>(acc[q][0][i] + bv[0]);
                    break;
                }
                union {
                    uint32_t u;
                    T h[2];
                } o;
                o.h[0] = round_to_store<DT>(acc[q][nt][i] + bv[nt]);
                o.h[1] = round_to_store<DT>(acc[q][nt + 1][i] + bv[nt + 1]);
                *(uint32_t *) (s_out + r * BN + ((ch[nt] >> 3) ^ (r & SWZ)) * 8 + (ch[nt] & 7)) = o.u;
            }
        }
    const int cidx = t % CHUNKS, cc = cidx * 8, rr0 = t / CHUNKS;
    float gv[8], sv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        gv[u] = epi.gamma != nullptr ? epi.gamma[col0 + cc + u] : 1.0f;
        sv[u] = epi.beta != nullptr ? epi.beta[col0 + cc + u] : 0.0f;
    }
    lds_barrier();
    auto passes = [&](auto mode_c, auto silu_c) {
        constexpr int MODE = decltype(mode_c)::value;
        constexpr bool SILU = decltype(silu_c)::value;
#pragma unroll 4
        for (int p = 0; p < PASSES; ++p) {
            const int rr = rr0 + p * (NTHR / CHUNKS);
            const int32_t row = s_perm[rr];
            int4 o = *(const int4 *) (s_out + rr * BN + (cidx ^ (rr & SWZ)) * 8);
            if constexpr (MODE == kEpiNorm) {
                float v[8];
                unpack_chunk<DT>(o, v);
                float sum = 0.0f;
#pragma unroll
                for (int u = 0; u < 8; ++u) sum += v[u];
                const float mean = row16_sum(sum) / (float) BN;
                float q = 0.0f;
#pragma unroll
                for (int u = 0; u < 8; ++u) q += (v[u] - mean) * (v[u] - mean);
                const float inv = 1.0f / sqrtf(row16_sum(q) / (float) BN + epi.eps);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    float r = (v[u] - mean) * inv;
                    r = r * gv[u] + sv[u];
                    if constexpr (SILU) r = r * __builtin_amdgcn_rcpf(1.0f + __expf(-r));
                    v[u] = r;
                }
                o = pack_chunk<DT>(v);
            } else if constexpr (MODE == kEpiAdd) {
                if (row >= 0) {
                    float v[8], rv[8];
                    unpack_chunk<DT>(o, v);
                    unpack_chunk<DT>(*(const int4 *) ((const T *) epi.residual + (int64_t) row * co + col0 + cc), rv);
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] += rv[u];
                    o = pack_chunk<DT>(v);
                }
            }
            if (row >= 0) *(int4 *) (y + (int64_t) row * co + col0 + cc) = o;
        }
    };
    using kNone = std::integral_constant<int, kEpiNone>;
    using kNorm = std::integral_constant<int, kEpiNorm>;
    using kAdd = std::integral_constant<int, kEpiAdd>;
    if (epi.mode == kEpiNorm) {
        if constexpr (BN == 128) {
            if (epi.silu) {
                passes(kNorm(), std::true_type());
            } else {
                passes(kNorm(), std::false_type());
            }
        }
    } else if (epi.mode == kEpiAdd) {
        passes(kAdd(), std::false_type());
    } else {
        passes(kNone(), std::false_type());
    }
}

template <int DT, int BM, int BN, int RW, int CW, int SLOTS, bool PP = false>
hipError_t launch_t(const void * x, const int32_t * rows, const int32_t * perm, const void * w16, const float * bias,
                    void * y, int64_t n, int ci, int co, hipStream_t s, const ConvEpilogue & epi) {
    using T = typename Store<DT>::T;
    const int64_t row_tiles = (n + BM - 1) / BM, col_tiles = co / BN;
    int64_t grid = row_tiles * col_tiles;
    if (col_tiles == 2 || col_tiles == 4 || col_tiles == 8) {
        const int64_t per = 8 / col_tiles;
        grid = (row_tiles + per - 1) / per * 8;
    }
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    k_conv_sorted<DT, BM, BN, RW, CW, SLOTS, PP><<<(unsigned) grid, 64 * RW * CW, 0, s>>>(
        (const T *) x, rows, perm, (const T *) w16, bias, (T *) y, n, ci, co, conv_stream_group(ci, co), epi);
    return hipGetLastError();
}

// Block shapes, largest first.  cost[b - 1]: time of one round with b blocks
// on every CU, as a fraction of a 256 x 256 block's (0.118 ms at 256 -> 256
// with all 27 offsets); blocks per CU follow from the LDS.  Measured on 128 ..
// 1024 channels and 2,000 .. 350,000 rows.
struct Shape {
    int id, bm, bn, per_cu;
    double cost[4];
};
constexpr Shape kShapes[] = {
    {0, 256, 256, 1, {1.0}},
    {1, 224, 256, 1, {0.89}},
    {2, 192, 256, 1, {0.83}},
    {3, 160, 256, 1, {0.77}},
    {4, 128, 256, 1, {0.66}},
    {5, 96, 256, 1, {0.58}},
    {6, 128, 128, 2, {0.44, 0.75}},
    {7, 64, 128, 2, {0.33, 0.46}},
    {8, 64, 64, 4, {0.24, 0.34, 0.50, 0.66}},
};

// The shape that finishes first: large blocks do the most MFMA work per
// fetched byte (256 -> 1024 on 350,000 rows: 2.77 ms with 256 x 256, 3.11 with
// 128 x 256), small ones fill the GPU on small sets (256 -> 256 on 5,003 rows:
// 0.113 ms with 256 x 256, 0.074 with 128 x 256, 0.061 with 96 x 256, 0.049
// with 128 x 128, 0.036 with 64 x 128, which is taken, 0.033 with 64 x 64), and
// between these the row count decides which fills its last round (1024 -> 1024
// on 18,216 rows: 0.93, 0.85, 0.81, 0.77 and 0.86 ms down the list; 256 -> 256
// on 80,000: 0.253, 0.234, 0.205, 0.193 and 0.213; on 20,000: 0.122, 0.116,
// 0.109, 0.095, 0.081 and 0.071; on 300,000: 0.70, 0.63, 0.65, 0.67, 0.68).
int pick_shape(int64_t n, int ci, int co, int cus, bool whole_rows) {
    // With more weights per column block than an XCD's L2 holds, blocks of few
    // columns that share a CU wait for them (512 -> 512 on 79,523 rows, 128 x
    // 128: 1.05 ms against 0.77; 1024 -> 1024 on 18,216: 1.21 against 0.86).
    const double heavy = ci <= 256 ? 1.0 : (ci <= 512 ? 1.3 : 1.6);
    int best = -1;
    double best_t = 0.0;
    for (const Shape & sh : kShapes) {
        if (co % sh.bn != 0 || (whole_rows && sh.bn != co)) continue;
        const int64_t blocks = (n + sh.bm - 1) / sh.bm * (co / sh.bn);
        const int64_t cap = (int64_t) cus * sh.per_cu;
        const int64_t rounds = blocks / cap, rest = blocks - rounds * cap;
        const double full = sh.cost[sh.per_cu - 1] * (sh.per_cu > 1 ? heavy : 1.0);
        double t = (double) rounds * full;
        if (rest > 0) {
            const int on = (int) ((rest + cus - 1) / cus);
            t += sh.cost[on - 1] * (on > 1 ? heavy : 1.0);
        }
        // Blocks are of unequal cost (as many offsets as their rows' masks
        // share): over more than two rounds that evens out all but a tail of
        // about one block.
        if (blocks > 2 * cap) t = ((double) blocks / (double) cap + 1.0) * full;
        if (best < 0 || t < best_t) {
            best = sh.id;
            best_t = t;
        }
    }
    return best;
}

template <int DT>
hipError_t launch_dt(const void * x, const int32_t * rows, const int32_t * perm, const void * w16, const float * bias,
                     void * y, int64_t n, int ci, int co, int cus, hipStream_t s, const ConvEpilogue & epi) {
#define TSH_SORTED(...) launch_t<DT, __VA_ARGS__>(x, rows, perm, w16, bias, y, n, ci, co, s, epi)
    // 16 and 32 channels: 128 rows of four wavefronts, four slots, three blocks
    // per CU.  Measured on ordered rows (us, conv alone; the compacted kernel
    // last): 64 -> 16 on 1,200,000 rows 225, with three slots (also three
    // blocks) 230, two 235, 256 rows and two slots 254, two wavefronts 242;
    // 252; 512 -> 16 on 5,000 rows 60, 83, 121, 148, 83; 169; on 60,000 140,
    // 146, 167, 204, 144; 182.  128 -> 32 on 1,200,000 rows 426, three slots
    // 433, two 453, 64 rows 459, 256 rows 470; 510; on 5,000 rows 17, 18, 24,
    // 14, 32; 54.
    if (co == 16) return TSH_SORTED(128, 16, 4, 1, 4);
    if (co == 32) return TSH_SORTED(128, 32, 4, 1, 4);
    if (co % 128 != 0) {
        // 64-channel blocks: 128 rows once those fill the GPU (3,788,747
        // rows, 64 -> 64: 0.85 ms, 0.90 with three slots and a block less per
        // CU; 5,000 rows: 0.014 against 0.010 ms).
        if ((n + 127) / 128 * (co / 64) < 2 * (int64_t) cus) return TSH_SORTED(64, 64, 2, 2, 4);
        return TSH_SORTED(128, 64, 4, 1, 2);
    }
    switch (pick_shape(n, ci, co, cus, epi.mode == kEpiNorm)) {
        case 0: return TSH_SORTED(256, 256, 2, 4, 4, true);
        case 1: return TSH_SORTED(224, 256, 2, 4, 4, true);
        case 2: return TSH_SORTED(192, 256, 2, 4, 4);
        case 3: return TSH_SORTED(160, 256, 2, 4, 4);
        case 4: return TSH_SORTED(128, 256, 2, 4, 4);
        case 5: return TSH_SORTED(96, 256, 2, 4, 3);
        case 6:
            // With 8 or fewer K steps per offset a block's start and end
            // weigh more: two slots instead of four leave room for a third
            // block per CU to run under them (1,159,741 rows, 128 -> 128:
            // 0.72 -> 0.66 ms; 256 -> 128 the same either way).
            if (ci <= 128 && (n + 127) / 128 * (co / 128) >= 6 * (int64_t) cus) return TSH_SORTED(128, 128, 2, 2, 2);
            return TSH_SORTED(128, 128, 2, 2, 4);
        case 7: return TSH_SORTED(64, 128, 2, 2, 4);
        case 8: return TSH_SORTED(64, 64, 2, 2, 4);
    }
#undef TSH_SORTED
    return hipErrorInvalidValue;
}

}  // namespace

// The loads address x and the weights through buffer resources with 32-bit
// byte ranges, of which a missing neighbour takes the upper half.
bool conv_sorted_supported(int dtype, int ci, int co, int64_t n) {
    return (dtype == kF16 || dtype == kBF16) && ci % 64 == 0 && ci > 0 &&
           (co == 16 || co == 32 || (co % 64 == 0 && co > 0)) && n > 0 && n <= INT32_MAX / (2 * (int64_t) ci) &&
           (int64_t) 54 * ci * co <= (int64_t) INT32_MAX;
}

hipError_t launch_conv_sorted(int dtype, const void * x, const int32_t * rows, const int32_t * perm, const void * w16,
                              const float * bias, void * y, int64_t n, int ci, int co, int cus, hipStream_t s,
                              const ConvEpilogue & epi) {
    if (!conv_sorted_supported(dtype, ci, co, n) || (epi.mode == kEpiNorm && co != 128)) return hipErrorInvalidValue;
    if (dtype == kBF16) return launch_dt<kBF16>(x, rows, perm, w16, bias, y, n, ci, co, cus, s, epi);
    return launch_dt<kF16>(x, rows, perm, w16, bias, y, n, ci, co, cus, s, epi);
}

}  // namespace tsh
