// kernels_gemm.hip - the wide linears (16-bit storage) as a GEMM through LDS.
#include "tsh_internal.h"
#include "mfma_ring.h"

namespace tsh {
namespace {

// y = x W^T + b (then SiLU) in the storage type, or the sum of that and a
// residual, rounded again as the slots linear and add do.  A block multiplies BM consecutive rows by BN columns with the
// sorted conv's K loop (mfma_ring.h), one "offset" of Ci channels.  A
// wavefront holds 128 columns, packed so that a lane's eight are adjacent
// channels: bias, SiLU and residual work on the sums where they are, and a row
// leaves as 16-byte stores (256 contiguous bytes per 16 lanes) with no pass
// through LDS and no barrier, under the K loop of the CU's other block.
template <int DT, int BM, int BN, int RW, int CW, int SLOTS>
__global__ void __launch_bounds__(64 * RW * CW, 1)
    k_gemm(const typename Store<DT>::T * __restrict__ x, const typename Store<DT>::T * __restrict__ w16,
           const float * __restrict__ bias, const typename Store<DT>::T * __restrict__ residual,
           typename Store<DT>::T * __restrict__ y, int64_t n, int ci, int co, int silu) {
    using T = typename Store<DT>::T;
    using R = RingShape<BM, BN, RW, CW>;
    constexpr int NW = R::NW, NTHR = 64 * NW, QB = R::QB, NT = R::NT, NA = R::NA, NB = R::NB, WL = R::WL;
    constexpr int SLOT = R::SLOT;
    constexpr int WR = BM / RW;                 // rows per wavefront row group
    constexpr int RING = SLOTS * SLOT;
    static_assert(NT == 8, "eight adjacent channels per lane");
    static_assert(R::AL % NW == 0, "whole loads of A");
    __shared__ __attribute__((aligned(1024))) unsigned char s_ring[RING];

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int rw = wave % RW, cw = wave / RW;
    const int l16 = lane & 15, lg = lane >> 4;

    // Blocks b, b + 8, ... run on one XCD, which multiplies a row block by
    // every column block in turn: the rows stay in its L2 (1 to 5 % faster
    // than keeping an XCD to some column blocks, also where the weights exceed
    // the L2).
    const int64_t row_tiles = (n + BM - 1) / BM;
    const int col_tiles = co / BN;
    const int64_t in_xcd = blockIdx.x / 8;
    const int64_t tile = in_xcd / col_tiles * 8 + blockIdx.x % 8;
    const int colb = (int) (in_xcd % col_tiles);
    if (tile >= row_tiles) return;
    const int64_t row0 = tile * BM;
    const int col0 = colb * BN;
    const int KS = ci >> 5;

    const __amdgpu_buffer_rsrc_t xres =
        __builtin_amdgcn_make_buffer_rsrc((void *) x, 0, (int) (n * ci * (int64_t) sizeof(T)), 0x00020000);
    const __amdgpu_buffer_rsrc_t wres =
        __builtin_amdgcn_make_buffer_rsrc((void *) w16, 0, (int) ((int64_t) ci * co * (int64_t) sizeof(T)), 0x00020000);
    const uint32_t ring = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) unsigned char *) s_ring;
    uint32_t av[NA], wv[NB];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const int64_t row = row0 + (wave * NA + j) * 16 + (lane >> 2);
        const uint32_t chunk = (uint32_t) (((lane & 3) ^ (((lane >> 5) & 1) << 1)) * 16);
        av[j] = row < n ? (uint32_t) (row * ci * 2) + chunk : 0x80000000u;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int e = (wave * NB + j) % WL * 64 + lane;  // granule: chunk e / BN, column e % BN
        wv[j] = (uint32_t) ((e / BN * co + col0 + e % BN) * 16);
    }
    int is = 0;
    uint32_t islot = ring;
    auto load = [&](int j) {
        if (j < NA) {
            dma_b128(xres, islot + (uint32_t) (wave * NA + j) * 1024u, av[j], (uint32_t) is * 64u);
        } else {
            dma_b128(wres, islot + (uint32_t) (BM * 64 + (wave * NB + j - NA) % WL * 1024), wv[j - NA],
                     (uint32_t) (is * 4 * co) * 16u);
        }
    };
    // Past the last step the loads repeat it (their slots are not read).
    auto advance = [&]() {
        islot = islot == ring + (SLOTS - 1) * SLOT ? ring : islot + SLOT;
        is = is + 1 < KS ? is + 1 : is;
    };
    f32x4 acc[QB][NT];
    ring_multiply<DT, BM, BN, RW, CW, SLOTS, false>(s_ring, KS, load, advance, acc);

    // Lane (l16, lg) holds rows 4 lg + i of each row block, channels
    // 8 l16 .. 8 l16 + 7 of the wavefront's 128.
    const int64_t c0 = col0 + cw * 128 + l16 * 8;
    float bv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) bv[u] = bias != nullptr ? bias[c0 + u] : 0.0f;
    auto store = [&](auto silu_c, auto res_c) {
#pragma unroll
        for (int q = 0; q < QB; ++q) {
            const int64_t r0 = row0 + rw * WR + q * 16 + lg * 4;
            int4 rc[4];
            if constexpr (decltype(res_c)::value) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    rc[i] = r0 + i < n ? *(const int4 *) (residual + (r0 + i) * co + c0) : int4{0, 0, 0, 0};
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = acc[q][u][i] + bv[u];
                if constexpr (decltype(silu_c)::value) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = v[u] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[u]));
                }
                if constexpr (decltype(res_c)::value) {
                    float rv[8];
                    unpack_chunk<DT>(pack_chunk<DT>(v), v);
                    unpack_chunk<DT>(rc[i], rv);
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] += rv[u];
                }
                if (r0 + i < n) *(int4 *) (y + (r0 + i) * co + c0) = pack_chunk<DT>(v);
            }
        }
    };
    if (silu) {
        store(std::true_type(), std::false_type());
    } else if (residual != nullptr) {
        store(std::false_type(), std::true_type());
    } else {
        store(std::false_type(), std::false_type());
    }
}

template <int DT, int BM, int BN, int RW, int CW, int SLOTS>
hipError_t launch_t(const void * x, const void * w16, const float * bias, const void * residual, void * y, int64_t n,
                    int ci, int co, int silu, hipStream_t s) {
    using T = typename Store<DT>::T;
    const int64_t row_tiles = (n + BM - 1) / BM, col_tiles = co / BN;
    const int64_t grid = (row_tiles + 7) / 8 * 8 * col_tiles;
    if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
    k_gemm<DT, BM, BN, RW, CW, SLOTS><<<(unsigned) grid, 64 * RW * CW, 0, s>>>(
        (const T *) x, (const T *) w16, bias, (const T *) residual, (T *) y, n, ci, co, silu);
    return hipGetLastError();
}

template <int DT>
hipError_t launch_dt(const void * x, const void * w16, const float * bias, const void * residual, void * y, int64_t n,
                     int ci, int co, int silu, int cus, hipStream_t s) {
#define TSH_GEMM(...) launch_t<DT, __VA_ARGS__>(x, w16, bias, residual, y, n, ci, co, silu, s)
    const auto blocks = [&](int bm, int bn) { return (n + bm - 1) / bm * (co / bn); };
    // Two blocks of 128 x 256 (or 256 x 128) share a CU, and one's stores run
    // under the other's K loop; where those would leave CUs idle, smaller
    // blocks.  Measured (ms, this kernel against k_linear_mfma): 512 -> 2048
    // with SiLU on 79,523 rows 0.26 (0.35), 2048 -> 512 0.19 (0.28), 1024 ->
    // 4096 with SiLU on 18,216 0.17 (0.25), 256 -> 1024 with SiLU on 300,000
    // 0.36 (0.42), 128 -> 128 on 1,000,000 0.118 (0.134); 2048 -> 512 on 5,003
    // rows: 128 x 256 0.028, 128 x 128 0.021.
    // SiLU's exponentials are VALU work at a block's end, which weighs on short K
    // loops: up to Ci = 256 and eight large blocks per CU smaller ones overlap it
    // better (us, 128 x 256 / 128 x 128 / 64 x 128; k_linear_mfma: 256 -> 1024 on
    // 12,000 rows 16.7 / 14.9 / 15.0; 15.6; 256 -> 256 on 80,000 24.8 / 21.9 /
    // 24.4; 23.8, on 300,000 83 / 88 / 115; 101; 256 x 128 on 128 -> 384, 80,000
    // rows 27.0 / 23.2 / 25.6; 26.5; 256 -> 1024 on 5,000 11.1 / 9.3 / 8.4; 11.1;
    // 128 -> 128 on 40,000 - / 8.1 / 7.3; 8.9; but 1024 -> 4096 on 12,000 99 /
    // 129).
    const bool short_silu = silu && ci <= 256;
    const int64_t b128 = blocks(128, 128);
    if (co % 256 == 0 && blocks(128, 256) >= (short_silu ? 8 : 1) * (int64_t) cus) return TSH_GEMM(128, 256, 2, 2, 3);
    if (co % 256 != 0 && blocks(256, 128) >= (short_silu ? 8 : 2) * (int64_t) cus) return TSH_GEMM(256, 128, 4, 1, 3);
    if (5 * b128 >= 3 * (int64_t) cus && !(short_silu && 2 * b128 < 3 * (int64_t) cus)) {
        // One block on a CU has room for a fourth slot, which pays on deep rows
        // (2048 -> 512 on 5,000: 20.2 -> 18.4 us, with SiLU 21.4 -> 19.4; 1024 ->
        // 256 on 12,000 11.7 -> 11.4; with more blocks 4096 -> 1024 on 5,000 52
        // -> 56).
        if (ci >= 512 && b128 <= cus) return TSH_GEMM(128, 128, 4, 1, 4);
        return TSH_GEMM(128, 128, 4, 1, 3);
    }
    return TSH_GEMM(64, 128, 4, 1, 4);
#undef TSH_GEMM
}

}  // namespace

// Of the widths whose weights launch_linear_mfma rounds to the storage type too,
// those with whole 128-column blocks: other multiples of 64 input channels
// (192, 320, ...), which the K loop could take, keep their fp32 weights on the
// VALU kernel.
bool gemm_supported(int dtype, int64_t n, int ci, int co) {
    return linear_mfma_supported(dtype, ci, co) && co % 128 == 0 && n > 0 &&
           n <= INT32_MAX / (2 * (int64_t) ci) && (int64_t) ci * co * 2 <= (int64_t) INT32_MAX;
}

hipError_t launch_gemm(int dtype, const void * x, const void * w16, const float * bias, const void * residual,
                       void * y, int64_t n, int ci, int co, int silu, int cus, hipStream_t s) {
    if (!gemm_supported(dtype, n, ci, co) || cus <= 0) return hipErrorInvalidValue;
    if (dtype == kBF16) return launch_dt<kBF16>(x, w16, bias, residual, y, n, ci, co, silu, cus, s);
    return launch_dt<kF16>(x, w16, bias, residual, y, n, ci, co, silu, cus, s);
}

}  // namespace tsh
