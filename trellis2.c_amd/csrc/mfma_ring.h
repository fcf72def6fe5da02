// mfma_ring.h - the K loop of the MFMA kernels whose operands go straight into LDS.
#pragma once
#include <type_traits>

#include "mfma_common.h"

namespace tsh {
namespace {

// A block of RW x CW wavefronts multiplies BM rows by BN columns, 32 K values
// a step.  A step's operands fill one LDS slot: BM rows of 64 bytes, then
// BN x 64 bytes of weights as granules [chunk of 8 K values][column].
template <int BM, int BN, int RW, int CW> struct RingShape {
    static constexpr int NW = RW * CW;
    static constexpr int QB = BM / RW / 16;  // row blocks per wavefront
    static constexpr int NT = BN / CW / 16;  // column tiles per wavefront
    // Loads of 1 KB per step, and per wavefront: 16 rows of A each, or 64
    // granules of weights.  Where the wavefronts do not divide them some fetch
    // the same ones, so that every wavefront counts the same number of loads.
    static constexpr int AL = BM / 16;
    static constexpr int NA = (AL + NW - 1) / NW;
    static constexpr int WL = BN / 16;
    static constexpr int NB = (WL + NW - 1) / NW;
    static constexpr int PER = NA + NB;
    static constexpr int SLOT = (BM + BN) * 64;
    static_assert(QB >= 1 && NT >= 1 && BM % (16 * RW) == 0 && BN % (16 * CW) == 0, "whole MFMA tiles");
};

// acc = sum over `steps` steps (at least 2, even) of rows x columns.  load(j)
// issues load j < PER of the step to be fetched next into its slot,
// advance() moves on to the following step and slot; both go on past the last
// step (loads that fetch zeros or repeat).  On return every load has landed,
// but the block's wavefronts may still read the ring: the caller's barrier
// comes before it writes there.
template <int DT, int BM, int BN, int RW, int CW, int SLOTS, bool PP, class Load, class Advance>
__device__ __forceinline__ void ring_multiply(const unsigned char * s_ring, int steps, Load & load, Advance & advance,
                                              f32x4 (&acc)[RingShape<BM, BN, RW, CW>::QB]
                                                          [RingShape<BM, BN, RW, CW>::NT]) {
    using V = typename Mfma<DT>::V;
    using R = RingShape<BM, BN, RW, CW>;
    constexpr int NW = R::NW, QB = R::QB, NT = R::NT, PER = R::PER, SLOT = R::SLOT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wave % RW, cw = wave / RW;
    const int l16 = lane & 15, lg = lane >> 4;
    const uint32_t a_at = (uint32_t) (rw * QB * 1024 + (l16 * 4 + (lg ^ ((l16 >> 3) << 1))) * 16);
    const uint32_t b_at = (uint32_t) (BM * 64 + (lg * BN + cw * NT * 16 + l16) * 16);
    V fa[2][QB], fb[2][NT];
#pragma unroll
    for (int q = 0; q < QB; ++q)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[q][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
        for (int j = 0; j < PER; ++j) load(j);
        advance();
    }
    uint32_t rslot = 0;  // slot offset of the step whose fragments are read next
    if constexpr (PP) {
        static_assert(NW == 8, "two wavefronts per SIMD");
        // Phases alternate at barriers; a slot is refilled once both halves
        // have read it.
        auto mem = [&](bool issue) {
#pragma unroll
            for (int q = 0; q < QB; ++q) fa[0][q] = *(const V *) (s_ring + rslot + a_at + q * 1024);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) fb[0][nt] = *(const V *) (s_ring + rslot + b_at + nt * 256);
            if (issue) {
#pragma unroll
                for (int j = 0; j < PER; ++j) load(j);
                advance();
            }
            rslot = rslot == (SLOTS - 1) * SLOT ? 0 : rslot + SLOT;
        };
        auto mm = [&]() {
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int q = 0; q < QB; ++q)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[q][nt] = Mfma<DT>::mac(fa[0][q], fb[0][nt], acc[q][nt]);
            __builtin_amdgcn_s_setprio(0);
        };
        wait_vmcnt<(SLOTS - 1) * PER>();
        lds_barrier();
        const bool second = wave >= NW / 2;
        if (second) {
            lds_barrier();
            for (int s = 0; s < steps; ++s) {
                mem(s > 0);
                wait_vmcnt<(SLOTS - 2) * PER>();
                lds_barrier();
                __builtin_amdgcn_sched_barrier(0);
                mm();
                __builtin_amdgcn_sched_barrier(0);
                lds_barrier();
            }
        } else {
            for (int s = 0; s < steps; ++s) {
                mem(s > 0);
                lds_barrier();
                __builtin_amdgcn_sched_barrier(0);
                mm();
                __builtin_amdgcn_sched_barrier(0);
                wait_vmcnt<(SLOTS - 2) * PER>();
                lds_barrier();
            }
            lds_barrier();
        }
    } else {
        auto read_a = [&](int p, int q) { fa[p][q] = *(const V *) (s_ring + rslot + a_at + q * 1024); };
        auto read_b = [&](int p, int nt) { fb[p][nt] = *(const V *) (s_ring + rslot + b_at + nt * 256); };
        wait_vmcnt<(SLOTS - 1) * PER>();
        lds_barrier();
#pragma unroll
        for (int q = 0; q < QB; ++q) read_a(0, q);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) read_b(0, nt);
        rslot = SLOT;

        // One K step: fragments p hold step s; step s + 1's are read, step
        // s + SLOTS's rows and weights go into step s's slot (every wavefront
        // read its fragments of that slot before the barrier).
        auto step = [&](auto pc) {
            constexpr int p = decltype(pc)::value;
            wait_vmcnt<(SLOTS - 2) * PER>();
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < QB; ++q) {
                read_a(p ^ 1, q);
                if (q < NT) read_b(p ^ 1, q);
                if constexpr (QB < NT) {
                    if (q == QB - 1)
#pragma unroll
                        for (int nt = QB; nt < NT; ++nt) read_b(p ^ 1, nt);
                }
                if (q < PER) load(q);
                if constexpr (QB < PER) {
                    if (q == QB - 1)
#pragma unroll
                        for (int j = QB; j < PER; ++j) load(j);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[q][nt] = Mfma<DT>::mac(fa[p][q], fb[p][nt], acc[q][nt]);
                __builtin_amdgcn_sched_barrier(0);
            }
            advance();
            rslot = rslot == (SLOTS - 1) * SLOT ? 0 : rslot + SLOT;
        };
        for (int s = 0; s < steps; s += 2) {
            step(std::integral_constant<int, 0>());
            step(std::integral_constant<int, 1>());
        }
    }
    wait_vmcnt<0>();
}

}  // namespace
}  // namespace tsh
