// gemm_ring.hpp -- mid-size block tiles for the RCR GEMMs: a ring of LDS
// stages with the next stage's DMA spread between the MFMAs, and the rule
// that picks the tile.
//
// What bounds these tiles (int8, one box): one 1 KiB LDS-DMA instruction
// takes a CU about 26 clocks, so a 128 x 128 stage's 32 take as long as
// 830 clocks of the 512 its MFMAs need, and a wave that issues its DMAs in
// one burst stalls in front of its MFMAs for all of that.  Reading the
// stage's fragments first and issuing one DMA per few MFMAs overlaps the
// two: 1024 x 4096 x 4096 on 256 tiles of 128 x 128, 23.5 us with the burst
// ahead of the fragment reads, 21.0 with the burst behind them, 19.1 spread
// (26.5 us for the two-stage loop of gemm_mfma2.hpp).  A third stage hides
// the load latency of a tile that has the CU to itself; a fourth gives
// nothing more (19.2 us).
#pragma once

#include "gemm_mfma2.hpp"

namespace bk {
namespace mfma2 {

// One DMA instruction of a stage: I < ROWS_PER_WAVE / 8 moves A row group I,
// the others B row groups.
template <class C, int I>
__device__ __forceinline__ void dma_piece(int8_t *stage, const DmaRows<false, false> &d, int kbyte) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NA = C::ROWS_PER_WAVE / 8;
    if constexpr (I < NA) {
        const int soff = __builtin_amdgcn_readfirstlane(kbyte + I * d.a.row_stride);
        dma16(d.a.rsrc, (I & 1) ? d.a.odd : d.a.even, soff, stage + (wave * C::ROWS_PER_WAVE + I * 8) * BK);
    } else {
        constexpr int J = I - NA;
        const int soff = __builtin_amdgcn_readfirstlane(kbyte + J * d.b.row_stride);
        dma16(d.b.rsrc, (J & 1) ? d.b.odd : d.b.even, soff,
              stage + C::OPER + (wave * C::ROWS_PER_WAVE_B + J * 8) * BK);
    }
}

// Gathered A rows (MoE): one per-lane offset per A piece.
template <class C, int I>
__device__ __forceinline__ void dma_piece(int8_t *stage, const DmaRows<true, false> &d, int kbyte) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NA = C::ROWS_PER_WAVE / 8;
    if constexpr (I < NA) {
        dma16(d.a.rsrc, d.a.off[I], __builtin_amdgcn_readfirstlane(kbyte), stage + (wave * C::ROWS_PER_WAVE + I * 8) * BK);
    } else {
        constexpr int J = I - NA;
        const int soff = __builtin_amdgcn_readfirstlane(kbyte + J * d.b.row_stride);
        dma16(d.b.rsrc, (J & 1) ? d.b.odd : d.b.even, soff,
              stage + C::OPER + (wave * C::ROWS_PER_WAVE_B + J * 8) * BK);
    }
}

// Row-major B (TBN = 256 columns, 8 waves): B pieces of four k-rows.
template <class C, int I>
__device__ __forceinline__ void dma_piece(int8_t *stage, const DmaRowsRrr &d, int kbyte) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NA = C::ROWS_PER_WAVE / 8;
    static_assert(C::TBN == BN && C::WAVES == 8, "row-major B tiles are 256 columns wide");
    if constexpr (I < NA) {
        const int soff = __builtin_amdgcn_readfirstlane(kbyte + I * d.a.row_stride);
        dma16(d.a.rsrc, (I & 1) ? d.a.odd : d.a.even, soff, stage + (wave * C::ROWS_PER_WAVE + I * 8) * BK);
    } else {
        constexpr int J = I - NA;
        const int soff = __builtin_amdgcn_readfirstlane((kbyte + 4 * J) * d.b.ld);
        dma16(d.b.rsrc, (J & 1) ? d.b.odd : d.b.even, soff, stage + C::OPER + (wave * 16 + 4 * J) * BN);
    }
}

template <class C, int I0, int I1, class D>
__device__ __forceinline__ void dma_pieces(int8_t *stage, const D &d, int kbyte) {
    if constexpr (I0 < I1) {
        dma_piece<C, I0>(stage, d, kbyte);
        dma_pieces<C, I0 + 1, I1>(stage, d, kbyte);
    }
}

// MFMA t of a stage's sub-steps, then the DMA pieces due after it.
template <class P, int T, int SPREAD, class D>
__device__ __forceinline__ void ring_mma(AccTile<P> &acc, const Frags<P> &f0, const Frags<P> &f1, int8_t *nxt, const D &d,
                                         int kbyte) {
    typedef typename P::Cfg C;
    constexpr int SUB = P::H * P::TI * P::TJ, TOT = P::SUBS * SUB, NI = C::DMA_PER_STAGE;
    if constexpr (T < TOT) {
        constexpr int r = T % SUB, h = r / (P::TI * P::TJ), j = r / P::TI % P::TJ, i = r % P::TI;
        const Frags<P> &f = T < SUB ? f0 : f1;
        P::mma(acc[i][j], f.b[j], f.a[i], h);
        constexpr int p0 = (T / SPREAD < NI ? T / SPREAD : NI);
        constexpr int p1 = ((T + 1) / SPREAD < NI ? (T + 1) / SPREAD : NI);
        constexpr int pe = T + 1 == TOT ? NI : p1;
        if constexpr (pe > p0) {
            __builtin_amdgcn_sched_barrier(0);
            dma_pieces<C, p0, pe>(nxt, d, kbyte);
            __builtin_amdgcn_sched_barrier(0);
        }
        ring_mma<P, T + 1, SPREAD>(acc, f0, f1, nxt, d, kbyte);
    }
}

// K loop over a ring of DEPTH stage buffers at `lds` (DEPTH * C::STAGE bytes,
// 1 KiB aligned), DEPTH - 1 stages in flight: the wait for stage kt leaves
// the later stages' DMAs outstanding (they complete in issue order), and the
// one barrier per stage both publishes stage kt and frees the buffer of
// stage kt - 1 for the DMA of stage kt + DEPTH - 1.  Ends with a barrier.
template <class P, int DEPTH, int SPREAD, class D>
__device__ __forceinline__ void mainloop_ring(int8_t *lds, D d, int K, AccTile<P> &acc) {
    typedef typename P::Cfg C;
    static_assert(DEPTH >= 2 && DEPTH <= 4 && DEPTH * C::STAGE <= 160 * 1024, "stage ring");
    static_assert(!P::SUMS && !P::FLIP, "the ring loop takes signed and float operands");
    constexpr int NI = C::DMA_PER_STAGE;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wave_m = wave / C::WAVES_N, wave_n = wave % C::WAVES_N;
#pragma unroll
    for (int i = 0; i < P::TI; ++i)
#pragma unroll
        for (int j = 0; j < P::TJ; ++j) acc[i][j] = P::zero();
    const int KT = (K + BK - 1) / BK;
    Frags<P> f0, f1;
    auto prep = [&](int kt) {
        if ((kt + 1) * BK > K) {
            if (kt >= KT) {
                d.a.rsrc[2] = 0;
                d.b.rsrc[2] = 0;
            } else {
                mask_tail<C, C::ROWS_PER_WAVE>(d.a, kt * BK, K);
                mask_tail<C, C::ROWS_PER_WAVE_B>(d.b, kt * BK, K);
            }
        }
    };
    for (int s = 0; s < DEPTH - 1; ++s) {
        prep(s);
        dma_stage<C>(lds + s * C::STAGE, d, s * BK);
    }
    int cur = 0, nxt = (DEPTH - 1) * C::STAGE;       // byte offsets of the ring slots
    for (int kt = 0; kt < KT; ++kt) {
        prep(kt + DEPTH - 1);
        wait_vmcnt<(DEPTH - 2) * NI>();
        __syncthreads();
        const int8_t *st = lds + cur;
        load_frags<P>(f0, st, 0, wave_m, wave_n, lane);
        if constexpr (P::SUBS == 2) load_frags<P>(f1, st, 1, wave_m, wave_n, lane);
        if constexpr (SPREAD == 0) {
            __builtin_amdgcn_sched_barrier(0);
            dma_pieces<C, 0, NI>(lds + nxt, d, (kt + DEPTH - 1) * BK);
            __builtin_amdgcn_sched_barrier(0);
            mma_block<P, 0, P::TJ>(acc, f0);
            if constexpr (P::SUBS == 2) mma_block<P, 0, P::TJ>(acc, f1);
        } else {
            ring_mma<P, 0, SPREAD>(acc, f0, f1, lds + nxt, d, (kt + DEPTH - 1) * BK);
        }
        nxt = cur;
        cur = cur + C::STAGE == DEPTH * C::STAGE ? 0 : cur + C::STAGE;
    }
    wait_dma();
    __syncthreads();
}

// ---- which tile -------------------------------------------------------------
// Tiles of the GEMMs.  The first five run the ring loop (LDS of all stages;
// 64-row tiles leave room for two workgroups per CU), 256 x 256 the two-stage
// kernel of gemm_mfma2.hpp, or the ring with two stages when K % 128 != 0.
enum RingTile { RT_64x64, RT_64x128, RT_128x128, RT_128x256, RT_192x256, RT_256x256 };
struct RingCost {
    int tm, tn;
    float stage;    // us per 128-byte stage of K, alone on its CU
    float paired;   // ... of two workgroups sharing a CU (0: LDS holds one)
    float fixed;    // us per round besides: launch, first loads, epilogue
};
// Measured over K = 1024 .. 8000 (int8, bf16 out, weights from HBM).
constexpr RingCost kRingCost[] = {
    {64, 64, 0.20f, 0.39f, 3.6f},   {64, 128, 0.30f, 0.56f, 3.9f},  {128, 128, 0.47f, 0.0f, 3.5f},
    {128, 256, 0.65f, 0.0f, 5.1f},  {192, 256, 1.00f, 0.0f, 5.8f},  {256, 256, 1.23f, 0.0f, 6.7f},
};

// Time of one tile shape: rounds over the 256 CUs, each of `fixed` plus the
// K stages.  The figures rank the shapes; a full chip is slower than they
// say (power), all shapes alike.  Picks, against the best of the six measured
// (us): 777 x 11008 x 4096 192x256 47.3 (256x256 49.4, 128x128 51.8), 1500 x
// 5120 x 2880 128x256 23.7 (192x256 31.6, 128x128 28.9), 810 x 2352 x 1856
// 64x128 9.3 (128x128 10.9), 200 x 11008 x 4096 128x128 20.3 (64x128 24.3),
// 3072 x 4096 x 4096 192x256 44.3 (256x256 47.0), 4096^3 256x256 55.5.
inline float ring_cost_tiles(const RingCost &c, int64_t tiles, int kbytes) {
    const float kt = (float)((kbytes + BK - 1) / BK);
    const int64_t per_cu = (tiles + 255) / 256;
    if (c.paired == 0.0f) return (float)per_cu * (c.fixed + kt * c.stage);
    const int64_t pairs = per_cu / 2;
    return (float)pairs * (c.fixed + kt * c.paired) + (float)(per_cu % 2) * (c.fixed + kt * c.stage);
}

inline float ring_cost(const RingCost &c, int M, int N, int kbytes) {
    return ring_cost_tiles(c, (int64_t)((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn), kbytes);
}

// `first`: the smallest shape the caller has (row-major B tiles are 256
// columns wide, so they start at 128 x 256).  Past three rounds of 256 x 256
// those: the last round overlaps the others, so that its idle CUs cost less than
// the model's whole round (int8, 3072 x 17920 x 4096, 3.3 rounds: 214 us, 225 on
// 128 x 256; e4m3, 3072 x 28672 x 2048, 5.25 rounds: 174, 186 on 192 x 256; at 2.3
// rounds, 600 x 50176 x 4096, 178 against 141 on 128 x 256).
inline RingTile ring_tile(int M, int N, int kbytes, float *cost = nullptr, RingTile first = RT_64x64) {
    if ((int64_t)((M + 255) / 256) * ((N + 255) / 256) > 3 * 256) {
        if (cost) *cost = ring_cost(kRingCost[RT_256x256], M, N, kbytes);
        return RT_256x256;
    }
    int best = first;
    float us = 0.0f;
    for (int i = first; i <= RT_256x256; ++i) {
        const float t = ring_cost(kRingCost[i], M, N, kbytes);
        if (i == first || t < us) {
            best = i;
            us = t;
        }
    }
    if (cost) *cost = us;
    return (RingTile)best;
}

// Row blocks of the staged last-rows kernels instead of tiles (33-512 rows):
// they split K over their waves, which a tile does not.
//  - Where 64 x 64 tiles would leave half of the CUs idle.  us, int8, blocks
//    against the best tile: 200 x 1024 x 4096 7.0 / 9.8, 128 x 4096 x 4096 8.5 /
//    10.0, 512 x 1024 x 4096 8.3 / 10.1, 128 x 4096 x 14336 25.9 / 33; past the
//    line 200 x 4096 x 4096 11.5 / 10.2, 384 x 2048 x 1024 5.7 / 4.9, 128 x 8192
//    x 4096 14.9 / 11.7, 64 x 14336 x 4096 17.8 / 15.7.
//  - Past one round of 64 x 64 tiles with a deep K, where the tiles wait for
//    the weights: 160 x 6144 x 8192 27.3 / 32.0, 256 x 8192 x 8192 32.8 / 34.4, 384
//    x 4096 x 14336 50.1 / 56.3, 300 x 5120 x 14336 45.1 / 57.0, 100 x 14336 x 8192
//    33.7 / 35.5, but 384 x 4096 x 8192 26.6 / 24.4; 80 x 14336 x 4096 19.7 / 20.3,
//    100 x 14336 x 4096 20.8 / 20.6.  Within one round later: 160 x 5120 x 14336
//    32.0 / 34.5, 200 x 4096 x 11264 24.2 / 26.3, 256 x 4096 x 11264 28.4 / 26.7,
//    256 x 4096 x 14336 35.0 / 35.9, 128 x 5120 x 14336 42.8 / 37.0, 300 x 2048 x
//    14336 31.7 / 26.8.
// There only as one round of workgroups (launch_row_blocks checks that for more
// than 128 rows): 100 x 11008 x 14336 as 344 of them 69.3 / 58.4.
inline bool row_blocks_pay(int M, int N, int kbytes) {
    const int64_t t64 = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
    if (t64 <= 128) return true;
    if (M <= 128 && N / (16 * last_rows_col_frags(N)) > 256) return false;
    if (t64 <= 256) return M > 128 && (M <= 224 ? kbytes >= 11264 : M <= 256 && kbytes > 12288);
    return kbytes >= (M <= 96 ? 4096 : M <= 256 ? 8192 : 9216);
}

// Whole 256-row tiles and a last-rows pass for more than 512 rows, against
// the cheapest tile over all rows: the pass reads the weights once more, at
// about 3.6 TB/s behind the tiles, and takes at least a launch.
inline bool last_rows_pay(int M, int N, int kbytes, int rem) {
    float all;
    ring_tile(M, N, kbytes, &all);
    return ring_cost(kRingCost[RT_256x256], M - rem, N, kbytes) + 3.0f + (float)N * (float)kbytes / 3.6e6f < all;
}

// A last round of `tail` 256 x 256 tiles behind `full` others split along K (with
// the caller's workspace) against the tiles and row blocks without one.  us, int8
// to bf16, split / without, weights rotated:
//  - No whole round: the split takes 26-30 us at any K for its slots and second
//    launch.  512 x 512 x 8192 31.0 / 11.5, 600 x 1024 x 8192 30.5 / 19.2, 768 x
//    1152 x 16384 40.5 / 34.0, but 768 x 768 x 20480 37.0 / 44.8, 200 x 520 x 24576
//    40.6 / 50.4; against row blocks, which split K themselves, 256 x 256 x 24576
//    44.8 / 27.5, 512 x 1024 x 20480 35.1 / 32.8.
//  - One whole round: N = 4096, K = 4096, M = 4296 / 4864 / 5120 / 6144 81.2 / 85.4,
//    91.0 / 90.4, 93.3 / 89.5, 107.0 / 101.7; M = 4296, K = 2048 / 3072 51.3 / 47.0,
//    63.7 / 65.5; K = 6144, M = 4864 / 5120 / 6144 121.1 / 127.9, 124.7 / 127.7, 144.4
//    / 146.0.
//  - Two: M = 8448 K = 4096 143.1 / 132.8, 8192 244.0 / 242.7, 14336 405.3 / 414.5, M
//    = 9216 K = 8192 262.1 / 252.8.  More, where the tiles are 256 x 256 too: M =
//    12544, K = 4096 / 8192 190.6 / 201.6, 337.7 / 376.6.
inline bool tail_split_pays(int M, int N, int kbytes, int full, int tail) {
    if (full == 0) {
        const bool blocks = N % 16 == 0 && M <= 512 && (int64_t)((M + 63) / 64) * ((N + 63) / 64) <= 128;
        return kbytes > (blocks ? 24576 : 16384);
    }
    if (full <= 256) return kbytes >= (tail <= 16 ? 3072 : 6144);
    return full > 512 || kbytes >= 14336;
}

}  // namespace mfma2
}  // namespace bk
