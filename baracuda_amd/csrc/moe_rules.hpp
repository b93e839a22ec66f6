// moe_rules.hpp -- which grouped-MoE kernels a problem fits, and its tile shape.
#pragma once

#include <algorithm>

#include "gemm_ring.hpp"

namespace bk {

struct MoeFit {
    bool decode;     // the kernels of up to 64 pairs; their stores take any output alignment
    bool ring;       // 64- and 128-row tiles: 16-byte stores
    bool tiles256;   // 256 x 256 tiles: N % 256 == 0, whole 128-byte K stages
};

// kb: bytes of an input / weight row; operands: 16-byte aligned inputs and
// what the kind's epilogue needs; out16: 16-byte aligned output.  Byte offsets
// have to fit 32 bits (per input / per expert slab).
inline MoeFit moe_fit(int64_t x_rows, int N, int64_t kb, bool operands, bool out16) {
    const bool units = operands && kb % 16 == 0 && N % 8 == 0 && (x_rows + 1) * kb < (1ll << 31) &&
                       (int64_t)(N + 256) * kb < (1ll << 31);
    return {units, units && out16,
            operands && kb % mfma2::BK == 0 && N % mfma2::BN == 0 && x_rows * kb < (1ll << 31) && (int64_t)N * kb < (1ll << 31)};
}

// Column fragments (of 16) per workgroup of the decode kernel, for `pairs` of
// at most 64 pairs and rows of kb bytes.  g4: 64-column workgroups with rows, of
// about half of the experts that the pairs could touch.  us by 1 / 2 / 4
// fragments, bf16, weights rotated:
//  - above 32 pairs (two row fragments) 64 columns: 8 experts, 64 pairs, N = 7168,
//    K = 2048 56.1 / 56.7 / 54.0, N = 2048 18.4 / 17.5 / 14.2; 32 on the smallest
//    grids (N = 1024 11.0 / 10.4 / 11.3);
//  - up to 32, rows of at most 4 KiB: 64 columns (16 experts, 8 pairs, N = 2048, K =
//    2048 15.1 / 12.5 / 11.0), but 32 where every expert has rows and they fill the
//    chip (8 experts, 16 pairs, N = 7168, K = 2048 45.5 / 40.0 / 47.2; 16 experts, 32
//    pairs, K = 1024 53.8 / 35.7 / 39.7) or are few (2 pairs, N = 2048, K = 1024 6.1 /
//    5.5 / 6.1), and 16 for fewer still (N = 1024 4.9 / 5.3 / 6.0);
//  - rows of 8 KiB: 64 columns against 16 by the same lines (16 experts, 4 pairs, N =
//    7168 42.5 / 43.8 / 37.2; 16 pairs, N = 2048 34.4 / 35.8 / 39.0).
inline int moe_decode_width(int pairs, int E, int N, int64_t kb) {
    const int64_t g4 = (int64_t)((N + 63) / 64) * std::max(1, std::min(E, pairs) / 2);
    const bool deep = kb > 6144, full = pairs >= E && g4 >= 256;
    if (pairs > 32) return g4 <= 64 && !deep ? 2 : 4;
    if (deep) return g4 <= 64 || full ? 1 : 4;
    if (g4 < 32) return 1;
    return g4 <= 64 || full ? 2 : 4;
}

// Tile shape by the dense tiles' model: an expert's rows end in a tile that is
// half empty on average, so about size_m / TB + experts / 2 slots of TB rows
// (the counts are on the GPU).  256 x 256 only where its kernel takes the
// problem.
inline mfma2::RingTile moe_tile_shape(int size_m, int E, int N, int kb, bool whole) {
    int best = -1;
    float us = 0.0f;
    for (const int i : {mfma2::RT_64x128, mfma2::RT_128x128, mfma2::RT_128x256, mfma2::RT_256x256}) {
        if (i == mfma2::RT_256x256 && !whole) continue;
        const mfma2::RingCost &c = mfma2::kRingCost[i];
        const float slots = (float)size_m / (float)c.tm + 0.5f * (float)std::min(E, size_m);
        const float t = mfma2::ring_cost_tiles(c, (int64_t)(slots * (float)((N + c.tn - 1) / c.tn) + 0.5f), kb);
        if (best < 0 || t < us) {
            best = i;
            us = t;
        }
    }
    return (mfma2::RingTile)best;
}

}  // namespace bk
