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
