// sfg_gemm_plan.hpp -- host only: which tile and K split a tiled MFMA product
// takes, by estimated time.  Shared by the launcher (sfg_gemm.hip) and the plan
// optimiser's cost estimates (runtime/sfg_optimizer.cpp).
#pragma once

#include <cstddef>
#include <cstdint>

#include "../../include/sfg_hip.h"

namespace sfg {

// With bf16 weights kRingTileV and kRingTileDma are gemm_dma_kernel's 256 x 256
// (64-k slabs) and 256 x 128 (two workgroups per CU) tiles; the rest, int8's 256 x
// 256 among them, are gemm_ring_kernel's.  `part` bytes of split-K partial sums
// ([splits][m][B rows] fp32) come from the caller's workspace; `us` is the estimate.
enum { kRingTileV = 1, kRingTile256x128, kRingTile128x128, kRingTile64x128, kRingTile128x64, kRingTile64x64,
       kRingTileSmall /* fp32 only: gemm_f32_small_kernel */, kRingTileDma };
constexpr size_t kRingNoLimit = ~size_t(0);
constexpr int64_t kRingBigMinRows = 1024;  // from here on no dense product splits K
constexpr int kRingCus = 256;
constexpr size_t kRingMaxPart = size_t(64) << 20;  // bytes of split-K partials

struct RingAsk {
    int b_dtype;
    int64_t m, n, k;
    int epi, c_dtype;   // sfg_epilogue (or the QKV one), output type
    int groups;         // 1: dense
    bool may_split, allow_v, allow_dma;
    size_t workspace;   // bytes
};
struct RingPlan {
    int tile, bm, bn, splits;
    size_t part;
    float us;
};

// What a tile costs: `slab` us per k-slab (64 k, fp32 32) of a CU that has the
// chip to itself and `busy` more with every CU at work, `tile` us around the slabs
// of a round, `kb` us per KB of output and residual with every CU at work, `start`
// us per launch.  Least squares over 12500 seeded products (m 65 .. 8192, n 1 ..
// 14336, k 64 .. 12000), each timed on every tile: errors of 3 - 10% (2 sigma
// 20% on 256 x 128 as two workgroups).  From 1024 rows up the choice they give
// costs 3% (bf16), 0.3% (int8) and 0.2% (fp32) more than the best tile of each
// product in sum; by slab time alone it was 7, 2 and 5%.  Each tile wins somewhere: 64
// x 64 29% of the bf16 and 26% of the fp32 products without GLU, the narrow ones (1295 x
// 320 x 4128 20.3 us, the next tile 29.6).
struct RingTile {
    int tile, bm, bn, per_cu;
    bool glu;
    float slab, busy, around, kb, start;
};
constexpr RingTile kRingBf16[] = {
    {kRingTileV, 256, 256, 1, true, 0.87f, 0.49f, 7.5f, 0.024f, 6.0f},
    {kRingTileDma, 256, 128, 2, true, 0.815f, 1.008f, 9.6f, 0.039f, 2.9f},
    {kRingTile256x128, 256, 128, 1, true, 0.478f, 0.286f, 6.8f, 0.021f, 1.8f},
    {kRingTile128x128, 128, 128, 1, true, 0.305f, 0.171f, 4.2f, 0.019f, 1.5f},
    {kRingTile64x128, 64, 128, 1, true, 0.219f, 0.086f, 4.6f, 0.011f, 1.2f},
    {kRingTile128x64, 128, 64, 1, false, 0.236f, 0.085f, 6.4f, 0.001f, 1.1f},
    {kRingTile64x64, 64, 64, 1, false, 0.194f, 0.f, 1.85f, 0.002f, 3.2f},
};
constexpr RingTile kRingI8[] = {
    {kRingTileV, 256, 256, 1, true, 1.06f, 0.41f, 9.0f, 0.022f, 6.0f},
    {kRingTile256x128, 256, 128, 1, true, 0.668f, 0.225f, 6.7f, 0.020f, 2.2f},
    {kRingTile128x128, 128, 128, 1, true, 0.440f, 0.107f, 7.25f, 0.012f, 1.5f},
    {kRingTile64x128, 64, 128, 1, true, 0.396f, 0.049f, 4.8f, 0.009f, 1.3f},
    {kRingTile128x64, 128, 64, 1, false, 0.355f, 0.037f, 7.0f, 0.f, 1.0f},
    {kRingTile64x64, 64, 64, 2, false, 0.315f, 0.085f, 4.2f, 0.011f, 1.3f},
};
constexpr RingTile kRingF32[] = {
    {kRingTile256x128, 256, 128, 1, true, 3.484f, 0.222f, 6.3f, 0.024f, 2.1f},
    {kRingTile128x128, 128, 128, 1, true, 1.802f, 0.102f, 4.3f, 0.020f, 1.6f},
    {kRingTile64x128, 64, 128, 1, true, 0.943f, 0.047f, 4.6f, 0.013f, 1.5f},
    {kRingTile128x64, 128, 64, 1, false, 0.935f, 0.050f, 6.5f, 0.001f, 1.2f},
    {kRingTile64x64, 64, 64, 1, false, 0.498f, 0.f, 1.9f, 0.f, 3.3f},
    {kRingTileSmall, 32, 32, 1, true, 0.140f, 0.004f, 3.4f, 0.035f, 1.6f},
};
// 65 .. 1023 dense rows of bf16 / int8 weights, the tile and the K split together,
// and grouped products.  Microseconds per slab as measured inside layers, where the
// weights come from HBM; a round takes 3 us more, a split its reduce launch and one
// write and one read of the partials (4 TB/s).  Over 4600 dense products this rule
// costs 4 - 5% more than the best tile and split of each, over 5300 grouped ones (1 -
// 64 groups, even and skewed) 3 - 8%.
struct RingSlab {
    int tile, bm, bn, per_cu;
    bool glu;
    float us_bf16, us_i8;
};
constexpr RingSlab kRingSlabs[] = {
    {kRingTileV, 256, 256, 1, true, 1.55f, 1.60f},
    {kRingTile256x128, 256, 128, 1, true, 1.10f, 1.05f},
    {kRingTile128x128, 128, 128, 1, true, 0.69f, 0.64f},
    {kRingTile64x128, 64, 128, 1, true, 0.52f, 0.52f},
    {kRingTile128x64, 128, 64, 1, false, 0.52f, 0.48f},
    {kRingTile64x64, 64, 64, 2, false, 0.56f, 0.50f},
};

inline bool ring_is_glu(int epi) { return epi == SFG_EPI_SWIGLU || epi == SFG_EPI_GLU_SILU_UP; }

inline RingPlan ring_plan_slabs(const RingAsk& q) {
    const bool glu = ring_is_glu(q.epi);
    const int64_t slabs = (q.k + 63) / 64, nb = glu ? 2 * q.n : q.n;
    RingPlan best{};
    for (const RingSlab& t : kRingSlabs) {
        if ((glu && !t.glu) || (t.tile == kRingTileV && (!q.allow_v || (q.b_dtype == SFG_BF16 && q.k % 64 != 0)))) continue;
        const float us = q.b_dtype == SFG_I8 ? t.us_i8 : t.us_bf16;
        const int64_t cols = glu ? t.bn / 2 : t.bn;
        int64_t rows = (q.m + t.bm - 1) / t.bm;
        if (q.groups > 1) {
            // half a tile of padding per group on average, and no less than a tile
            // for each group that has a row
            const int64_t live = q.groups < q.m ? q.groups : q.m;
            rows += q.groups / 2;
            if (rows < live) rows = live;
        }
        const int64_t tiles = rows * ((q.n + cols - 1) / cols);
        for (int s = 1; s <= 16; ++s) {
            const size_t part = s > 1 ? static_cast<size_t>(s) * q.m * nb * 4 : 0;
            if (s > 1 && (!q.may_split || q.groups > 1 || t.tile == kRingTileV || q.n % 4 != 0 || slabs / s < 4 || part > kRingMaxPart ||
                          part > q.workspace))
                break;
            const int64_t room = static_cast<int64_t>(kRingCus) * t.per_cu;
            const float rounds = static_cast<float>((tiles * s + room - 1) / room);
            float time = rounds * (static_cast<float>((slabs + s - 1) / s) * us + 3.f);
            if (s > 1) time += 4.f + static_cast<float>(part) * 2.f / 4.0e6f;
            if (best.tile == 0 || time < best.us) best = RingPlan{t.tile, t.bm, t.bn, s, part, time};
        }
    }
    return best;
}

template <size_t N>
RingPlan ring_plan_whole(const RingAsk& q, const RingTile (&table)[N]) {
    const bool glu = ring_is_glu(q.epi);
    const int64_t slab_k = q.b_dtype == SFG_F32 ? 32 : 64;
    const float slabs = static_cast<float>((q.k + slab_k - 1) / slab_k);
    const bool residual = q.epi == SFG_EPI_RESIDUAL;
    const int out = (q.c_dtype == SFG_F32 ? 4 : 2) + (residual ? 4 : 0);  // bytes per output
    RingPlan best{};
    for (const RingTile& t : table) {
        if ((glu && !t.glu) || (t.tile == kRingTileV && (!q.allow_v || (q.b_dtype == SFG_BF16 && q.k % 64 != 0))) ||
            (t.tile == kRingTileDma && (!q.allow_dma || q.m < kRingBigMinRows || q.k % 64 != 0)))
            continue;
        const bool small = t.tile == kRingTileSmall;  // 32 output columns either way
        const int64_t cols = glu && !small ? t.bn / 2 : t.bn;
        const int64_t tiles = ((q.m + t.bm - 1) / t.bm + (q.groups > 1 ? q.groups / 2 : 0)) * ((q.n + cols - 1) / cols);
        const int64_t room = static_cast<int64_t>(kRingCus) * t.per_cu;
        const float rounds = static_cast<float>((tiles + room - 1) / room);
        const float used = tiles < room ? static_cast<float>(tiles) / static_cast<float>(room) : 1.f;
        float around = t.around;
        // a residual is read before the stores; 128 x 128 a wave with 2-byte stores
        // has no registers to do so for the whole block
        if (t.tile == kRingTileV && residual) around += q.c_dtype == SFG_F32 ? 2.f : 12.f;
        const float us = t.start + rounds * ((small && glu ? 2.f : 1.f) * slabs * (t.slab + t.busy * used) + around +
                                             t.kb * used * static_cast<float>(t.bm * cols * out) / 1024.f);
        if (best.tile == 0 || us < best.us) best = RingPlan{t.tile, t.bm, t.bn, 1, 0, us};
    }
    return best;
}

inline RingPlan ring_plan(const RingAsk& q) {
    if (q.b_dtype == SFG_F32) return ring_plan_whole(q, kRingF32);
    if (q.groups > 1 || q.m < kRingBigMinRows) return ring_plan_slabs(q);
    return q.b_dtype == SFG_I8 ? ring_plan_whole(q, kRingI8) : ring_plan_whole(q, kRingBf16);
}

// Products of few slabs and several rounds of tiles, where it counts how many
// workgroups a CU holds at once: the 128 x 128 register-staged tile (41 KB of LDS)
// instead of one ring a CU.  Its speed against the best ring tile: bf16 GLU, K 32,
// over 512 tiles 1.6 x, K 96 1.2 x (without GLU, or in one round, 0.3 - 1.0 x); int8 groups
// of up to 32 rows, K 256 GLU 1.3 - 1.6 x, K 512 1.4 x.
inline bool gemm_short_k(int b_dtype, int64_t m, int64_t n, int64_t k, bool glu, int groups) {
    const int64_t cols = (n + (glu ? 63 : 127)) / (glu ? 64 : 128);
    if (groups == 1) return b_dtype == SFG_BF16 && glu && k <= 96 && (m + 127) / 128 * cols > kRingCus;
    if (m >= kRingBigMinRows || groups * cols < kRingCus) return false;
    if (b_dtype == SFG_I8)
        return glu ? (k <= 512 && m <= 64 * groups) || (k <= 1024 && m <= 16 * groups) : k <= 384 && m <= 32 * groups;
    return glu && k <= 256 && m <= 32 * groups;
}

// Grouped products of more rows in a group than one pass of the skinny kernel
// takes (32): the ring tiles read each weight once, the skinny kernel once per
// pass.  Over 7250 products of 1 .. 64 groups and up to 512 rows, ring against
// skinny: largest group up to 32 rows 0.83 x the speed, 33 .. 48 1.16 x, more 1.42 x.
// The host knows the average only, and routed groups are uneven, so from four
// groups up the line lies lower (24 - 28 rows on average: bf16 without GLU 0.8 -
// 1.4 x, mean 1.1; 28 - 32: GLU 0.9 - 1.8, int8 0.9 - 2.2).
inline int64_t gemm_ring_rows(int b_dtype, bool glu, int groups) {
    return groups < 4 ? 33 : (b_dtype == SFG_I8 || glu ? 28 : 24);
}

// fp32 GLU products of one or two slabs and few 32 x 32 tiles: the VALU kernel (K 32 up
// to 512 tiles 1.1 - 1.3 x as fast as the MFMA tiles, K 64 up to 128 1.1 - 1.3 x;
// without GLU 0.5 - 1.0 x).
inline bool gemm_f32_short_k(int64_t m, int64_t n, int64_t k, bool glu) {
    return glu && k <= 64 && (m + 31) / 32 * ((n + 31) / 32) * k * k <= 512 * 32 * 32;
}

}  // namespace sfg
