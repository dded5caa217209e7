// The K-split sum of the mid-batch and wide-tile GEMMs, as a launch of its own.
#pragma once

#include "sg_mid_kernel.h"

namespace sg {

// Second launch of a mid-batch GEMM whose split-K sum was deferred: every wave adds the split_k partials of
// kReduceFrags 16 x 16 fragments of the output in split order - what the last workgroup to arrive does in the single
// launch, so the result bits are the same - and applies scale, row and column factors and the rounding.  A wave's
// work is a chain of round trips (partials, scale, store), so it takes several fragments at once and requests all
// their partials of a split before it adds any: with one fragment per wave the launch took 7-12 us for 8-33 MB of
// partials that the GEMM had just left in the caches.  The tile geometry comes as run-time values: rgw x mh
// fragments per wave of the GEMM, wn x 2 waves per tile.
// FACTORS: there are row or column factors (requested ahead of the partials, in 34 registers that the other build does not
// hold: five waves a SIMD instead of eight).
// FRAGS, BATCH: fragments of a wave and splits it asks for at once, up to eight 1 KB loads in flight.  Four and two; one and four or
// eight where four would make so few waves that the launch is the chain of their round trips (launch_mid_reduce).
constexpr int kReduceFrags = 4;
template <bool FACTORS, int FRAGS, int BATCH>
__global__ void __launch_bounds__(256) mid_reduce_kernel(const StreamArgs a, int rgw, int mh, int wn) {
    const int fr = rgw * mh, frags_wg = 2 * wn * fr;   // fr is a multiple of FRAGS (launch_mid_reduce)
    const int lane = lane_id();
    // a workgroup takes 4 * FRAGS consecutive fragments of one tile; the workgroups of a weight tile sit on the
    // XCD that computed it (the grid is n_tiles * m_tiles * chunks workgroups, chunks per tile)
    const int chunks = (frags_wg + 4 * FRAGS - 1) / (4 * FRAGS);   // (the last one may have idle waves)
    int pos;
    const int tile_n = xcd_weight_tile((int)blockIdx.x, (int)gridDim.x, a.m_tiles * chunks, a.n_tiles, pos);
    const int tile_m = pos / chunks, chunk = pos - tile_m * chunks;
    if (tile_n >= a.n_tiles || tile_m >= a.m_tiles) return;
    const unsigned tile_id = (unsigned)(tile_m * a.n_tiles + tile_n);
    const unsigned rem = (unsigned)((chunk * 4 + wave_id()) * FRAGS);     // (wave of the tile, fragment of the wave)
    if (rem >= (unsigned)frags_wg) return;
    const int wave = (int)rem / fr, f0 = (int)rem - wave * fr;
    const int wq = wave % wn, wm = wave / wn;
    const int r = lane & 15, g = lane >> 4;
    const float scale = scalar_scale(a);
    auto place = [&](int j, int& m_idx, int& n_idx) __attribute__((always_inline)) {
        const int f = f0 + j, rg = f / mh, mb = f - rg * mh;
        m_idx = tile_m * (32 * mh) + (wm * mh + mb) * 16 + r;
        n_idx = tile_n * (16 * rgw * wn) + (wq * rgw + rg) * 16 + 4 * g;
    };
    f32x4 col[FRAGS];
    float row[FRAGS];
    if constexpr (FACTORS) {
#pragma unroll
        for (int j = 0; j < FRAGS; j++) {
            int m_idx, n_idx;
            place(j, m_idx, n_idx);
            col[j] = col_scale_ahead(a, n_idx);
            row[j] = row_scale_ahead(a, m_idx);
        }
    }
    const f32x4* p = reinterpret_cast<const f32x4*>(a.ws + ((size_t)tile_id * a.split_k) * ((size_t)frags_wg * 256) +
                                                    (size_t)wave * (fr * 256) + (size_t)f0 * 256) + lane;
    const size_t split_stride = (size_t)frags_wg * 64;
    f32x4 v[FRAGS];
#pragma unroll
    for (int j = 0; j < FRAGS; j++) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (FRAGS > 1) {
#pragma unroll BATCH
        for (int sp = 0; sp < a.split_k; sp++) {
            f32x4 t[FRAGS];
#pragma unroll
            for (int j = 0; j < FRAGS; j++) t[j] = p[(size_t)sp * split_stride + j * 64];
#pragma unroll
            for (int j = 0; j < FRAGS; j++) v[j] += t[j];
        }
    } else {
        for (int sp = 0; sp < a.split_k; sp += BATCH) {   // (behind the last split it is read again and not added)
            f32x4 t[BATCH];
#pragma unroll
            for (int i = 0; i < BATCH; i++) t[i] = p[(size_t)(sp + i < a.split_k ? sp + i : a.split_k - 1) * split_stride];
#pragma unroll
            for (int i = 0; i < BATCH; i++)
                if (sp + i < a.split_k) v[0] += t[i];
        }
    }
#pragma unroll
    for (int j = 0; j < FRAGS; j++) {
        int m_idx, n_idx;
        place(j, m_idx, n_idx);
        if constexpr (FACTORS) {
            store_fragment(a, v[j], scale, m_idx, n_idx, row[j], col[j]);
        } else {
            v[j] *= scale;
            store_scaled(a, v[j], m_idx, n_idx);
        }
    }
}

}  // namespace sg
