// Mid-batch FP8 GEMM for rows that start off their 128-byte lines:  D[m,n] = scale * sum_k A[m,k] * B[n,k].
//
// What bounds a mid-batch launch is the rate at which a CU's L1 takes lines in (sg_mid_kernel.h), and the mid-batch kernel's
// stage is 128 bytes of K of every row: where a row's pitch - of the weights, or k itself, the activations' - is not a
// multiple of 128, every such piece lies on two lines, both are asked for, and the next stage asks for the second again.
// 128 x 8192 x 8208 took 36.7 us where 128 x 8192 x 8320 takes 24.2.
//
// So the stages here follow the lines, row by row: line j of a row are the 128 bytes from 128 * j on, counted from the start
// of the line its first byte lies on, and a stage's DMA fetches line j of every row of the tile, whatever columns that is.
// A row that starts `shift` 16-byte pieces into its line then holds piece p of K block b at piece p + shift of its byte
// stream, on line b or b + 1: the shift is applied where the operand is read from LDS.  Pitches are multiples of 16 bytes, so
// 16 rows on is a multiple of 256 bytes on: all fragments of an operand have the same shifts, one per lane, and a lane's two
// pieces of a block come from slot b or b + 1 by two constants.  (The LDS swizzle of sg_mid_kernel.h stays conflict-free: with d = pitch / 16
// the sixteen lanes of a pass read pieces (g + c + r * d) & 7 of rows r, and x -> (a + 2 d x) ^ x permutes 0..7.)
//
// Nothing outside a row is read: a piece before its row's first byte or behind its last is replaced by the first or last
// piece of the same row.  The former are never used; the latter meet zeroed activations, and a NaN among them is one that the
// row's last block holds as well.
//
// Waves, K splits (summed by mid_reduce_kernel) and the rotated start of K are the mid-batch kernel's; both operands have the
// same ring, as deep as 160 KB allow, because two lines are in use at once (the 64 x 64 tile's nine slots, 144 KB, measured ahead
// of the ten that fit: 60 x 12192 x 2064 12.4 us against 12.8, 266 x 1308 x 5760 16.2 against 16.6, level at best).  What it comes to (us, before -> now, cold weights):
// 128 x 8192 x 8208 36.7 -> 24.9, where rows on their lines (K = 8320) take 24.2; 47 x 28666 x 10320 83.9 -> 52.9,
// 96 x 4828 x 11984 43.5 -> 23.1, 352 x 9388 x 17200 143 -> 101, 100 x 2374 x 5440 on a stride of 5456 15.6 -> 13.1.  Which
// shapes and tiles: line_config (sg_api.hip).
//
// Tiles timed and not built: 64 x 128, 96 x 128, 32 x 128 and 256 x 64 - without them the best choice is 0.3 % slower in the
// geometric mean of 302 shapes; without any one of the five that are here 1.3 to 2.9 %.
#pragma once

#include "sg_mid_kernel.h"

namespace sg {

// RGW x MH fragments per wave on WN x 2 waves, DEPTH ring slots of both operands
template <int RGW, int MH, int WN, int DEPTH>
__global__ void __launch_bounds__(WN * 128) line_gemm_kernel(const StreamArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring[];   // [DEPTH][BN][128] | [DEPTH][BM][128]
    Stamps stamps;
    stamps.begin();

    constexpr int WAVES = 2 * WN;
    constexpr int BN = 16 * RGW * WN, BM = 32 * MH;
    constexpr int WI = BN / 8 / WAVES, XI = BM / 8 / WAVES, PER_STAGE = WI + XI;   // DMA instructions of a wave and line
    static_assert(BN % (8 * WAVES) == 0 && BM % (8 * WAVES) == 0, "rows split evenly over the waves' DMA instructions");
    static_assert(DEPTH >= 4, "two lines in use, one in flight, one being refilled");
    constexpr int W_BYTES = BN * 128, X_BYTES = BM * 128;
    constexpr int IN_FLIGHT = (DEPTH - 3) * PER_STAGE;
    static_assert(IN_FLIGHT <= 63, "vmcnt");

    const int lane = lane_id();
    const int wave = wave_id();
    const int wn = wave % WN, wm = wave / WN;

    int tile_n, split, tile_m;
    {
        const int per_tile = a.split_k * a.m_tiles;
        int p;
        tile_n = xcd_weight_tile((int)blockIdx.x, (int)gridDim.x, per_tile, a.n_tiles, p);
        split = p / a.m_tiles;
        tile_m = p - split * a.m_tiles;
    }
    const int n0 = tile_n * BN, m0 = tile_m * BM;
    const int blocks_total = (a.k + 127) >> 7;         // K splits take within one block of each other
    const int b_begin = (int)fast_div((unsigned)(blocks_total * split), (unsigned)a.split_k, a.inv_split_k);
    const int n_blk = (int)fast_div((unsigned)(blocks_total * (split + 1)), (unsigned)a.split_k, a.inv_split_k) - b_begin;
    // Blocks are taken from k_rot on and wrapped.  The lines in the order in which they are fetched: k_rot .. n_blk (the line
    // behind the last block's own, which that block needs too), then 0 .. k_rot; block and line v share their slot.
    const int k_rot = (int)((((unsigned)tile_n >> 3) * 5u) % (unsigned)n_blk);
    const int n_lines = n_blk + (k_rot ? 2 : 1);
    auto line_of = [&](int v) __attribute__((always_inline)) { return b_begin + (v + k_rot <= n_blk ? v + k_rot : v + k_rot - n_blk - 1); };

    // ---- DMA: instruction i of this wave covers stage rows 8 * (WAVES * i + wave) .. +7, a line each ----------
    const int d_row = lane >> 3, d_pp = lane & 7;
    const uint8_t* const w_src = a.B + (size_t)n0 * a.b_stride;
    const uint8_t* const x_src = a.A + (size_t)m0 * a.k;
    unsigned wrow[WI], xrow[XI];     // 32-bit: the launcher refuses pitches beyond 8 MB
    int wcol[WI], xcol[XI];          // this lane's column on line 0; negative in front of the row
#pragma unroll
    for (int i = 0; i < WI; i++) {
        const int row_l = 8 * (WAVES * i + wave) + d_row;
        const int row = row_l < a.n - n0 ? row_l : a.n - 1 - n0;
        wrow[i] = (unsigned)row * (unsigned)a.b_stride;
        wcol[i] = ((d_pp ^ ((row_l >> 1) & 7)) << 4) - (int)((unsigned)(reinterpret_cast<uintptr_t>(w_src) + wrow[i]) & 127u);
    }
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int row_l = 8 * (WAVES * i + wave) + d_row;
        const int row = row_l < a.m - m0 ? row_l : a.m - 1 - m0;
        xrow[i] = (unsigned)row * (unsigned)a.k;
        xcol[i] = ((d_pp ^ ((row_l >> 1) & 7)) << 4) - (int)((unsigned)(reinterpret_cast<uintptr_t>(x_src) + xrow[i]) & 127u);
    }
    const int last_piece = a.k - 16;
    const unsigned ring_lds = lds_addr(ring) + (unsigned)wave * 1024;
    auto column = [&](int col0, int line) __attribute__((always_inline)) {
        const int c = col0 + (line << 7);
        return (unsigned)(c < 0 ? 0 : (c > last_piece ? last_piece : c));
    };
    auto issue_one = [&](int i, int line, int slot) __attribute__((always_inline)) {
        if (i < XI)
            dma_1kb_at(x_src, xrow[i] + column(xcol[i], line), ring_lds + DEPTH * W_BYTES + (unsigned)slot * X_BYTES + WAVES * i * 1024);
        else
            dma_1kb_stream_at(w_src, wrow[i - XI] + column(wcol[i - XI], line), ring_lds + (unsigned)slot * W_BYTES + WAVES * (i - XI) * 1024);
    };

    // ---- LDS reads: lane (r, g) wants pieces g and g + 4 of a block, at g + shift and g + 4 + shift of row r's stream -------
    const int r = lane & 15, g = lane >> 4, swizzle = (r >> 1) & 7;
    const int w_shift = (int)((reinterpret_cast<uintptr_t>(w_src) + (unsigned)r * (unsigned)a.b_stride) & 127u) >> 4;
    const int x_shift = (int)((reinterpret_cast<uintptr_t>(x_src) + (unsigned)r * (unsigned)a.k) & 127u) >> 4;
    auto place = [&](int piece, bool& next) __attribute__((always_inline)) {
        next = piece >= 8;
        return r * 128 + (((piece & 7) ^ swizzle) << 4);
    };
    bool w_next[2], x_next[2];       // on the line behind the block's own
    int w_at[2], x_at[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        w_at[h] = wn * RGW * 16 * 128 + place(g + 4 * h + w_shift, w_next[h]);
        x_at[h] = DEPTH * W_BYTES + wm * MH * 16 * 128 + place(g + 4 * h + x_shift, x_next[h]);
    }
    const int new_pieces = (a.k - ((blocks_total - 1) << 7)) >> 4;   // of K's last block

    f32x4 acc[RGW][MH];
#pragma unroll
    for (int rg = 0; rg < RGW; rg++)
#pragma unroll
        for (int mb = 0; mb < MH; mb++) acc[rg][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ---- prologue: lines 0 .. DEPTH-2 ------------------------------------------------------------------------
#pragma unroll
    for (int v = 0; v < DEPTH - 1; v++)
        if (v < n_lines) {
#pragma unroll
            for (int i = 0; i < PER_STAGE; i++) issue_one(i, line_of(v), v);
        }
    stamps.mark(1);

    int slot = 0;
    for (int v = 0; v + 1 < n_lines; v++) {
        // lines v and v + 1 have landed - behind v + 1, v + 2 .. v + DEPTH - 2 have been issued - and v - 1 is consumed
        if (v + DEPTH - 1 <= n_lines) wait_vmcnt<IN_FLIGHT>();
        else wait_vmcnt_upto((n_lines - v - 2) * PER_STAGE);
        __syncthreads();
        if (v == 0) stamps.mark(2);
        __builtin_amdgcn_sched_barrier(0);
        const int next_slot = slot + 1 == DEPTH ? 0 : slot + 1, prev_slot = slot == 0 ? DEPTH - 1 : slot - 1;
        if (v + DEPTH - 1 < n_lines) {
            const int line = line_of(v + DEPTH - 1);
#pragma unroll
            for (int i = 0; i < PER_STAGE; i++) issue_one(i, line, prev_slot);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (v + k_rot != n_blk) {        // (line n_blk has no block of its own)
            const uint8_t* wp[2];
            const uint8_t* xp[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                wp[h] = ring + (w_next[h] ? next_slot : slot) * W_BYTES + w_at[h];
                xp[h] = ring + (x_next[h] ? next_slot : slot) * X_BYTES + x_at[h];
            }
            i32x8 x[MH];
#pragma unroll
            for (int mb = 0; mb < MH; mb++) {
                const i32x4 lo = *reinterpret_cast<const i32x4*>(xp[0] + mb * 2048);
                const i32x4 hi = *reinterpret_cast<const i32x4*>(xp[1] + mb * 2048);
                x[mb] = i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            }
            if (new_pieces < 8 && line_of(v) == blocks_total - 1) {
                const bool zero_lo = g >= new_pieces, zero_hi = g + 4 >= new_pieces;
#pragma unroll
                for (int mb = 0; mb < MH; mb++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        if (zero_lo) x[mb][e] = 0;
                        if (zero_hi) x[mb][4 + e] = 0;
                    }
            }
#pragma unroll
            for (int rg = 0; rg < RGW; rg++) {
                const i32x4 lo = *reinterpret_cast<const i32x4*>(wp[0] + rg * 2048);
                const i32x4 hi = *reinterpret_cast<const i32x4*>(wp[1] + rg * 2048);
                const i32x8 w = i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                for (int mb = 0; mb < MH; mb++) acc[rg][mb] = mfma_e4m3_16x16x128(w, x[mb], acc[rg][mb]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        slot = next_slot;
    }
    stamps.mark(3);

    if (a.split_k == 1) {
        store_wave_tile<RGW, MH>(a, [&](int rg, int mb) { return acc[rg][mb]; }, m0 + wm * MH * 16 + r, n0 + wn * RGW * 16 + 4 * g);
    } else {
        store_wave_partials<RGW, MH, WAVES>(a, acc, tile_m * a.n_tiles + tile_n, split, wave, lane);
    }
    stamps.end(a);
}

}  // namespace sg
