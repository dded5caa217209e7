// FP8 GEMM on wide tiles for gfx950 (a prefill chunk): D[m,n] = scale * sum_k A[m,k] * B[n,k].
//
// What bounds it is the matrix cores (2 * 1024 flops per weight byte at 1024 rows), and next to them the LDS: every
// operand byte is written to it once and read by each wave that needs it, at 128 bytes a clock.  So the workgroup is
// four waves, one per SIMD, in a 2 x 2 grid that own RGW x MH fragments of 16 x 16 each: a stage of 256 x 256 outputs
// and 128 bytes of K is 2048 clocks of MFMA and 1536 of LDS traffic; on eight waves it is 2048 of LDS traffic too (2970
// clocks a stage measured).  Both operands of a K block are staged in LDS by direct-to-LDS loads (the layout, swizzle
// and the window of a partial last block are the mid-batch kernel's, sg_mid_kernel.h).
//
// With one wave per SIMD whatever that wave waits for is idle time of its matrix core, so nothing is read in front of
// its use and no burst of memory instructions stands between two MFMAs:
//   * the wave's activation fragments of a stage are held in registers, two sets; the weight fragments stream through a
//     ring of WR, read AHEAD groups (of MH MFMAs) ahead of their use: WR is RGW, 4 on the 8 x 8 tile, whose registers that
//     leaves, and AHEAD one less, five at most;
//   * the barrier between two stages stands AHEAD groups before the end of a stage, where the last LDS read of the stage
//     has been issued; behind it the remaining groups read the next stage's first operands;
//   * LDS reads and refills are dealt out one by one to the MFMAs they are issued in front of.
// 1024 x 57344 x 8192 on 224 x 256 tiles, four full rounds: 2310 clocks a stage, 1792 of them MFMA, at 1.92 GHz, the clock
// that power leaves (profiles/wide_tile_gemm_time_stamps_and_counters.md; the mid-batch kernel 3230), 469 -> 366 us;
// 1024 x 10240 x 8192 on 160 x 256 tiles 106 -> 73.  Tried and not kept: eight waves (410 us on the first), loads masked by
// EXEC instead of skipped by a branch (100 clocks a stage more).
//
// All workgroups of one XCD walk K in step (the start of the walk depends on the XCD only), so that one XCD's L2
// serves an activation line to all of them while it is there; the mid-batch kernel's rotation by weight tile spreads
// 32 workgroups over most of an activation matrix that is larger than the L2.
#pragma once

#include <type_traits>

#include "sg_mid_kernel.h"

namespace sg {

// Op `d` of `ops` dealt evenly to `slots` slots goes to slot spread(d): the list of ops of a slot is the range
// [first op whose slot is q, ...).
constexpr int wide_first_op(int q, int slots, int ops) { return (q * ops + slots - 1) / slots; }

// A direct-to-LDS load that is issued where `on` (wave-uniform) is positive, without a basic block of its own: a stage
// stays one block.
template <bool STREAM>
__device__ __forceinline__ void dma_1kb_if(const void* sbase, unsigned voff, unsigned lds_base, int on) {
    lds_base = __builtin_amdgcn_readfirstlane(lds_base);
    if constexpr (STREAM)
        asm volatile("s_mov_b32 m0, %2\n\ts_cmp_gt_i32 %3, 0\n\ts_cbranch_scc0 .Lwide%=\n\tglobal_load_lds_dwordx4 %0, %1 nt\n.Lwide%=:"
                     ::"v"(voff), "s"(sbase), "s"(lds_base), "s"(on) : "memory", "m0", "scc");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_cmp_gt_i32 %3, 0\n\ts_cbranch_scc0 .Lwide%=\n\tglobal_load_lds_dwordx4 %0, %1\n.Lwide%=:"
                     ::"v"(voff), "s"(sbase), "s"(lds_base), "s"(on) : "memory", "m0", "scc");
}
// vmcnt(N) where `on` is positive, vmcnt(0) otherwise, likewise
template <int N>
__device__ __forceinline__ void wait_vmcnt_if(int on) {
    asm volatile("s_cmp_gt_i32 %0, 0\n\ts_cbranch_scc1 .Lwide%=\n\ts_waitcnt vmcnt(0)\n.Lwide%=:\n\ts_waitcnt vmcnt(%1)"
                 ::"s"(on), "n"(N) : "memory", "scc");
}
// The matrix instruction as text, accumulators in the accumulation registers: up to 256 of them beside 200 of
// everything else, which the builtin (free to take either file) turns into 300 moves a stage.  Volatile, so it stays where
// it is written among the memory instructions.  The two idle states in front of it are what a vector instruction that
// wrote an operand would need.
//
// The compiler does not know how long the result takes and may read, copy or spill an accumulator right behind the text.
// So the instruction that ends a stage is followed, in its own text, by the 32 idle states the longest one needs, where
// `left` (wave-uniform) is not positive: behind the last stage every accumulator is complete before anything else can be
// issued.  (Inside the loop nothing but the next stage's instruction touches one: tests/test_wide_codegen.py.)
__device__ __forceinline__ void mfma_acc(f32x4& c, const i32x8& a, const i32x8& b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b) : "memory");
}
__device__ __forceinline__ void mfma_acc_drain(f32x4& c, const i32x8& a, const i32x8& b, int left) {
    asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0\n\ts_cmp_gt_i32 %3, 0\n\ts_cbranch_scc1 .Lwide%=\n\t"
                 "s_nop 15\n\ts_nop 15\n.Lwide%=:"
                 : "+a"(c) : "v"(a), "v"(b), "s"(left) : "memory", "scc");
}
// Holds the copy of an accumulator to vector registers back to where the epilogue uses it.  On the largest tile the compiler
// otherwise copies all 256 at the epilogue's top and spills what does not fit (21 registers; the smaller tiles fit).
__device__ __forceinline__ void keep_in_accumulator(f32x4& c) { asm volatile("" : "+a"(c)); }

// RGW x MH fragments per wave on WN x 2 waves; DW, DX: ring slots of the weights and of the activations (2 <= DX <= DW)
template <int RGW, int MH, int WN, int DW, int DX, bool TAIL>
__global__ void __launch_bounds__(WN * 128) wide_gemm_kernel(const StreamArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring[];   // [DW][BN][128] | [DX][BM][128]
    Stamps stamps;
    stamps.begin();

    constexpr int WM = 2, WAVES = WN * WM;
    constexpr int BN = 16 * RGW * WN, BM = 16 * MH * WM;
    constexpr int NW = BN / 8, NX = BM / 8;                 // 1 KB DMA instructions of a stage
    constexpr int WI = NW / WAVES, XI = NX / WAVES;         // ... and of a wave
    static_assert(NW % WAVES == 0 && NX % WAVES == 0 && RGW >= 4 && MH >= 4, "tile");
    static_assert(DX >= 2 && DX <= DW && DW - 2 <= DX, "rings");
    constexpr int W_BYTES = BN * 128, X_BYTES = BM * 128;
    // weight fragments are read AHEAD groups early, into a ring of WR
    constexpr int WR = RGW * MH > 56 ? 4 : RGW, AHEAD = WR > 6 ? 5 : WR - 1;
    static_assert(AHEAD < WR && 2 * RGW % WR == 0, "the loop's two stages leave both register rings in phase");
    constexpr int LATE = RGW - AHEAD;                       // first group behind the barrier

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
    int b_begin, b_end;
    const int blocks_total = (a.k + 127) >> 7;
    split_range(a, blocks_total, split, b_begin, b_end);
    const int n_blk = b_end - b_begin;
    const int old_pieces = TAIL ? (128 - (a.k & 127)) >> 4 : 0;
    const int k_rot = (int)(((unsigned)(tile_n & 7) * (unsigned)n_blk) >> 3);
    auto k_block = [&](int s) __attribute__((always_inline)) {
        const int b = s + k_rot;
        return b_begin + (b >= n_blk ? b - n_blk : b);
    };

    // ---- DMA: instruction i of this wave covers stage rows 8 * (WAVES * i + wave) .. +7 --------------------
    const int d_row = lane >> 3, d_pp = lane & 7;
    unsigned woff[WI], xoff[XI];                            // 32-bit: the launcher refuses pitches beyond 8 MB
#pragma unroll
    for (int i = 0; i < WI; i++) {
        const int row_l = 8 * (WAVES * i + wave) + d_row;
        const int row = row_l < a.n - n0 ? row_l : a.n - 1 - n0;
        woff[i] = (unsigned)row * (unsigned)a.b_stride + ((d_pp ^ ((row_l >> 1) & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int row_l = 8 * (WAVES * i + wave) + d_row;
        const int row = row_l < a.m - m0 ? row_l : a.m - 1 - m0;
        xoff[i] = (unsigned)row * (unsigned)a.k + ((d_pp ^ ((row_l >> 1) & 7)) << 4);
    }
    const uint8_t* const w_src = a.B + (size_t)n0 * a.b_stride;
    const uint8_t* const x_src = a.A + (size_t)m0 * a.k;
    const unsigned ring_lds = lds_addr(ring) + (unsigned)wave * 1024;
    auto k_offset = [&](int s) __attribute__((always_inline)) {
        const int kb = k_block(s);
        return ((size_t)kb << 7) - ((TAIL && kb == blocks_total - 1) ? (size_t)(old_pieces << 4) : 0);
    };
    auto issue_x = [&](int i, size_t koff, int slot, int on = 1) __attribute__((always_inline)) {
        dma_1kb_if<false>(x_src + koff, xoff[i], ring_lds + DW * W_BYTES + (unsigned)slot * X_BYTES + WAVES * i * 1024, on);
    };
    auto issue_w = [&](int i, size_t koff, int slot, int on = 1) __attribute__((always_inline)) {
        dma_1kb_if<true>(w_src + koff, woff[i], ring_lds + (unsigned)slot * W_BYTES + WAVES * i * 1024, on);
    };

    // ---- LDS reads: lane (r, g) reads pieces g and g + 4 of row r of a fragment -----------------------------
    const int r = lane & 15, g = lane >> 4;
    const int rd0 = r * 128 + ((g ^ ((r >> 1) & 7)) << 4);
    const int flip = ((rd0 & 64) ? -64 : 64);               // from piece g to piece g + 4 of the swizzled row
    const uint8_t* const w_lds = ring + (wn * RGW * 16) * 128 + rd0;
    const uint8_t* const x_lds = ring + DW * W_BYTES + (wm * MH * 16) * 128 + rd0;
    auto read_half = [&](i32x8& f, const uint8_t* p, int half) __attribute__((always_inline)) {
        const i32x4 v = *reinterpret_cast<const i32x4*>(half ? p + flip : p);
#pragma unroll
        for (int e = 0; e < 4; e++) f[half * 4 + e] = v[e];
    };

    f32x4 acc[RGW][MH];
#pragma unroll
    for (int rg = 0; rg < RGW; rg++)
#pragma unroll
        for (int mb = 0; mb < MH; mb++) acc[rg][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    i32x8 w[WR], x[2][MH];

    // Refill group j: activations of stage j + DX (issued behind the barrier of stage j), then weights of stage j + DW
    // (in front of the barrier of stage j + 1).  In front of the barrier of stage s the youngest group is s - 1; behind
    // the last instruction of X(s+1) and of W(s+1) the queue then holds this many younger ones:
    constexpr int PER = WI + XI;
    constexpr int IN_FLIGHT = (WI + (DX - 2) * PER) < (DW - 2) * PER ? (WI + (DX - 2) * PER) : (DW - 2) * PER;
    static_assert(IN_FLIGHT <= 63, "vmcnt");

    // ---- prologue: groups -DW .. -1 without the weights of group -1, then stage 0's first operands ----------------
#pragma unroll
    for (int j = -DW; j < 0; j++) {
        if (j + DX >= 0 && j + DX < n_blk) {
#pragma unroll
            for (int i = 0; i < XI; i++) issue_x(i, k_offset(j + DX), j + DX);
        }
        if (j < -1 && j + DW < n_blk) {
#pragma unroll
            for (int i = 0; i < WI; i++) issue_w(i, k_offset(j + DW), j + DW);
        }
    }
    stamps.mark(1);
    if (n_blk < DW) wait_vmcnt<0>();
    else wait_vmcnt<IN_FLIGHT>();
    __syncthreads();
    stamps.mark(2);
#pragma unroll
    for (int i = 0; i < AHEAD; i++) { read_half(w[i], w_lds + i * 2048, 0); read_half(w[i], w_lds + i * 2048, 1); }
#pragma unroll
    for (int mb = 0; mb < MH; mb++) { read_half(x[0][mb], x_lds + mb * 2048, 0); read_half(x[0][mb], x_lds + mb * 2048, 1); }

    int slot_w = 0, slot_x = 0;
    // stage s, the u-th of the unrolled loop's: consumes x[u & 1] and the weight ring from index u * RGW on
    auto stage = [&](int s, auto uc) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        const int next_w = slot_w + 1 == DW ? 0 : slot_w + 1, next_x = slot_x + 1 == DX ? 0 : slot_x + 1;
        const int prev_w = slot_w == 0 ? DW - 1 : slot_w - 1;
        const uint8_t* wcur = w_lds + slot_w * W_BYTES;
        const uint8_t* wnext = w_lds + next_w * W_BYTES;
        const uint8_t* xnext = x_lds + next_x * X_BYTES;
        const int fill_w = n_blk - (s - 1 + DW), fill_x = n_blk - (s + DX);   // positive: there is such a stage
        const size_t koff_w = k_offset(s - 1 + DW), koff_x = k_offset(s + DX);
        if constexpr (TAIL) {
            if (k_block(s) == blocks_total - 1) {     // the last window: its activation pieces below the boundary are zero
                const bool zero_lo = g < old_pieces, zero_hi = g + 4 < old_pieces;
#pragma unroll
                for (int mb = 0; mb < MH; mb++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        if (zero_lo) x[u & 1][mb][e] = 0;
                        if (zero_hi) x[u & 1][mb][4 + e] = 0;
                    }
            }
        }
#pragma unroll
        for (int rg = 0; rg < RGW; rg++) {
            if (rg == LATE) {
                // this wave's reads of stage s have arrived, its loads of stage s + 1 have landed; behind the barrier
                // that holds for all waves.  (Behind the last stage the barrier and the reads - of a slot that holds an
                // older stage, never used - stay unconditional: the compiler then knows how many LDS reads are
                // outstanding in every group.)
                wait_vmcnt_if<IN_FLIGHT>(fill_w);
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int mb = 0; mb < MH; mb++) {
                // weight fragment rg + AHEAD, of this stage or the next, in the first two slots of the group
                if (mb < 2) {
                    const uint8_t* p = rg + AHEAD < RGW ? wcur + (rg + AHEAD) * 2048 : wnext + (rg + AHEAD - RGW) * 2048;
                    read_half(w[(u * RGW + rg + AHEAD) % WR], p, mb);
                }
                // the other slots: behind the barrier the next stage's activation reads and, alternating with the first
                // of them, the activation refill; in front of it the weight refill of the stage before
                const int free_slot = rg < LATE ? rg * (MH - 2) + mb - 2 : (rg - LATE) * (MH - 2) + mb - 2;
                if (mb >= 2 && rg >= LATE) {
                    constexpr int Q = AHEAD * (MH - 2), OPS = 2 * MH + XI;
#pragma unroll
                    for (int op = wide_first_op(free_slot, Q, OPS); op < wide_first_op(free_slot + 1, Q, OPS); op++) {
                        const int read = op < 2 * XI ? op / 2 : op - XI;
                        if (op < 2 * XI && op % 2 == 0) issue_x(op / 2, koff_x, slot_x, fill_x);
                        else read_half(x[(u + 1) & 1][read >> 1], xnext + (read >> 1) * 2048, read & 1);
                    }
                }
                if (mb >= 2 && rg < LATE) {
                    constexpr int Q = LATE * (MH - 2);
#pragma unroll
                    for (int op = wide_first_op(free_slot, Q, WI); op < wide_first_op(free_slot + 1, Q, WI); op++)
                        issue_w(op, koff_w, prev_w, fill_w);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (rg == RGW - 1 && mb == MH - 1) mfma_acc_drain(acc[rg][mb], w[(u * RGW + rg) % WR], x[u & 1][mb], n_blk - 1 - s);
                else mfma_acc(acc[rg][mb], w[(u * RGW + rg) % WR], x[u & 1][mb]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        slot_w = next_w;
        slot_x = next_x;
    };
    int s = 0;
    for (; s + 1 < n_blk; s += 2) {
        stage(s, std::integral_constant<int, 0>{});
        stage(s + 1, std::integral_constant<int, 1>{});
    }
    if (s < n_blk) stage(s, std::integral_constant<int, 0>{});
    stamps.mark(3);

    // ---- epilogue --------------------------------------------------------------------------------
    if (a.split_k > 1) {
        // partials [tile][split][wave][fragment][lane], summed by mid_reduce_kernel
        constexpr int FRAGS_WG = WAVES * RGW * MH;
        const size_t tile_id = (size_t)tile_m * a.n_tiles + tile_n;
        f32x4* mine = reinterpret_cast<f32x4*>(a.ws + (tile_id * a.split_k + split) * (FRAGS_WG * 256) + (size_t)wave * (RGW * MH * 256)) + lane;
#pragma unroll
        for (int rg = 0; rg < RGW; rg++)
#pragma unroll
            for (int mb = 0; mb < MH; mb++) mine[(rg * MH + mb) * 64] = acc[rg][mb];
        stamps.end(a);
        return;
    }
    // The wave turns its tile around in LDS and stores whole runs of 32 * RGW bytes a row (a fragment as it is ends in
    // 32-byte runs: 9.5 us for the stores of a 256 x 256 tile, 7.5 this way).  No barrier: nobody reads the ring any more, and no load
    // is under way (behind the last stages' barriers).
    const float scale = scalar_scale(a);
    constexpr int PITCH = 32 * RGW + 16;                    // bytes; + 16 spreads the rows over the banks
    constexpr int ROWS = 16 * MH;
    uint8_t* const mine = ring + (size_t)wave * (ROWS * PITCH);
    const int m_wave = m0 + wm * ROWS, n_wave = n0 + wn * RGW * 16;
    float rs[MH];
#pragma unroll
    for (int mb = 0; mb < MH; mb++) rs[mb] = row_scale_ahead(a, m_wave + mb * 16 + r);
#pragma unroll
    for (int rg = 0; rg < RGW; rg++) {
        const f32x4 cs = col_scale_ahead(a, n_wave + rg * 16 + 4 * g);
#pragma unroll
        for (int mb = 0; mb < MH; mb++) {
            if (RGW * MH == 64) keep_in_accumulator(acc[rg][mb]);
            f32x4 v = acc[rg][mb];
            // scale, then the row factor, then the column factors: three separately rounded fp32 products
            v *= scale;
            if (a.row_scale) v *= rs[mb];
            if (a.col_scale) v *= cs;
            *reinterpret_cast<u32x2*>(mine + (mb * 16 + r) * PITCH + rg * 32 + 8 * g) =
                u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    uint16_t* const d = reinterpret_cast<uint16_t*>(a.D);
    constexpr int PIECES = 2 * RGW;                         // 16-byte pieces of a row
    // D is 8-byte aligned and n even: a piece starts at a multiple of four bytes, which is all a 16-byte store needs.
    // (With eight 2-byte stores a piece where 8 does not divide n: 1159 x 22756 x 880 78.0 us, now 44.7; 778 x 22364 x 2048
    // 80.1, now 51.8; the mid-batch kernel takes 48.6 and 63.0.)
    using u32x4_at4 = u32x4 __attribute__((aligned(4)));
    auto store_rows = [&](auto ragged) __attribute__((always_inline)) {
#pragma unroll 4
        for (int i = lane; i < ROWS * PIECES; i += 64) {
            const int row = i / PIECES, c = i - row * PIECES;
            const int m_idx = m_wave + row, n_idx = n_wave + 8 * c;
            if (m_idx >= a.m || n_idx >= a.n) continue;
            uint16_t* const to = d + (size_t)m_idx * a.n + n_idx;
            const u32x4 v = *reinterpret_cast<const u32x4*>(mine + row * PITCH + 16 * c);
            if (!decltype(ragged)::value || n_idx + 8 <= a.n) {
                *reinterpret_cast<u32x4_at4*>(to) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 3; e++)
                    if (n_idx + 2 * e < a.n) reinterpret_cast<uint32_t*>(to)[e] = v[e];
            }
        }
    };
    if ((a.n & 7) == 0) store_rows(std::false_type{});   // no piece crosses n
    else store_rows(std::true_type{});
    stamps.end(a);
}

}  // namespace sg
