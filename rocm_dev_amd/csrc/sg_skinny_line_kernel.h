// FP8 skinny GEMM (up to 32 activation rows) for rows that start off their 128-byte lines:
//     D[m,n] = scale * sum_k A[m,k] * B[n,k].
//
// The LDS ring of sg_lds_kernel.h asks for 256 bytes of K of every weight row at a time.  Where the rows' pitch is no
// multiple of 128 such a piece lies on three lines instead of two, all three are asked for, and the next stage asks for the
// third again: the L1 sees half as many requests more, and it is what a weight stream is bound by.  Counted (requests of the L1 to
// the L2, thousands, ring -> these kernels; time of the launch by itself): 32 x 32768 x 4112 2292 -> 1373, 31.2 -> 27.3 us; 13 x
// 20660 x 9664 on rows of 9680 2812 -> 1845, 54 -> 36; 8 x 8192 x 16448 1595 -> 1349, 34 -> 25.
//
// So, as in sg_line_kernel.h, the stages here follow the lines row by row: pair j of a row are the 256 bytes from 256 * j on,
// counted from the start of the line that its first byte lies on.  A row that starts `shift` 16-byte pieces into its line
// holds piece p of K block b (256 bytes) at piece p + shift of its stream, in pair b or b + 1; the shift is applied where the
// operand is read from LDS.  Pitches are multiples of 16 bytes, so 16 rows on is a multiple of 256 bytes on and a lane has
// one shift per operand.  In the ring's layout the lanes (r, g) of one pass then read piece (g + shift) % 4 of 64-byte run
// (g + shift) / 4, and the shifts of rows 4 apart differ by a multiple of 4: the sixteen lanes still hit sixteen bank groups.
//
// Nothing outside a row, or outside a wave's share of K, is read: a piece before or behind it is replaced by the share's
// first or last piece.  The former are never used; the latter meet zeroed activations, and a NaN among them is one that the
// share's last block holds as well.
#pragma once

#include "sg_lds_kernel.h"

namespace sg {

// An operand's rows of one tile as pairs of lines: the addresses of its DMA instructions (4 rows x 256 bytes each) and the
// places in LDS of the pieces that a lane feeds to the matrix instructions.
template <int INSTR>
struct LineRows {
    unsigned row[INSTR];                 // 32-bit offsets: the host keeps 64 rows below 2 GB
    int col[INSTR < 4 ? INSTR : 4];      // this lane's column in pair 0; negative in front of the row
    int at;                              // LDS offset of the lane's piece of chunk 0 in its pair's slot
    int run;                             // 64-byte runs that the shift adds: 0, 1 or 2

    // `src`: the tile's first row at the start of the share of K; rows past `last` re-read it and are never stored
    __device__ __forceinline__ void init(const uint8_t* src, int pitch, int last, int lane) {
        const int q = lane >> 2, p = lane & 3, r = lane & 15, g = lane >> 4;
#pragma unroll
        for (int u = 0; u < INSTR; u++) {
            const int row_l = 4 * u + (q & 3);
            row[u] = (unsigned)(row_l < last ? row_l : last) * (unsigned)pitch;
            if (u < 4)
                col[u] = (q >> 2) * 64 + ((p + u) & 3) * 16 - (int)((unsigned)(reinterpret_cast<uintptr_t>(src) + (unsigned)row_l * (unsigned)pitch) & 127u);
        }
        const int piece = g + ((int)((unsigned)(reinterpret_cast<uintptr_t>(src) + (unsigned)r * (unsigned)pitch) & 127u) >> 4);
        run = piece >> 2;
        at = 1024 * (r >> 2) + 64 * (r & 3) + 16 * (((piece & 3) - (r >> 2)) & 3) + 256 * run;
    }
    __device__ __forceinline__ unsigned offset(int u, int pair, int last_piece) const {
        const int c = col[u & 3] + (pair << 8);
        return row[u] + (unsigned)(c < 0 ? 0 : (c > last_piece ? last_piece : c));
    }
    // where chunk i (64 bytes) of a K block is, given the slots of its pair and of the one behind
    __device__ __forceinline__ const uint8_t* chunk(const uint8_t* slot, const uint8_t* next, int i) const {
        return (i + run >= 4 ? next - 1024 : slot) + at + 256 * i;
    }
};

__device__ __forceinline__ i32x8 join_pieces(const uint8_t* lo, const uint8_t* hi) {
    const i32x4 a = *reinterpret_cast<const i32x4*>(lo), b = *reinterpret_cast<const i32x4*>(hi);
    return i32x8{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
}
// zeroes what lies behind K in the last block, which has `pieces` 16-byte pieces: lane (r, g) holds piece 4 * i + g of chunk i
template <int MT>
__device__ __forceinline__ void zero_behind(i32x8 (&x)[MT][2], int pieces, int g) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const bool lo = 8 * h + g >= pieces, hi = 8 * h + 4 + g >= pieces;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (lo) x[mt][h][e] = 0;
                if (hi) x[mt][h][4 + e] = 0;
            }
    }
}

// The last DEPTH pairs of a stream: all are issued; step(i) needs pair i + 1 as well.
template <int D, int DEPTH, int PER_STAGE, class Step>
__device__ __forceinline__ void drain_pairs(Step& step, int i) {
    constexpr int BEHIND = DEPTH - 2 - D > 0 ? DEPTH - 2 - D : 0;
    wait_vmcnt<BEHIND * PER_STAGE>();
    step(i + D);
    if constexpr (D + 1 < DEPTH) drain_pairs<D + 1, DEPTH, PER_STAGE>(step, i);
}

// One workgroup per 16 * RG row tile and K split; its waves share the K range in contiguous parts and meet in LDS.
template <int MT, int RG, int XU, int DEPTH>
__global__ void __launch_bounds__(512) skinny_line_kernel(const StreamArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring[];  // [wave][DEPTH][weights RG*4 KB | activations XU KB]
    __shared__ unsigned arrival;
    __shared__ __attribute__((aligned(16))) float factor_lds[kStagedFactors];

    constexpr int PER_STAGE = RG * 4 + XU;
    constexpr int STAGE_BYTES = PER_STAGE * 1024;
    static_assert(DEPTH >= 3 && (DEPTH - 2) * PER_STAGE <= 63, "ring");
    static_assert(XU <= 4 * MT, "more activation rows than the tile has");

    Stamps stamps;
    stamps.begin();
    const int lane = lane_id();
    const int wave = wave_id();
    const int g = lane >> 4;

    int tile_n, split, tile_m;
    decode_tile(a, xcd_order((int)blockIdx.x, (int)gridDim.x), tile_n, split, tile_m);
    const int n0 = tile_n * (16 * RG);
    const int m0 = tile_m * (16 * MT);

    int b_begin, b_end;
    const int blocks_total = (a.k + 255) >> 8;
    split_range(a, blocks_total, split, b_begin, b_end);
    const int first = b_begin + (int)fast_div((unsigned)((b_end - b_begin) * wave), (unsigned)a.waves, a.inv_waves);
    const int end = b_begin + (int)fast_div((unsigned)((b_end - b_begin) * (wave + 1)), (unsigned)a.waves, a.inv_waves);
    const int blocks = end - first;
    const int share = (end < blocks_total ? end << 8 : a.k) - (first << 8);     // columns
    const int pairs = blocks > 0 ? (share + 112 + 255) >> 8 : 0;                // the last block may need one more
    const int tail_i = end == blocks_total ? blocks - 1 : -1;
    const int tail_pieces = (a.k - ((blocks_total - 1) << 8)) >> 4;

    const uint8_t* const w_src = a.B + (size_t)n0 * a.b_stride + ((size_t)first << 8);
    const uint8_t* const x_src = a.A + (size_t)m0 * a.k + ((size_t)first << 8);
    LineRows<RG * 4> w;
    LineRows<XU> x;
    w.init(w_src, a.b_stride, a.n - 1 - n0, lane);
    x.init(x_src, a.k, a.m - 1 - m0, lane);
    const uint8_t* const my_ring = ring + (size_t)wave * (DEPTH * STAGE_BYTES);
    const unsigned my_ring_lds = lds_addr(my_ring);

    auto issue = [&](int j) __attribute__((always_inline)) {
        const unsigned slot = my_ring_lds + (unsigned)(j % DEPTH) * STAGE_BYTES;
#pragma unroll
        for (int u = 0; u < RG * 4; u++) dma_1kb_stream_at(w_src, w.offset(u, j, share - 16), slot + u * 1024);
#pragma unroll
        for (int u = 0; u < XU; u++) dma_1kb_at(x_src, x.offset(u, j, share - 16), slot + (RG * 4 + u) * 1024);
    };

    f32x4 acc[RG][MT];
#pragma unroll
    for (int rg = 0; rg < RG; rg++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[rg][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto consume = [&](int i) __attribute__((always_inline)) {
        if (i >= blocks) return;
        const uint8_t* slot = my_ring + (size_t)(i % DEPTH) * STAGE_BYTES;
        // (with no pair behind, the lanes that would read it hold pieces behind K: anything of the row will do)
        const uint8_t* next = i + 1 < pairs ? my_ring + (size_t)((i + 1) % DEPTH) * STAGE_BYTES : slot;
        i32x8 xv[MT][2];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                xv[mt][h] = join_pieces(x.chunk(slot, next, 2 * h) + RG * 4096 + mt * 4096, x.chunk(slot, next, 2 * h + 1) + RG * 4096 + mt * 4096);
        if (i == tail_i) zero_behind<MT>(xv, tail_pieces, g);
#pragma unroll
        for (int rg = 0; rg < RG; rg++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const i32x8 wv = join_pieces(w.chunk(slot, next, 2 * h) + rg * 4096, w.chunk(slot, next, 2 * h + 1) + rg * 4096);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[rg][mt] = mfma_e4m3_16x16x128(wv, xv[mt][h], acc[rg][mt]);
            }
    };

    // the factors behind the first pair, older than every other one
    const StagedFactors factors{factor_lds};
    const float scale = scalar_scale(a);
    if (pairs >= DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            issue(d);
            if (d == 0 && wave == 0) factors.fetch(a, m0, n0, lane);
        }
        stamps.mark(1);
        asm volatile("" ::"s"(scale));   // (here, not where the outputs are ready)
        int i = 0;
        for (; i + DEPTH < pairs; i++) {
            wait_vmcnt<(DEPTH - 2) * PER_STAGE>();   // pairs i and i + 1 have landed
            if (i == 0) stamps.mark(2);
            consume(i);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            issue(i + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
        }
        drain_pairs<0, DEPTH, PER_STAGE>(consume, i);
    } else {
        for (int j = 0; j < pairs; j++) issue(j);
        if (wave == 0) factors.fetch(a, m0, n0, lane);
        stamps.mark(1);
        asm volatile("" ::"s"(scale));
        wait_vmcnt<0>();
        stamps.mark(2);
        for (int i = 0; i < blocks; i++) consume(i);
    }

    // the ring is reused for the cross-wave reduction: every wave must be done reading it
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    stamps.mark(3);
    __syncthreads();
    finish_tile<RG, MT>(a, acc, reinterpret_cast<f32x4*>(ring), &arrival, scale, factors, tile_m, tile_n, split, m0, n0);
    stamps.end(a);
}

// Many tiles: one workgroup per CU with the whole activation matrix in LDS (by K blocks, as in lds_gemm_wavetile_kernel);
// every wave owns whole 16-row tiles over all of K, its ring of weight pairs running across tile boundaries.  No rotation of
// the K start: rows off their lines do not meet in one memory channel - but for some pitches next to a power of two, which
// skinny_line_config (sg_api.hip) leaves to the ring.
template <int MT, int XU, int DEPTH>
__global__ void __launch_bounds__(512) skinny_line_resident_kernel(const StreamArgs a) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t ring[];  // X[blocks][XU KB] | [wave][DEPTH][4 KB]
    constexpr int PER_STAGE = 4, STAGE_BYTES = 4096;
    static_assert(DEPTH >= 3 && XU <= 4 * MT, "ring");

    Stamps stamps;
    stamps.begin();
    const int lane = lane_id();
    const int wave = wave_id();
    const int waves = a.waves;
    const int r = lane & 15, g = lane >> 4;
    const int blocks = (a.k + 255) >> 8;
    const int pairs = (a.k + 112 + 255) >> 8;
    const int tail_pieces = (a.k - ((blocks - 1) << 8)) >> 4;
    // tiles are dealt to workgroups first, so that a few tiles per CU still put a stream on every CU
    const int first = (int)blockIdx.x + (int)gridDim.x * wave, tile_step = (int)gridDim.x * waves;
    const int my_tiles = first < a.n_tiles ? (a.n_tiles - first + tile_step - 1) / tile_step : 0;
    const int total = my_tiles * pairs;

    const int q = lane >> 2, p = lane & 3;
    const int rd_off = 1024 * (r >> 2) + 64 * (r & 3) + 16 * ((g - (r >> 2)) & 3);
    const uint8_t* const my_ring = ring + (size_t)blocks * XU * 1024 + (size_t)wave * (DEPTH * STAGE_BYTES);
    const unsigned my_ring_lds = lds_addr(my_ring), x_lds = lds_addr(ring);

    // ---- resident activations: K block kb is fetched by wave kb % waves --------------------------------------
    int x_issued = 0;
    for (int kb = wave; kb < blocks; kb += waves) {
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int row_l = 4 * u + (q & 3), row = row_l < a.m ? row_l : a.m - 1;
            int c = (kb << 8) + (q >> 2) * 64 + ((p + (u & 3)) & 3) * 16;
            c = c < a.k ? c : a.k - 16;
            dma_1kb(a.A + (size_t)row * a.k + c, x_lds + (unsigned)(kb * XU + u) * 1024);
        }
        x_issued += XU;
    }

    // tiles are 16 rows apart, a multiple of 256 bytes: the shifts are the same in every one
    LineRows<4> w;
    w.init(a.B, a.b_stride, 15, lane);
    int iss_tile = first, iss_pair = 0;
    auto issue = [&](int i) __attribute__((always_inline)) {     // called for i = 0, 1, 2, ... in order
        const int n0 = iss_tile * 16;
        const uint8_t* const src = a.B + (size_t)n0 * a.b_stride;
        const unsigned slot = my_ring_lds + (unsigned)(i % DEPTH) * STAGE_BYTES;
        const unsigned last = (unsigned)(a.n - 1 - n0 < 15 ? a.n - 1 - n0 : 15) * (unsigned)a.b_stride;   // rows past the edge re-read the last one
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int c = w.col[u] + (iss_pair << 8), last_piece = a.k - 16;
            const unsigned row = w.row[u] < last ? w.row[u] : last;
            dma_1kb_stream_at(src, row + (unsigned)(c < 0 ? 0 : (c > last_piece ? last_piece : c)), slot + u * 1024);
        }
        if (++iss_pair == pairs) {
            iss_pair = 0;
            iss_tile += tile_step;
        }
    };

    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float scale = scalar_scale(a);
    int tile = first, pair = 0;
    auto step = [&](int i) __attribute__((always_inline)) {
        if (pair < blocks) {
            const uint8_t* slot = my_ring + (size_t)(i % DEPTH) * STAGE_BYTES;
            const uint8_t* next = pair + 1 < pairs ? my_ring + (size_t)((i + 1) % DEPTH) * STAGE_BYTES : slot;
            const uint8_t* xs = ring + (size_t)pair * (XU * 1024) + rd_off;
            i32x8 xv[MT][2];
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int h = 0; h < 2; h++) xv[mt][h] = join_pieces(xs + mt * 4096 + 512 * h, xs + mt * 4096 + 512 * h + 256);
            if (pair == blocks - 1) zero_behind<MT>(xv, tail_pieces, g);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const i32x8 wv = join_pieces(w.chunk(slot, next, 2 * h), w.chunk(slot, next, 2 * h + 1));
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[mt] = mfma_e4m3_16x16x128(wv, xv[mt][h], acc[mt]);
            }
        }
    };
    auto close = [&]() __attribute__((always_inline)) {
        if (++pair == pairs) {      // the tile is complete: scale, round, store, start the next one
            pair = 0;
            // The result of a matrix instruction may be read 12 wait states behind it.  The compiler did not see that across
            // the branches between the two (the store read the accumulators 3 states behind the last instruction, and took
            // them without it).  Tied to every accumulator, so that none of their last instructions sinks behind it.
            static_assert(MT <= 2);
            if constexpr (MT == 2) asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[1]));
            else asm volatile("s_nop 15" : "+v"(acc[0]));
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                store_fragment(a, acc[mt], scale, mt * 16 + r, tile * 16 + 4 * g);
                acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            tile += tile_step;
        }
    };

    // the first weights behind the activations, so that HBM is busy while those arrive from L2; once at most the prologue's DMAs
    // are outstanding this wave's share of the activations has landed, and the barrier publishes everyone's
    const int pro = total < DEPTH ? total : DEPTH;
    for (int d = 0; d < pro; d++) issue(d);
    stamps.mark(1);
    if (x_issued > 0) wait_vmcnt_upto(pro * PER_STAGE);
    __syncthreads();
    stamps.mark(2);
    if (total >= DEPTH) {
        int i = 0;
        for (; i + DEPTH < total; i++) {
            wait_vmcnt<(DEPTH - 2) * PER_STAGE>();
            step(i);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            issue(i + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
            close();
        }
        auto step_and_close = [&](int ii) __attribute__((always_inline)) {
            step(ii);
            close();
        };
        drain_pairs<0, DEPTH, PER_STAGE>(step_and_close, i);
    } else {
        wait_vmcnt<0>();
        for (int i = 0; i < total; i++) {
            step(i);
            close();
        }
    }
    stamps.mark(3);
    stamps.end(a);
}

}  // namespace sg
