// Per-row FP8 codec for gfx950: the local compute on either side of an FP8 all-reduce
// exchange.  All three kernels are pure HBM streaming; arithmetic per element is kept to a
// handful of VALU operations so the memory pipe stays the limit.
//
//   encode  scales[r] = absmax(X[r,:]) / 448 (1 for an all-zero row);
//           Q[r,c]    = e4m3_rne_sat( fp32(X[r,c]) / scales[r] )          (bit exact)
//   decode  Y[r,c]    = bf16( dec(Q[r,c]) * scales[r] )
//   reduce  Y[r,c]    = bf16( sum_i dec(Q_i[r,c]) * scales_i[r] ), fp32, buffer order,
//           multiply and add rounded separately (no fused multiply-add)
//
// The quotient x / s must be the correctly rounded fp32 quotient, because the E4M3
// rounding that follows makes a one-ulp slip visible at a tie.  A hardware IEEE divide is
// about ten VALU operations per element, too many for a streaming kernel, so the kernel
// divides once per row (y = 1/s, correctly rounded) and per element uses Markstein's
// correction  q = x*y;  r = fma(-s, q, x);  q' = fma(r, y, q).  x and the row maximum are
// bf16 values; for every bf16 maximum with biased exponent 60..190 and every bf16 x below
// it this sequence has been checked exhaustively on the CPU against the IEEE quotient
// wherever |q| >= 2^-12 (smaller quotients all encode to zero).  Rows whose maximum lies
// outside that exponent window take the plain IEEE divide.
#include "sg_device.h"
#include "sg_host.h"
#include "sg_quant.h"

namespace sg {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t cvt_bf16x2(float lo, float hi) {
    f32x2 v = {lo, hi};
    bf16x2_t h = __builtin_convertvector(v, bf16x2_t);
    return __builtin_bit_cast(uint32_t, h);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// A row is held in registers, so it is read from memory exactly once: thread t of the THREADS that share a row holds
// its chunks t, t + THREADS, ... of 8 bf16 each, CH of them.  HBM-bound at 3 bytes per element (30.5 us for 8192 x 8192 at
// the 6.6 TB/s a stream reaches, measured 34.4); what a row shape can lose on top is idle lanes, workgroup launches and
// the reduction of the maximum, which is why there is one build per range of row lengths (launch_fp8_encode_rows).
//
// All chunks are asked for before any is looked at.  A thread beyond the row's end takes its last chunk again, which changes
// no maximum, and stores nothing: a load that only some lanes issue, into registers that are zero in the others, made the
// compiler wait for the second load before it issued the third (2048 x 4112 8.3 us, 7.2 this way).
template <int STEP, int CH>
__device__ __forceinline__ float load_chunks(u32x4 (&raw)[CH], const u32x4* xrow, int t, int nchunks) {
#pragma unroll
    for (int c = 0; c < CH; c++) {
        // a 32-bit offset from the row: one register of address a load where the row is the workgroup's
        const unsigned at = (unsigned)(c * STEP + t < nchunks ? c * STEP + t : nchunks - 1) * 16;
        raw[c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(xrow) + at));
    }
    float amax = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; c++) amax = absmax8_bf16(raw[c], amax);
    return amax;
}
template <int STEP, int CH>
__device__ __forceinline__ void store_chunks(const u32x4 (&raw)[CH], RowQuant rq, u32x2* qrow, int t, int nchunks) {
    auto store = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const u32x2 q = quantize8_bf16(raw[c], rq);
            if (c * STEP + t < nchunks) __builtin_nontemporal_store(q, qrow + c * STEP + t);
        }
    };
    // one branch over all chunks
    if (rq.fast) {
        rq.fast = true;
        store();
    } else {
        rq.fast = false;
        store();
    }
}

// One workgroup per row, the maximum through LDS.
template <int THREADS, int CH>
__global__ void __launch_bounds__(THREADS) fp8_encode_row_kernel(const uint16_t* __restrict__ X, uint8_t* __restrict__ Q,
                                                                 float* __restrict__ scales, int cols) {
    __shared__ float wmax[THREADS / 64];
    const int row = blockIdx.x;
    const int t = threadIdx.x;
    const int nchunks = cols >> 3;
    u32x4 raw[CH];
    float amax = wave_max(load_chunks<THREADS>(raw, reinterpret_cast<const u32x4*>(X + (size_t)row * cols), t, nchunks));
    if (THREADS > 64) {
        if (lane_id() == 0) wmax[t >> 6] = amax;
        __syncthreads();
        amax = wmax[0];
#pragma unroll
        for (int w = 1; w < THREADS / 64; w++) amax = fmaxf(amax, wmax[w]);
    }
    RowQuant rq = row_quant(amax);
    rq.fast = __builtin_amdgcn_readfirstlane(rq.fast);      // the row is the workgroup's
    if (t == 0) scales[row] = rq.s;
    store_chunks<THREADS>(raw, rq, reinterpret_cast<u32x2*>(Q + (size_t)row * cols), t, nchunks);
}

// Short rows: LANES lanes of a wave (a power of two) share a row, 256 / LANES rows per workgroup, the maximum by
// shuffles.  A workgroup per row spends a launch of its own and most of a wave's lanes on them: 16384 rows of 16 / 64 /
// 240 / 512 columns 8.7 / 7.8 / 8.3 / 8.1 us that way, 2.5 / 2.9 / 4.5 / 6.7 this way.
template <int LANES, int CH>
__global__ void __launch_bounds__(256) fp8_encode_short_rows_kernel(const uint16_t* __restrict__ X, uint8_t* __restrict__ Q,
                                                                    float* __restrict__ scales, int rows, int cols) {
    const unsigned mine = blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
    const unsigned row = mine < (unsigned)rows ? mine : (unsigned)rows - 1;      // lanes past the last row store nothing
    const int t = (int)threadIdx.x % LANES;
    const int nchunks = cols >> 3;
    u32x4 raw[CH];
    float amax = load_chunks<LANES>(raw, reinterpret_cast<const u32x4*>(X + (size_t)row * cols), t, nchunks);
#pragma unroll
    for (int o = LANES / 2; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
    const RowQuant rq = row_quant(amax);
    if (mine >= (unsigned)rows) return;
    if (t == 0) scales[row] = rq.s;
    store_chunks<LANES>(raw, rq, reinterpret_cast<u32x2*>(Q + (size_t)row * cols), t, nchunks);
}

// Rows too long to hold in registers (more than 65536 columns): two passes over the row (the second mostly from L2).
__global__ void __launch_bounds__(1024) fp8_encode_rows_long_kernel(const uint16_t* __restrict__ X, uint8_t* __restrict__ Q,
                                                                    float* __restrict__ scales, int cols) {
    __shared__ float wmax[16];
    const int row = blockIdx.x;
    const int t = threadIdx.x;
    const int nchunks = cols >> 3;
    const u32x4* xrow = reinterpret_cast<const u32x4*>(X + (size_t)row * cols);
    float amax = 0.0f;
    for (int idx = t; idx < nchunks; idx += 1024) amax = absmax8_bf16(xrow[idx], amax);
    amax = wave_max(amax);
    if (lane_id() == 0) wmax[t >> 6] = amax;
    __syncthreads();
    amax = wmax[0];
#pragma unroll
    for (int w = 1; w < 16; w++) amax = fmaxf(amax, wmax[w]);
    const RowQuant rq = row_quant(amax);
    if (t == 0) scales[row] = rq.s;
    u32x2* qrow = reinterpret_cast<u32x2*>(Q + (size_t)row * cols);
    for (int idx = t; idx < nchunks; idx += 1024) qrow[idx] = quantize8_bf16(xrow[idx], rq);
}

// Eight codes per thread: one 8-byte load, one 16-byte store, both contiguous over a wave, the store non-temporal.
// (8192 x 8192: 33.3 us; with 16 codes a thread the two stores of a lane interleave at 32 bytes and the launch takes 37.8,
// and the 64-bit division for the row, now a multiply-high, another 0.3.)  cols % 16 == 0: no chunk straddles two rows.
__global__ void __launch_bounds__(256) fp8_decode_rows_kernel(const uint8_t* __restrict__ Q, const float* __restrict__ scales,
                                                              uint16_t* __restrict__ Y, unsigned chunks_per_row,
                                                              unsigned inv_chunks_per_row, unsigned nchunks) {
    const unsigned idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= nchunks) return;
    const float s = scales[fast_div(idx, chunks_per_row, inv_chunks_per_row)];
    const u32x2 q = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(Q) + idx);
    u32x4 o;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(q[j], false);
        const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(q[j], true);
        o[2 * j] = cvt_bf16x2(__fmul_rn(lo.x, s), __fmul_rn(lo.y, s));
        o[2 * j + 1] = cvt_bf16x2(__fmul_rn(hi.x, s), __fmul_rn(hi.y, s));
    }
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(Y) + idx);
}

// NBUF > 0: all buffers' codes requested before any is added; 0: any number, one after the other.
template <int NBUF>
__global__ void __launch_bounds__(256) fp8_reduce_rows_kernel(const uint8_t* __restrict__ Q, const float* __restrict__ scales,
                                                              uint16_t* __restrict__ Y, int nbuf_rt, size_t q_buf_stride,
                                                              size_t s_buf_stride, unsigned chunks_per_row,
                                                              unsigned inv_chunks_per_row, unsigned nchunks) {
    const unsigned idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= nchunks) return;
    const int nbuf = NBUF > 0 ? NBUF : nbuf_rt;
    const unsigned row = fast_div(idx, chunks_per_row, inv_chunks_per_row);
    float acc[16];
#pragma unroll
    for (int e = 0; e < 16; e++) acc[e] = 0.0f;

    auto accumulate = [&](const u32x4 q, const float s) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(q[j], false);
            const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(q[j], true);
            acc[4 * j + 0] = __fadd_rn(acc[4 * j + 0], __fmul_rn(lo.x, s));
            acc[4 * j + 1] = __fadd_rn(acc[4 * j + 1], __fmul_rn(lo.y, s));
            acc[4 * j + 2] = __fadd_rn(acc[4 * j + 2], __fmul_rn(hi.x, s));
            acc[4 * j + 3] = __fadd_rn(acc[4 * j + 3], __fmul_rn(hi.y, s));
        }
    };

    if (NBUF > 0) {
        u32x4 q[NBUF > 0 ? NBUF : 1];
        float s[NBUF > 0 ? NBUF : 1];
#pragma unroll
        for (int b = 0; b < NBUF; b++) {
            q[b] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(Q + (size_t)b * q_buf_stride) + idx);
            s[b] = scales[(size_t)b * s_buf_stride + row];
        }
#pragma unroll
        for (int b = 0; b < NBUF; b++) accumulate(q[b], s[b]);
    } else {
        for (int b = 0; b < nbuf; b++) {
            const u32x4 q = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(Q + (size_t)b * q_buf_stride) + idx);
            accumulate(q, scales[(size_t)b * s_buf_stride + row]);
        }
    }

    u32x4 o[2];
#pragma unroll
    for (int j = 0; j < 8; j++) o[j >> 2][j & 3] = cvt_bf16x2(acc[2 * j], acc[2 * j + 1]);
    // plain stores: with 32 bytes per lane the non-temporal hint costs a third of the bandwidth
    // (measured 3.9 vs 6.0 TB/s for a 1-read : 2-write pattern)
    u32x4* y = reinterpret_cast<u32x4*>(Y) + 2 * (size_t)idx;
    y[0] = o[0];
    y[1] = o[1];
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int launch_fp8_encode_rows(const void* X, uint8_t* Q, float* scales, int rows, int cols, hipStream_t stream) {
    if (!X || !Q || !scales || rows <= 0 || cols <= 0 || (cols & 15)) return SG_BAD_ARGUMENT;
    if (!aligned16(X) || !aligned16(Q)) return SG_BAD_ALIGNMENT;
    const int nchunks = cols >> 3;
    const uint16_t* x = reinterpret_cast<const uint16_t*>(X);
#define SG_SHORT(LANES, CH) \
    fp8_encode_short_rows_kernel<LANES, CH><<<((unsigned)rows + 256 / LANES - 1) / (256 / LANES), 256, 0, stream>>>(x, Q, scales, rows, cols)
#define SG_ROW(THREADS, CH) fp8_encode_row_kernel<THREADS, CH><<<rows, THREADS, 0, stream>>>(x, Q, scales, cols)
    // The smallest group of threads that holds the row in two chunks each (from 32 columns on), lanes of a shared wave up
    // to 512 columns and a workgroup beyond; from 4112 columns on, with more than 1024 rows (and 256 beyond 8192 columns),
    // half as many threads of four chunks (2048 x 4112 7.8 us in two chunks, 7.2 in four; 1024 x 4112 the other way round).
    // us, cold, against 64 / 128 / 256 threads a row as many as needed: 16384 x 1024 15.0 -> 11.1, 16384 x 2048 28.5 -> 19.7,
    // 8192 x 4096 19.8 -> 19.1, 1024 x 8192 6.5 -> 6.3, 16 x 14336 4.2 -> 3.2, 2048 x 16384 20.9 -> 19.6, but 1500 x 6144
    // 6.9 -> 7.3 and 1200 x 8192 7.3 -> 7.6; above 16384 columns against two passes over the row: 512 x 32768 23.3 -> 11.4,
    // 64 x 65536 29.3 -> 7.6.
    if (nchunks <= 2) SG_SHORT(2, 1);
    else if (nchunks <= 4) SG_SHORT(4, 1);
    else if (nchunks <= 8) SG_SHORT(8, 1);
    else if (nchunks <= 16) SG_SHORT(16, 1);
    else if (nchunks <= 32) SG_SHORT(16, 2);
    else if (nchunks <= 64) SG_SHORT(32, 2);
    else if (nchunks <= 128) SG_ROW(64, 2);
    else if (nchunks <= 256) SG_ROW(128, 2);
    else if (nchunks <= 512) SG_ROW(256, 2);
    else if (nchunks <= 1024 && rows <= 1024) SG_ROW(512, 2);
    else if (nchunks <= 1024) SG_ROW(256, 4);
    else if (nchunks <= 2048 && rows <= 256) SG_ROW(1024, 2);
    else if (nchunks <= 2048) SG_ROW(512, 4);
    else if (nchunks <= 4096) SG_ROW(1024, 4);
    else if (nchunks <= 8192) SG_ROW(1024, 8);
    else fp8_encode_rows_long_kernel<<<rows, 1024, 0, stream>>>(x, Q, scales, cols);
#undef SG_SHORT
#undef SG_ROW
    return hipGetLastError() == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}

// The decode and reduce kernels count chunks in 32 bits: a larger matrix goes in slabs of whole rows, at most 2^30 chunks
// each.  launch(first row, rows) enqueues one slab.
template <class Launch>
static int in_slabs(int rows, unsigned chunks_per_row, Launch&& launch) {
    const size_t slab = 0x40000000u / chunks_per_row;   // (cols is an int: at least four rows)
    for (size_t r0 = 0; r0 < (size_t)rows; r0 += slab) {
        launch(r0, (size_t)rows - r0 < slab ? (size_t)rows - r0 : slab);
        if (hipGetLastError() != hipSuccess) return SG_LAUNCH_FAILED;
    }
    return SG_SUCCESS;
}

int launch_fp8_decode_rows(const uint8_t* Q, const float* scales, void* Y, int rows, int cols, hipStream_t stream) {
    if (!Q || !scales || !Y || rows <= 0 || cols <= 0 || (cols & 15)) return SG_BAD_ARGUMENT;
    if (!aligned16(Q) || !aligned16(Y)) return SG_BAD_ALIGNMENT;
    const unsigned per_row = (unsigned)cols >> 3, inv = div_reciprocal(per_row);
    return in_slabs(rows, per_row, [&](size_t r0, size_t nrows) {
        const unsigned nchunks = (unsigned)nrows * per_row;
        fp8_decode_rows_kernel<<<(nchunks + 255) / 256, 256, 0, stream>>>(
            Q + r0 * (size_t)cols, scales + r0, reinterpret_cast<uint16_t*>(Y) + r0 * (size_t)cols, per_row, inv, nchunks);
    });
}

int launch_fp8_reduce_rows(const uint8_t* Q, const float* scales, void* Y, int nbuf, size_t q_buf_stride, int rows,
                           int cols, hipStream_t stream) {
    if (!Q || !scales || !Y || nbuf <= 0 || rows <= 0 || cols <= 0 || (cols & 15)) return SG_BAD_ARGUMENT;
    if (!aligned16(Q) || !aligned16(Y) || (q_buf_stride & 15)) return SG_BAD_ALIGNMENT;
    if (nbuf > 1 && q_buf_stride < (size_t)rows * cols) return SG_BAD_ARGUMENT;
    const unsigned per_row = (unsigned)cols >> 4, inv = div_reciprocal(per_row);
    return in_slabs(rows, per_row, [&](size_t r0, size_t nrows) {
        const unsigned nchunks = (unsigned)nrows * per_row;
        const unsigned grid = (nchunks + 255) / 256;
        const uint8_t* q = Q + r0 * (size_t)cols;
        uint16_t* y = reinterpret_cast<uint16_t*>(Y) + r0 * (size_t)cols;
#define SG_REDUCE(NBUF) \
    fp8_reduce_rows_kernel<NBUF><<<grid, 256, 0, stream>>>(q, scales + r0, y, nbuf, q_buf_stride, (size_t)rows, per_row, inv, nchunks)
        switch (nbuf) {
            case 1: SG_REDUCE(1); break;
            case 2: SG_REDUCE(2); break;
            case 3: SG_REDUCE(3); break;
            case 4: SG_REDUCE(4); break;
            case 5: SG_REDUCE(5); break;
            case 6: SG_REDUCE(6); break;
            case 7: SG_REDUCE(7); break;
            case 8: SG_REDUCE(8); break;
            default: SG_REDUCE(0); break;
        }
#undef SG_REDUCE
    });
}

}  // namespace sg
