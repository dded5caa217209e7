// fp32 batch sum for gfx950:  D[m,n] = sum_b (A[b,m,n] + B[b,m,n]).
//
// Restates tiled_sum_reduce/src.cu:11-50: per element the batches are visited in order and
// each step adds (A + B) to the running sum, so the result is bit-identical to the host
// loop in tiled_sum_reduce/test.cu:5-26.  The reference gives every wave an 8 x 64 tile of
// 8 scalar loads per lane; here a lane owns CH pieces of four consecutive floats, a workgroup's width
// apart, so that a workgroup reads CH * 4 KB contiguous bytes of every operand and batch.  The 2*b
// streams of this kernel start whole multiples of m*n*4 bytes apart - typically the same
// channel and bank, different rows - and what decides the rate of a large sum is how much of a DRAM row a
// stream takes per visit: 32 KB per workgroup and stream (CH = 8) with one batch in flight
// reaches 6.4-7.0 TB/s on 8-16 batches of 16-32 MB, 4 KB with four batches in flight 5.3-5.6.
// Below that it is how evenly the workgroups go over the CUs, and for small sums how many round trips to memory
// stand one behind the other (kSums, below).  Any m, n: the piece that crosses m*n is summed
// four floats back and stored in part.
//
// tiled_sum_reduce_async/src.cu:13-177 stages the same sum through an LDS queue: producer waves copy
// batch slices of A and B into QSIZE slots, consumer waves wait on flag bytes, add and free the slots.
// Its counterpart here (tiled_sum_reduce_ring_kernel) keeps the queue and drops the flags: every wave
// fills its own slots with direct-to-LDS loads (global_load_lds_dwordx4, 1 KB per instruction, no
// registers in between), DEPTH batches ahead, and consumes them in batch order behind s_waitcnt
// vmcnt - loads complete in issue order, so the counter is the queue's head.  Same sums, same order.
#include <type_traits>

#include "sg_device.h"
#include "sg_host.h"
#include "sg_lds_kernel.h"

namespace sg {

// the part of [first, first + count) below mn, one float per lane and step, batches in order
__device__ __forceinline__ void tiled_sum_reduce_elementwise(const float* A, const float* B, float* D, int b, size_t mn,
                                                             size_t first, int steps, int stride) {
    for (int j = 0; j < steps; j++) {
        const size_t i = first + (size_t)j * stride;
        if (i >= mn) break;
        float acc = 0.f;
        for (int ib = 0; ib < b; ib++) acc = __fadd_rn(acc, __fadd_rn(A[(size_t)ib * mn + i], B[(size_t)ib * mn + i]));
        D[i] = acc;
    }
}

// A piece is loaded as four floats at an address that is a multiple of four bytes only: batch ib of an m*n that four does
// not divide starts 4, 8 or 12 bytes off, and the memory pipeline takes such 16-byte loads as they are.  One float per
// lane, step and batch - a chain of 4 * CH * b round trips - is what those sizes, and the last, partial workgroup of every
// size, took before.  8 x 1023 x 8191 163 -> 92 us, 2 x 2051 x 2051 36.6 -> 17.6, 8 x 1024 x 8190 (a ragged end) 114 -> 89.
using f32x4_at4 = f32x4 __attribute__((aligned(4)));

// The sums of a lane's CH pieces, T * 4 floats apart and all inside [0, mn), U batches asked for at once.
template <int CH, int U, int T>
__device__ __forceinline__ void tiled_sum_reduce_pieces(const float* A, const float* B, float* D, int b, size_t mn, size_t base) {
    f32x4 acc[CH];
#pragma unroll
    for (int c = 0; c < CH; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto batches = [&](int ib, auto count, int left) __attribute__((always_inline)) {   // the first `left` of `count` batches
        constexpr int N = decltype(count)::value;
        f32x4 va[N][CH], vb[N][CH];
#pragma unroll
        for (int u = 0; u < N; u++)
            if (u < left)
#pragma unroll
                for (int c = 0; c < CH; c++) {
                    const size_t at = (size_t)(ib + u) * mn + base + c * (T * 4);
                    va[u][c] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_at4*>(A + at));
                    vb[u][c] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_at4*>(B + at));
                }
#pragma unroll
        for (int u = 0; u < N; u++)
            if (u < left)
#pragma unroll
                for (int c = 0; c < CH; c++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[c][e] = __fadd_rn(acc[c][e], __fadd_rn(va[u][c][e], vb[u][c][e]));
    };
    int ib = 0;
    for (; ib + U <= b; ib += U) batches(ib, std::integral_constant<int, U>{}, U);
    if constexpr (U > 1) {
        if (ib < b) batches(ib, std::integral_constant<int, U - 1>{}, b - ib);
    }
#pragma unroll
    for (int c = 0; c < CH; c++) *reinterpret_cast<f32x4*>(D + base + c * (T * 4)) = acc[c];
}

// One piece a lane at the ragged end (mn >= 4).  The piece that crosses mn is read from [mn - 4, mn), and its floats from
// `base` on are stored.  A small launch is a chain of round trips, so four batches are asked for at once (15 x 1 x 617
// 6.2 us with floats one by one, 3.1 this way); with eight the kernel takes 76 registers, two waves per SIMD fewer, and
// 14 x 1416 x 1220 goes from 34 to 40 us.
__device__ __forceinline__ void tiled_sum_reduce_end(const float* A, const float* B, float* D, int b, size_t mn, size_t base) {
    if (base >= mn) return;
    const size_t at = base + 4 <= mn ? base : mn - 4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int ib = 0; ib < b; ib += 4) {
        f32x4 va[4], vb[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (ib + j < b) {
                va[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_at4*>(A + (size_t)(ib + j) * mn + at));
                vb[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_at4*>(B + (size_t)(ib + j) * mn + at));
            }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (ib + j < b)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] = __fadd_rn(acc[e], __fadd_rn(va[j][e], vb[j][e]));
    }
    if (at == base) {
        *reinterpret_cast<f32x4*>(D + base) = acc;
    } else {
#pragma unroll
        for (int e = 1; e < 4; e++)
            if (at + e >= base) D[at + e] = acc[e];
    }
}

// `whole` workgroups of CH pieces a lane, then one-piece workgroups for what is left: a ragged end costs no workgroup
// 8 pieces of mostly nothing.  WAVES per SIMD: with registers for all 16 loads of a batch of eight pieces the compiler issues
// them at once and the launch is slower for it (8 x 1024 x 8192 93.0 us on 128 registers, 88.2 on 79).
template <int CH, int U, int T, int WAVES>
__global__ void __launch_bounds__(T, WAVES) tiled_sum_reduce_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                  float* __restrict__ D, int b, size_t mn, unsigned whole) {
    if (blockIdx.x < whole)
        tiled_sum_reduce_pieces<CH, U, T>(A, B, D, b, mn, (size_t)blockIdx.x * (T * 4 * CH) + threadIdx.x * 4);
    else if (T != 256 || mn > 256)
        tiled_sum_reduce_end(A, B, D, b, mn, (size_t)whole * (T * 4 * CH) + (size_t)(blockIdx.x - whole) * (T * 4) + threadIdx.x * 4);
    else   // a float a lane is all there is: the shorter code is ahead (9 x 1 x 5 2.13 us, 2.58 by pieces; 2 x 1 x 82 2.07, 2.16)
        tiled_sum_reduce_elementwise(A, B, D, b, mn, threadIdx.x, 1, 0);
}

// LDS-queue variant.  WAVES waves per workgroup, each owning P pieces of 1 KB (256 floats), contiguous, of every
// operand and batch: a stage is one batch = 2*P load instructions into a slot of 2*P KB, DEPTH slots per wave.
// A lane reads back exactly the 16 bytes it asked for, so nothing is shared between lanes and the only ordering
// needed is the wave's own vmcnt (the loads) and lgkmcnt (the LDS reads, which the additions wait for before the
// slot is refilled).
template <int WAVES, int P, int DEPTH>
__global__ void __launch_bounds__(WAVES * 64) tiled_sum_reduce_ring_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                           float* __restrict__ D, int b, size_t mn) {
    constexpr int PER_STAGE = 2 * P, STAGE_BYTES = PER_STAGE * 1024, WG_FLOATS = WAVES * P * 256;
    static_assert((DEPTH - 1) * PER_STAGE <= 63, "vmcnt is a 6-bit counter");
    extern __shared__ __align__(16) uint8_t tsr_ring[];
    if ((mn & 3) != 0 || (size_t)(blockIdx.x + 1) * WG_FLOATS > mn) {
        tiled_sum_reduce_elementwise(A, B, D, b, mn, (size_t)blockIdx.x * WG_FLOATS + threadIdx.x, WG_FLOATS / (WAVES * 64),
                                     WAVES * 64);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    const size_t base = (size_t)blockIdx.x * WG_FLOATS + (size_t)wave * (P * 256) + lane * 4;
    const unsigned ring = lds_addr(tsr_ring) + (unsigned)wave * (DEPTH * STAGE_BYTES);
    const uint8_t* mine = tsr_ring + (size_t)wave * (DEPTH * STAGE_BYTES) + lane * 16;

    auto issue = [&](int ib) {
        const unsigned slot = ring + (unsigned)(ib % DEPTH) * STAGE_BYTES;
        const float* a = A + (size_t)ib * mn + base;
        const float* bb = B + (size_t)ib * mn + base;
#pragma unroll
        for (int u = 0; u < P; u++) {
            dma_1kb_stream(a + u * 256, slot + u * 1024);
            dma_1kb_stream(bb + u * 256, slot + (P + u) * 1024);
        }
    };
    f32x4 acc[P];
#pragma unroll
    for (int u = 0; u < P; u++) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto consume = [&](int ib) {
        const uint8_t* slot = mine + (size_t)(ib % DEPTH) * STAGE_BYTES;
#pragma unroll
        for (int u = 0; u < P; u++) {
            const f32x4 va = *reinterpret_cast<const f32x4*>(slot + u * 1024);
            const f32x4 vb = *reinterpret_cast<const f32x4*>(slot + (P + u) * 1024);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[u][e] = __fadd_rn(acc[u][e], __fadd_rn(va[e], vb[e]));
        }
    };
    // prologue: up to DEPTH batches in flight; batches beyond b are never issued, so the waits below count
    // what is really outstanding
    const int ahead = b < DEPTH ? b : DEPTH;
    for (int ib = 0; ib < ahead; ib++) issue(ib);
    int ib = 0;
    for (; ib + DEPTH < b; ib++) {
        wait_vmcnt<(DEPTH - 1) * PER_STAGE>();
        consume(ib);
        // the additions above have waited for the LDS reads of this slot: it may be overwritten
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(ib + DEPTH);
    }
    for (; ib < b; ib++) {                       // the last min(b, DEPTH) batches: b - 1 - ib younger stages in flight
        wait_vmcnt_upto((b - 1 - ib) * PER_STAGE);
        consume(ib);
    }
    wait_vmcnt<0>();
#pragma unroll
    for (int u = 0; u < P; u++) *reinterpret_cast<f32x4*>(D + base + u * 256) = acc[u];
}

template <int CH, int U, int T, int WAVES>
static int launch_sum(const float* A, const float* B, float* D, int b, size_t mn, hipStream_t stream) {
    constexpr size_t per = (size_t)T * 4 * CH;
    const size_t whole = mn / per, grid = whole + (mn - whole * per + T * 4 - 1) / (T * 4);
    if (grid > 0x7fffffffu) return SG_BAD_ARGUMENT;
    tiled_sum_reduce_kernel<CH, U, T, WAVES><<<(unsigned)grid, T, 0, stream>>>(A, B, D, b, mn, (unsigned)whole);
    return hipGetLastError() == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}

// Which build sums up to `most` floats, by floats a CU (of 256).  209 random sums timed on every build, us before -> now (before:
// a piece a lane below 4M floats, eight from there on):
//   * up to 1152 floats a CU the launch is b round trips, one behind the other: one-wave workgroups, so that every CU has one,
//     with eight batches in flight (15 x 32 x 2333 9.5 -> 4.7, 8 x 99 x 430 6.0 -> 3.1, 2 x 708 x 155 2.9 -> 2.5); to 2048
//     floats two pieces a lane and four batches, one workgroup a CU (15 x 40 x 9343 11.8 -> 9.5);
//   * from there on bandwidth counts, and workgroups that come out at just under one, two or three a CU: 14 x 189 x 9956
//     (230 workgroups of 8192 floats) 40.8 -> 33.5, 8 x 512 x 6000 (2.9 a CU of 4096) 38.7 -> 33.5, 16 x 1021 x 4093 (2.0 a CU of
//     8192) 96.4 -> 83.8.  In between two such marks shorter workgroups are ahead: 12 x 78 x 14953 20.4, 22-24 with longer ones;
//   * beyond 20480 floats a CU the length of a stream's visit decides, but not with up to four batches, whose few streams
//     do better on more workgroups: 2 x 5061 x 4226 73.6 -> 68.3, 1 x 157034 x 89 32.7 -> 29.7; 5 x 6246 x 2092 level.
// 250 other random sums, one launch behind the other: 0.74 of the time before in the geometric mean, nine more than 3 % behind (7 x 53 x
// 14392 9.0 -> 9.9, 1 x 2519 x 869 6.2 -> 6.8, whose launch is the one before).
struct SumBuild {
    size_t most;
    int (*launch)(const float*, const float*, float*, int, size_t, hipStream_t);
};
constexpr size_t kSumCus = 256;
constexpr int kOnePiece = 2, kLargeSum = 11;
static const SumBuild kSums[] = {
    {1152 * kSumCus, launch_sum<1, 8, 64, 6>},   {2048 * kSumCus, launch_sum<2, 4, 256, 6>},  {2944 * kSumCus, launch_sum<1, 1, 256, 8>},
    {4096 * kSumCus, launch_sum<2, 1, 256, 8>},  {5120 * kSumCus, launch_sum<1, 1, 256, 8>},  {6144 * kSumCus, launch_sum<2, 1, 256, 8>},
    {8192 * kSumCus, launch_sum<4, 1, 512, 8>},  {9728 * kSumCus, launch_sum<2, 1, 256, 8>},  {12288 * kSumCus, launch_sum<4, 1, 256, 8>},
    {16384 * kSumCus, launch_sum<8, 1, 256, 6>}, {20480 * kSumCus, launch_sum<4, 1, 256, 8>}, {0, launch_sum<2, 1, 256, 8>},
    {0, launch_sum<8, 1, 256, 6>}};

// Sums that take a piece a lane out of their turn: a float a lane or one batch, where nothing is gained by asking for several at
// once, and up to four batches of 2944 to 4096 floats a CU (one behind the other 1.045 times as long with two pieces, on 109 random
// sums; 2 x 1217 x 664 by itself 4.7 us, 5.0).  Timed by itself, a sum of two or three batches of up to 4096 or 2048 floats, or of up to
// 1024 floats, is 0.1 to 0.5 us ahead that way too (2 x 12 x 79 1.8 us against 2.3 with eight batches asked for), but 0.75 to 0.95 times as
// long with eight asked for where launches stand one behind the other.
static bool one_piece_sum(size_t mn, int b) {
    return mn <= 256 || (b < 2 && mn <= kSums[kOnePiece].most) || (b <= 4 && mn > 2944 * kSumCus && mn <= 4096 * kSumCus);
}

int launch_tiled_sum_reduce(const float* A, const float* B, float* D, int b, int m, int n, hipStream_t stream) {
    if (!A || !B || !D || b < 0 || m <= 0 || n <= 0) return SG_BAD_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(D)) & 15u)
        return SG_BAD_ALIGNMENT;
    const size_t mn = (size_t)m * n;
    if (one_piece_sum(mn, b)) return kSums[kOnePiece].launch(A, B, D, b, mn, stream);
    int i = 0;
    while (i < kLargeSum && mn > kSums[i].most) i++;
    if (i == kLargeSum && b > 4) i++;
    return kSums[i].launch(A, B, D, b, mn, stream);
}

int launch_tiled_sum_reduce_ring(const float* A, const float* B, float* D, int b, int m, int n, hipStream_t stream) {
    if (!A || !B || !D || b < 0 || m <= 0 || n <= 0) return SG_BAD_ARGUMENT;
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(D)) & 15u)
        return SG_BAD_ALIGNMENT;
    const size_t mn = (size_t)m * n;
    // 32 KB of every operand and batch per workgroup (eight waves x 4 KB), two batches in flight: 128 KB of LDS,
    // one workgroup per CU; small problems take 4 KB per workgroup, four batches in flight
    if (mn >= ((size_t)4 << 20)) {
        constexpr int WAVES = 8, P = 4, DEPTH = 2;
        static bool configured[64] = {};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return SG_LAUNCH_FAILED;
        constexpr unsigned lds = WAVES * DEPTH * 2 * P * 1024;
        if (!configured[dev]) {
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(tiled_sum_reduce_ring_kernel<WAVES, P, DEPTH>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
                return SG_LAUNCH_FAILED;
            configured[dev] = true;
        }
        const size_t grid = (mn + WAVES * P * 256 - 1) / (WAVES * P * 256);
        if (grid > 0x7fffffffu) return SG_BAD_ARGUMENT;
        tiled_sum_reduce_ring_kernel<WAVES, P, DEPTH><<<(unsigned)grid, WAVES * 64, lds, stream>>>(A, B, D, b, mn);
    } else {
        constexpr int WAVES = 4, P = 1, DEPTH = 4;
        const size_t grid = (mn + WAVES * P * 256 - 1) / (WAVES * P * 256);
        tiled_sum_reduce_ring_kernel<WAVES, P, DEPTH><<<(unsigned)grid, WAVES * 64, WAVES * DEPTH * 2 * P * 1024, stream>>>(A, B, D, b, mn);
    }
    return hipGetLastError() == hipSuccess ? SG_SUCCESS : SG_LAUNCH_FAILED;
}

}  // namespace sg
