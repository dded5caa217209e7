// 2:4 prune + compress of a dense E4M3 weight matrix for gfx950: the producer side of the format
// sg_sparse24_gemm reads (values [n][k/2], one metadata nibble per group of four k).
//
// Per group of four consecutive codes the two with the largest magnitude are kept (magnitude =
// code & 0x7f, which orders E4M3 values by |x|; ties keep the lower position, so an input that is
// already 2:4 keeps its non-zeros and pads with the lowest free positions).  Kept codes are stored
// in k order; the nibble is first | second << 2 with first < second, the group with the lower k in
// the low nibble of the byte.  No counterpart in the reference, which has no compressed format.
//
// HBM-bound at 1.625 bytes per code (95 MB for 14336 x 4096: 14.5 us at the 6.6 TB/s a stream reaches).  What kept it
// at 27 us was the vector unit: ~30 integer operations per group of four, and a 64-bit division per lane for the row.
// Two groups are therefore ranked at once in the halves of packed 16-bit integers (pick_pairs, 27 operations per eight
// codes), and the row is found with one multiply-high where there is a row pitch and not at all where there is none:
// 18.1 us with 16 codes a lane.  With 32 codes a lane the stores are 16 bytes of values and 4 of metadata; lanes that
// loaded 32 adjacent bytes would ask for every line twice, so the loads stay 16 bytes apart, one contiguous KB per
// instruction, and the two lanes of a pair swap halves (one DPP move per word): 17.4 us, and 16.8 us with non-temporal
// stores, nothing being read back (14336 x 4096, cold).
#include "sg_device.h"
#include "sg_host.h"

namespace sg {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t min_u16x2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// Two groups of four codes, w0 and w1 -> their kept codes (w0's in the low half) and the complement of their metadata
// byte.  key[i] holds, for each group in a half of its own, magnitude i above 3 - i: the keys of a group are distinct and
// their order is "larger magnitude, then lower position".
__device__ __forceinline__ void pick_pairs(uint32_t w0, uint32_t w1, uint32_t& kept, uint32_t& meta_complement) {
    uint32_t key[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        // byte i of w0 to byte 1, byte i of w1 to byte 3, zero (selector 0x0c) elsewhere
        const uint32_t sel = 0x000c000cu | ((uint32_t)i << 8) | ((uint32_t)(4 + i) << 24);
        key[i] = (__builtin_amdgcn_perm(w1, w0, sel) & 0x7f007f00u) | (uint32_t)(3 - i) * 0x00010001u;
    }
    const uint32_t hi_a = max_u16x2(key[0], key[1]), lo_a = min_u16x2(key[0], key[1]);
    const uint32_t hi_b = max_u16x2(key[2], key[3]), lo_b = min_u16x2(key[2], key[3]);
    const uint32_t top = max_u16x2(hi_a, hi_b) & 0x00030003u;
    const uint32_t second = max_u16x2(min_u16x2(hi_a, hi_b), max_u16x2(lo_a, lo_b)) & 0x00030003u;
    const uint32_t a = max_u16x2(top, second), b = min_u16x2(top, second);   // 3 - first position, 3 - second position
    kept = __builtin_amdgcn_perm(w1, w0, (a | (b << 8)) ^ 0x07070303u);
    const uint32_t nibbles = a | (b << 2);                                   // 15 - nibble, per half
    meta_complement = (nibbles | (nibbles >> 12)) & 0xffu;
}

// 16 codes -> 8 values and two metadata bytes
__device__ __forceinline__ void compress16(const u32x4 w, u32x2& vals, uint32_t& meta) {
    uint32_t k0, k1, m0, m1;
    pick_pairs(w[0], w[1], k0, m0);
    pick_pairs(w[2], w[3], k1, m1);
    vals = u32x2{k0, k1};
    meta = (m0 | (m1 << 8)) ^ 0xffffu;
}

// The 16-code piece `piece` (counted row by row, per_row of them a row).
__device__ __forceinline__ const u32x4* piece_at(const uint8_t* B, unsigned piece, unsigned per_row, unsigned inv_per_row, int b_stride) {
    if ((unsigned)b_stride == per_row * 16) return reinterpret_cast<const u32x4*>(B) + piece;   // wave-uniform
    const unsigned row = fast_div(piece, per_row, inv_per_row);
    return reinterpret_cast<const u32x4*>(B + (size_t)row * (size_t)b_stride) + (piece - row * per_row);
}

// 32 codes a lane: per wave 128 pieces, loaded as two contiguous KB; even lanes take the pairs of the first, odd lanes
// those of the second.
__global__ void __launch_bounds__(256) sparse24_compress_kernel(const uint8_t* __restrict__ B, uint8_t* __restrict__ vals,
                                                                uint8_t* __restrict__ meta, unsigned pieces, unsigned per_row,
                                                                unsigned inv_per_row, int b_stride) {
    const unsigned lane = threadIdx.x & 63, odd = lane & 1;
    const unsigned first = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 128;
    u32x4 w[2] = {};
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const unsigned piece = first + h * 64 + lane;
        if (piece < pieces) w[h] = __builtin_nontemporal_load(piece_at(B, piece, per_row, inv_per_row, b_stride));
    }
    u32x4 lo, hi;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t send = odd ? w[0][e] : w[1][e];
        const uint32_t got = __builtin_amdgcn_update_dpp(0, send, 0xb1, 0xf, 0xf, false);   // quad_perm [1, 0, 3, 2]
        lo[e] = odd ? got : w[0][e];
        hi[e] = odd ? w[1][e] : got;
    }
    const unsigned pair = first / 2 + odd * 32 + (lane >> 1);
    if (pair >= pieces / 2) return;
    u32x2 v0, v1;
    uint32_t m0, m1;
    compress16(lo, v0, m0);
    compress16(hi, v1, m1);
    __builtin_nontemporal_store(u32x4{v0.x, v0.y, v1.x, v1.y}, reinterpret_cast<u32x4*>(vals) + pair);
    __builtin_nontemporal_store(m0 | (m1 << 16), reinterpret_cast<uint32_t*>(meta) + pair);
}

// 16 codes a lane, for rows of an odd number of pieces and outputs aligned to 8 and 2 bytes only.
__global__ void __launch_bounds__(256) sparse24_compress16_kernel(const uint8_t* __restrict__ B, uint8_t* __restrict__ vals,
                                                                  uint8_t* __restrict__ meta, unsigned pieces, unsigned per_row,
                                                                  unsigned inv_per_row, int b_stride) {
    const unsigned piece = blockIdx.x * 256 + threadIdx.x;
    if (piece >= pieces) return;
    u32x2 v;
    uint32_t m;
    compress16(__builtin_nontemporal_load(piece_at(B, piece, per_row, inv_per_row, b_stride)), v, m);
    reinterpret_cast<u32x2*>(vals)[piece] = v;
    reinterpret_cast<uint16_t*>(meta)[piece] = (uint16_t)m;
}

int launch_sparse24_compress(const uint8_t* B, uint8_t* vals, uint8_t* meta, int n, int k, int b_stride, hipStream_t stream) {
    const unsigned per_row = (unsigned)k >> 4, inv = div_reciprocal(per_row);
    const bool wide = k % 32 == 0 && (reinterpret_cast<uintptr_t>(vals) & 15u) == 0 && (reinterpret_cast<uintptr_t>(meta) & 3u) == 0;
    // the kernels count pieces in 32 bits: a larger matrix goes in slabs of whole rows, at most 2^30 pieces each
    const size_t slab = 0x40000000u / per_row;   // (k is an int: at least eight rows)
    for (size_t r0 = 0; r0 < (size_t)n; r0 += slab) {
        const size_t rows = (size_t)n - r0 < slab ? (size_t)n - r0 : slab;
        const unsigned pieces = (unsigned)rows * per_row;
        const uint8_t* b = B + r0 * (size_t)b_stride;
        uint8_t* v = vals + r0 * (size_t)(k >> 1);
        uint8_t* m = meta + r0 * (size_t)(k >> 3);
        if (wide) sparse24_compress_kernel<<<(pieces + 511) / 512, 256, 0, stream>>>(b, v, m, pieces, per_row, inv, b_stride);
        else sparse24_compress16_kernel<<<(pieces + 255) / 256, 256, 0, stream>>>(b, v, m, pieces, per_row, inv, b_stride);
        if (report_hip("sparse24_compress launch", hipGetLastError()) != hipSuccess) return SG_LAUNCH_FAILED;
    }
    return SG_SUCCESS;
}

}  // namespace sg
