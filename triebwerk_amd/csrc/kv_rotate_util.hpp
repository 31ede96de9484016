// kv_rotate_util.hpp -- pieces shared by the kernels that apply the 128x128 rotation on matrix cores: as the reference's fp32 chain with
// v_mfma_f32_16x16x4_f32 (kv_rotate.hip), and as sums of v_mfma_f32_16x16x32_f16 that decide a code where they can, with that chain behind
// them (kv_append_tokens.hip, kv_decode_fused.hip, kv_decode_layers.hip).  Lane (i = lane % 16, kk = lane / 16) of a wave
// holds, for one row of R and one vector, the coordinates 4s + kk, s = 0..31.
#pragma once

#include "kv_common.hpp"
#include "kv_kernels.hpp"

namespace twkv {

// fp16 at index (4s + kk) of a row held as 16 x (8 halves): s = 2*q + e picks dword (2e + kk/2) of 16-byte
// piece q, half kk%2.
__device__ __forceinline__ float pick_half(const uint4& piece, int e, int kk) {
    uint32_t lo = e ? piece.z : piece.x;
    uint32_t hi = e ? piece.w : piece.y;
    uint32_t w = (kk & 2) ? hi : lo;
    w = (kk & 1) ? (w >> 16) : (w & 0xffffu);
    union { uint16_t u; half_t h; } cv;
    cv.u = (uint16_t)w;
    return (float)cv.h;
}

// An operand tile in LDS: 16 rows of 128 halves (4 KB) regrouped so that lane kk * 16 + i finds its 32 halves
// (coordinates 4s + kk of row i) in one 64-byte row, row number = lane.  The four 16-byte pieces of a row are
// stored swizzled (piece p of row r at p ^ ((r / 4) % 4)): 16 lanes reading the same piece of 16 consecutive rows
// then touch all 64 banks once.
constexpr int kOperandTileDwords = 64 * 16;

__device__ __forceinline__ int operand_tile_dword(int row, int q) {
    return row * 16 + ((((q >> 2) ^ (row >> 2)) & 3) << 2) + (q & 3);
}

// raw[j] = 16-byte piece j * 64 + lane of the tile as it lies in memory (piece q = lane % 16 of row 4j + lane / 16):
// its halves e and 4 + e go to row e * 16 + (4j + lane / 16), dword q.
__device__ __forceinline__ void stage_operand_tile(uint32_t* tile, const uint4 (&raw)[4], int lane) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = 4 * j + (lane >> 4), q = lane & 15;
        tile[operand_tile_dword(0 * 16 + i, q)] = (raw[j].x & 0xffffu) | (raw[j].z << 16);
        tile[operand_tile_dword(1 * 16 + i, q)] = (raw[j].x >> 16) | (raw[j].z & 0xffff0000u);
        tile[operand_tile_dword(2 * 16 + i, q)] = (raw[j].y & 0xffffu) | (raw[j].w << 16);
        tile[operand_tile_dword(3 * 16 + i, q)] = (raw[j].y >> 16) | (raw[j].w & 0xffff0000u);
    }
}

// Lane kk * 16 + i reads row kk * 16 + i: out[s] = coordinate 4s + kk of row i of the tile.
__device__ __forceinline__ void read_operand_tile(const uint32_t* tile, int lane, float (&out)[32]) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const uint4 p = *reinterpret_cast<const uint4*>(tile + operand_tile_dword(lane, 4 * t));
        const uint32_t w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            union { uint32_t u; half_t h[2]; } cv;
            cv.u = w[e];
            out[8 * t + 2 * e] = (float)cv.h[0];
            out[8 * t + 2 * e + 1] = (float)cv.h[1];
        }
    }
}

// Sum of squares of a vector held as xv[s] = coordinate 4s + kk, in the reference's order (kernels.cu:1509-1520):
// a 32-lane shuffle-down tree per group of 32 coordinates -- its offsets 16, 8 and 4 combine coordinates that are
// congruent mod 4, which one lane owns (local j and j+4, j+2, j+1 of the group's 8 registers); offsets 2 and 1
// cross the lane groups kk -- then (s0 + s2) + (s1 + s3) over the four groups.  Every lane of a vector gets the sum.
__device__ __forceinline__ float rotation_tree_sum_sq(const float (&xv)[32]) {
    float sgrp[4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; j++) t[j] = xv[8 * w + j] * xv[8 * w + j];
        float a0 = t[0] + t[4], a1 = t[1] + t[5], a2 = t[2] + t[6], a3 = t[3] + t[7];
        float b0 = a0 + a2, b1 = a1 + a3;
        float c = b0 + b1;                                   // c_kk of the tree
        // offset 2: c0+c2 | c1+c3, offset 1: d0+d1, on the vector ALU (a shuffle is a trip through LDS)
        lane_pair_t p = __builtin_amdgcn_permlane32_swap(__float_as_uint(c), __float_as_uint(c), false, false);
        const float d = __uint_as_float(p[0]) + __uint_as_float(p[1]);
        p = __builtin_amdgcn_permlane16_swap(__float_as_uint(d), __float_as_uint(d), false, false);
        sgrp[w] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
    return (sgrp[0] + sgrp[2]) + (sgrp[1] + sgrp[3]);
}

// Buckets of the 4-bit decision boundaries: boundary i lies in a bucket of its own, at least 0.15 bucket widths from the
// bucket's edges (checked below), far more than bucket_of rounds.  A 4-bit code then comes from its bucket -- at most one
// boundary lies in each -- instead of 15 comparisons.
constexpr int kBuckets = 32;
constexpr float kBucketScale = 72.30f, kBucketShift = 16.50f;
constexpr bool edges_have_buckets() {
    int before = 0;                                // bucket 0 holds no boundary: -inf is code 0 by it
    for (int i = 0; i < 15; i++) {
        const double at = (double)kEdges4[i] * kBucketScale + kBucketShift;
        const int b = (int)at;
        if (b <= before || b >= kBuckets || at - b < 0.15 || b + 1 - at < 0.15) return false;
        before = b;
    }
    return before == kBuckets - 1;                 // the last bucket holds one: +inf and NaN are code 15 by it
}
static_assert(edges_have_buckets(), "each boundary in a bucket of its own, the last one in the last bucket");
// (the smaller bound comes last: a NaN ends up in the last bucket)
__host__ __device__ __forceinline__ int bucket_of(float x) {
    return (int)fmaxf(fminf(__builtin_fmaf(x, kBucketScale, kBucketShift), (float)(kBuckets - 1)), 0.0f);
}
// {boundary in bucket b, codes below it}
__device__ __forceinline__ float2 bucket_entry(int b) {
    float lim = 3.0e38f;
    int below = 0;
#pragma unroll
    for (int i = 0; i < 15; i++) {
        if (bucket_of(kEdges4[i]) == b) lim = kEdges4[i];
        if (bucket_of(kEdges4[i]) < b) below++;
    }
    return float2{lim, __builtin_bit_cast(float, below)};
}
// turbo_quantize by the table of the kBuckets entries (2 bit: its three comparisons, no table)
template <int BITS>
__device__ __forceinline__ uint32_t bucket_quantize(const float2* buckets, float val) {
    if constexpr (BITS == 4) {                     // (a NaN takes the last bucket, whose comparison it passes: 15, as turbo_quantize)
        const float2 e = buckets[bucket_of(val)];
        return __builtin_bit_cast(uint32_t, e.y) + (!(val < e.x) ? 1u : 0u);
    } else {
        return (uint32_t)turbo_quantize(val, 2);
    }
}

// Vectors that the forms of a step rotate back on fp16 matrix instructions are held as hi = half(x) and lo = half((x - hi) * kLowScale), whose
// products are summed apart: hi + lo / 2^11 is within 2^-23 of x itself, and within 2^-36 where x is small.  (The remainder as it is is a
// subnormal half below values of 2^-3: for values of 1e-4 one output in five was not the half nearest to its sum, with the enlarged one
// it is one in 5000, as on fp32 matrix instructions.)
constexpr float kLowScale = 2048.0f;           // a remainder is at most 2^-12 of the next power of two: no overflow
// hi and lo of x = xs / kLowScale (one instruction each from the vector held kLowScale times as large)
__device__ __forceinline__ void split_scaled(float xs, half_t& hi, half_t& lo) {
    hi = (half_t)__builtin_fmaf(xs, 1.0f / kLowScale, 0.0f);
    lo = (half_t)__builtin_fmaf((float)hi, -kLowScale, xs);
}

// K and V codes from v_mfma_f32_16x16x32_f16 -- raw fp16 coordinates, the sum scaled by 1 / |x| afterwards -- where they are sure to be those
// of the fp32 chain, whose codes the reference's are.  How far can the two be apart, for a row of R of norm |R|?
// The chain's fused multiply-adds lose at most 2^-24 of a partial sum s_k each, and the unit coordinates 2^-24 of |R| in all.  The
// matrix instructions leave the sums S_1 .. S_4 over the first 32, 64, 96 and 128 coordinates (operand j holds coordinates 32j .. 32j + 31); a
// partial sum in between is at most (|S_j| + |S_j+1| + t_j) / 2, t_j the sum of the block's |products|, and the four t_j are at most
// |R| |x| together (Cauchy-Schwarz).  With T = 2 (|S_1| + |S_2| + |S_3|) + |S_4|, the sum of all |s_k| is at most 16 T + 16 |R|, in units of |x|.
// A matrix instruction adds its 32 products to the accumulator in four groups of eight (a group: the coordinates of one lane group).  Within
// a group a product is cut off below 2^-24 of the largest one's power of two, a subnormal factor counting as 2^-14; group sums
// and additions are rounded to nearest.  (Read from the sums of single large, cancelling and small products; a test holds the instruction
// to it.)  So S_4 loses 2^-24 of at most 2 T + 2 |R| in its 16 additions, |R| in the groups' own roundings, and 7 |R'| |x'| in what is cut off, R' and
// x' with every coordinate raised to 2^-14: |R'| <= |R| + 7e-4.  Altogether 18 T + (27 + 7 * 7e-4 / |x|) |R'|, one more for y's own rounding; taken as
// 18 T + (47 + 7e-3 / |x|) |R'|.
constexpr float kUlp = 5.9604645e-8f;                          // 2^-24
// Code of y = S[3][r] * inv, inv = 1 / |x|, row_norm >= |R'|; doubt is set where y is not further than that from a boundary (or no number).
// (A value is compared with its own bucket's boundary.  Another one is at least 0.15 of a bucket away (edges_have_buckets), which the bound
// stays below for rows of norms up to kLongestRows and any vector, T being at most 7 |R| and 1 / |x| 1e6; matrices of longer rows, no
// rotations, leave no value sure.  Looking at that distance for every value instead cost 1 % of a step of 4 x 613 tokens.)
constexpr float kLongestRows = 4.0f;
static_assert(0.149 / kBucketScale > kLongestRows * (18 * 7 + 47 + 7e-3 * 1e6) * kUlp && kUnitRows < kLongestRows, "no boundary of the next bucket within the bound");
template <int BITS>
__device__ __forceinline__ uint32_t bucket_quantize_sure(const float2* buckets, const float4_t (&S)[4], int r, float inv, float row_norm, bool& doubt) {
    const float val = S[3][r] * inv;
    const float sums = __builtin_fmaf(2.0f, fabsf(S[0][r]) + fabsf(S[1][r]) + fabsf(S[2][r]), fabsf(S[3][r]));
    const float eps = __builtin_fmaf(inv, __builtin_fmaf(sums, 18.0f * kUlp, row_norm * (7e-3f * kUlp)), row_norm * (47.0f * kUlp));
    if constexpr (BITS == 4) {
        const float2 e = buckets[bucket_of(val)];
        doubt = doubt || !(fabsf(val - e.x) > eps);
        return __builtin_bit_cast(uint32_t, e.y) + (!(val < e.x) ? 1u : 0u);
    } else {
        doubt = doubt || !(fminf(fabsf(val), fabsf(fabsf(val) - kEdges2[2])) > eps);
        return (uint32_t)turbo_quantize(val, 2);
    }
}
// What a known rotation is given as (kUnitRows) is above |R'|, its rows being of norm 1 within 1e-4; for any other R the kernels take the norm
// from its rows.
static_assert(kUnitRows > 1.0001f + 7e-4f, "the norm of R'");
__device__ __forceinline__ float larger_norm(float x, float y) { return x > y || x != x ? x : y; }      // (a NaN in x stays, one in y is taken)
// |R'| of the longest of the 16 rows of R whose halves the lanes of a wave hold as operands (16 lanes a row quarter); a row that is no
// number, or longer than kLongestRows, leaves none sure.
__device__ __forceinline__ float operand_rows_norm(const uint4 (&rows)[4]) {
    float n2 = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t w[4] = {rows[j].x, rows[j].y, rows[j].z, rows[j].w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const half2_t h = __builtin_bit_cast(half2_t, w[i]);
            n2 = __builtin_amdgcn_fdot2(h, h, n2, false);
        }
    }
    typedef unsigned swapped_t __attribute__((ext_vector_type(2)));
    swapped_t w = __builtin_amdgcn_permlane16_swap(__float_as_uint(n2), __float_as_uint(n2), false, false);
    n2 = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    w = __builtin_amdgcn_permlane32_swap(__float_as_uint(n2), __float_as_uint(n2), false, false);
    n2 = __uint_as_float(w[0]) + __uint_as_float(w[1]);
    auto larger = [](float x, int moved) { return larger_norm(x, __builtin_bit_cast(float, moved)); };
    n2 = larger(n2, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, n2), 0xB1, 0xf, 0xf, true));      // 1, 2, then 4 and 8 rows apart
    n2 = larger(n2, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, n2), 0x4E, 0xf, 0xf, true));
    n2 = larger(n2, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, n2), 0x141, 0xf, 0xf, true));
    n2 = larger(n2, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, n2), 0x140, 0xf, 0xf, true));
    const float n = __builtin_fmaf(1.001f, __builtin_amdgcn_sqrtf(n2), 7e-4f);
    return n <= kLongestRows ? n : __builtin_inff();
}

}  // namespace twkv
