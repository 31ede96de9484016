// kv_producer_util.hpp -- per-head RMSNorm and rotary embedding of one head vector held by one wave
// (lane l: coordinates l and l + 64), with the reference's roundings (qk_norm_batch_kernel, kernels.cu:880-923;
// rope_batch_kernel, 927-961; rope_kernel, 193-235): kv_producer.hip with few vectors.  Second half:
// the same with a vector on 16 lanes (kv_decode_fused.hip, kv_append_tokens.hip, kv_producer.hip with many vectors).
//
// Every product is rounded to fp32 before anything else happens to it, as in the reference's separate
// kernels: no fused multiply-add where the source has none, and no multiply fused into the conversion to
// fp16 (one rounding instead of two changes a result in a few hundred thousand).
#pragma once

#include "kv_common.hpp"

namespace twkv {

// sum over the 128 coordinates of a head in the reference's order; lane l passes (x[l], x[l + 64])
__device__ __forceinline__ float head_tree_sum(float a, float b) {
#pragma clang fp contract(off)
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {     // lanes 0 and 32 end up with the sums of their 32 coordinates
        a += __shfl_down(a, off, 32);
        b += __shfl_down(b, off, 32);
    }
    const float t = a + b;                        // lane 0: s0 + s2, lane 32: s1 + s3
    return __shfl(t, 0, 64) + __shfl(t, 32, 64);
}

struct HeadXform {
    const half_t* weight;   // NULL: no RMSNorm
    float eps;
    int biased;
    const half_t* cos_row;  // NULL: no rotation; row of rope_dim / 2 entries for this position
    const half_t* sin_row;
    int rope_dim;
    int single_order;       // second output as fma(x1, c, x0 * s)
};

// RMSNorm and rotation of one head held as (x0 = coordinate lane, x1 = coordinate lane + 64), with the
// fp16 rounding after each step
__device__ __forceinline__ void xform_head(float& x0, float& x1, int lane, const HeadXform& t) {
#pragma clang fp contract(off)
    if (t.weight) {
        const float sum = head_tree_sum(x0 * x0, x1 * x1);
        const float rms = 1.0f / sqrtf(sum / (float)kHeadDim + t.eps);
        float w0 = (float)t.weight[lane], w1 = (float)t.weight[lane + 64];
        if (t.biased) { w0 += 1.0f; w1 += 1.0f; }
        x0 = as_half_value((x0 * rms) * w0);
        x1 = as_half_value((x1 * rms) * w1);
    }
    if (t.cos_row) {
        const int half = t.rope_dim >> 1;
        if (half == 64) {
            const float c = (float)t.cos_row[lane], s = (float)t.sin_row[lane];
            const float o0 = __builtin_fmaf(x0, c, -(x1 * s));
            const float o1 = t.single_order ? __builtin_fmaf(x1, c, x0 * s) : __builtin_fmaf(x0, s, x1 * c);
            x0 = as_half_value(o0);
            x1 = as_half_value(o1);
        } else {
            // coordinate d < rope_dim pairs with d + half (d < half) or d - half; only x0's coordinates
            // (d = lane < 64) can be inside a partial rotation
            const bool first = lane < half, inside = lane < t.rope_dim;
            const int partner = first ? lane + half : lane - half;
            const float other = __shfl(x0, inside ? partner : lane, 64);
            if (inside) {
                const int j = first ? lane : partner;
                const float c = (float)t.cos_row[j], s = (float)t.sin_row[j];
                const float a = first ? x0 : other, b = first ? other : x0;      // (x_d, x_{d + half})
                const float o = first ? __builtin_fmaf(a, c, -(b * s))
                                      : (t.single_order ? __builtin_fmaf(b, c, a * s) : __builtin_fmaf(a, s, b * c));
                x0 = as_half_value(o);
            }
        }
    }
}

// ---------------------------------------------------------------- one vector on 16 lanes
// Lane c = lane % 16 holds coordinates 8c .. 8c + 7, which is one 16-byte access, and every exchange inside the vector is a
// DPP modifier or (partial rotations) one cross-lane read of packed halves: a wave does four vectors with a quarter of
// the instructions of the layout above.  All 16 lanes of a vector must be active.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
constexpr int kDppQuadXor1 = 0xB1, kDppQuadXor2 = 0x4E, kDppRowRor4 = 0x124, kDppRowRor8 = 0x128;

// The sum of the reference's tree over t[e] of coordinate 8c + e: offsets 16 and 8 of the 32-lane tree are two lanes and one
// lane away, offsets 4, 2, 1 are a lane's own; then (s0 + s2) + (s1 + s3).  Every addition has the operands of
// head_tree_sum, at most swapped, so every lane of the vector gets the same bits.
__device__ __forceinline__ float head_tree_sum16(const float (&t)[8]) {
#pragma clang fp contract(off)
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float a = t[e] + dpp_move<kDppQuadXor2>(t[e]);
        v[e] = a + dpp_move<kDppQuadXor1>(a);
    }
    float s = ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
    s = s + dpp_move<kDppRowRor8>(s);
    return s + dpp_move<kDppRowRor4>(s);
}

__device__ __forceinline__ void unpack_halves(const uint4& p, float (&x)[8]) {
    const uint32_t w[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        union { uint32_t u; half_t h[2]; } cv;
        cv.u = w[i];
        x[2 * i] = (float)cv.h[0];
        x[2 * i + 1] = (float)cv.h[1];
    }
}
// of values that are fp16 values already
__device__ __forceinline__ uint4 pack_halves(const float (&x)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        union { uint32_t u; half_t h[2]; } cv;
        cv.h[0] = (half_t)x[2 * i];
        cv.h[1] = (half_t)x[2 * i + 1];
        w[i] = cv.u;
    }
    return uint4{w[0], w[1], w[2], w[3]};
}

// per-head RMSNorm; w: the lane's eight weights
__device__ __forceinline__ void norm_head16(float (&x)[8], const uint4& w, float eps, int biased) {
#pragma clang fp contract(off)
    float t[8], wv[8];
#pragma unroll
    for (int e = 0; e < 8; e++) t[e] = x[e] * x[e];
    const float rms = 1.0f / sqrtf(head_tree_sum16(t) / (float)kHeadDim + eps);
    unpack_halves(w, wv);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        if (biased) wv[e] += 1.0f;
        x[e] = as_half_value((x[e] * rms) * wv[e]);
    }
}

// Which 16-byte piece of a rotary table row lane c wants (rope_dim 128, or a multiple of 16 up to 64)
__device__ __forceinline__ int rope_piece16(int c, int rope_dim) {
    const int half_pieces = rope_dim >> 4;
    return c < half_pieces ? c : (c < 2 * half_pieces ? c - half_pieces : 0);
}

// rotary embedding; cp, sp: piece rope_piece16() of the position's table rows
__device__ __forceinline__ void rope_head16(float (&x)[8], const uint4& cp, const uint4& sp, int c, int rope_dim, int single_order) {
#pragma clang fp contract(off)
    const int half_pieces = rope_dim >> 4;
    const bool first = c < half_pieces, inside = c < 2 * half_pieces;
    float o[8], cs[8], sn[8];
    if (half_pieces == 8) {
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = dpp_move<kDppRowRor8>(x[e]);
    } else {
        const int from = (int)(threadIdx.x & 48) + (first ? c + half_pieces : (inside ? c - half_pieces : c));
        const uint4 p = pack_halves(x);
        const uint4 other = {(uint32_t)__shfl((int)p.x, from, 64), (uint32_t)__shfl((int)p.y, from, 64),
                             (uint32_t)__shfl((int)p.z, from, 64), (uint32_t)__shfl((int)p.w, from, 64)};
        unpack_halves(other, o);
    }
    unpack_halves(cp, cs);
    unpack_halves(sp, sn);
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float a = __builtin_fmaf(x[e], cs[e], -(o[e] * sn[e]));
        const float b = single_order ? __builtin_fmaf(x[e], cs[e], o[e] * sn[e]) : __builtin_fmaf(o[e], sn[e], x[e] * cs[e]);
        if (inside) x[e] = as_half_value(first ? a : b);
    }
}

}  // namespace twkv
