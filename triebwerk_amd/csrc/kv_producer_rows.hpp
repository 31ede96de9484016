// kv_producer_rows.hpp -- the producers of q and k over the rows of many tokens, a vector on 16 lanes: the body of
// producer_rows_kernel, and of the workgroups of append_tokens_kernel that transform a prompt's queries.
#pragma once

#include "kv_common.hpp"
#include "kv_kernels.hpp"
#include "kv_producer_util.hpp"

namespace twkv {

constexpr int kProducerThreads = 256;
constexpr int kProducerSteps = 2;              // vectors of a 16-lane group: their loads are under way together
constexpr int kProducerVecs = kProducerThreads / 16 * kProducerSteps;      // vectors of a workgroup

// Vectors first_vec .. first_vec + kProducerVecs - 1 of (row, head): per_row heads to a row, Q heads first, then K heads, then
// (write_cache) V heads, as in producer_kernel.
__device__ __forceinline__ void producer_rows(const ProducerArgs& a, long long first_vec, int per_row) {
    const int c = threadIdx.x & 15;
    const long long total = (long long)a.rows * per_row;
    const bool roped = a.cos_table != nullptr;
    uint4 raw[kProducerSteps], cp[kProducerSteps] = {}, sp[kProducerSteps] = {};
    half_t* dst[kProducerSteps];
    const half_t* weight[kProducerSteps];
    bool live[kProducerSteps], xform[kProducerSteps];
#pragma unroll
    for (int i = 0; i < kProducerSteps; i++) {
        const long long v = first_vec + i * (kProducerThreads / 16) + (threadIdx.x >> 4);
        live[i] = v < total;
        const unsigned vc = (unsigned)(live[i] ? v - first_vec : 0);           // (a group past the end: any vector, not stored)
        const unsigned row0 = (unsigned)(first_vec / per_row), off = (unsigned)(first_vec - (long long)row0 * per_row) + vc;
        const int row = (int)(row0 + off / (unsigned)per_row);
        int head = (int)(off % (unsigned)per_row);
        const int pos = a.positions ? a.positions[row] : a.pos_scalar;
        const half_t* src;
        xform[i] = true;
        if (head < a.num_heads) {
            src = dst[i] = a.q + (long long)row * a.q_stride + (long long)head * kHeadDim;
            weight[i] = a.q_weight;
        } else {
            head -= a.num_heads;
            const bool is_v = head >= a.num_kv_heads;
            if (is_v) head -= a.num_kv_heads;
            half_t* at = (is_v ? a.v : a.k) + (long long)row * a.kv_stride + (long long)head * kHeadDim;
            src = dst[i] = at;
            weight[i] = a.k_weight;
            xform[i] = !is_v;
            if (a.write_cache) {
                const long long crow = cache_row(a.block_table, a.bt_stride, a.seq_stride_rows, row, pos);
                dst[i] = (is_v ? a.cache_v : a.cache_k) + crow * a.kv_dim + (long long)head * kHeadDim;
            }
        }
        raw[i] = reinterpret_cast<const uint4*>(src)[c];
        if (roped) {
            const long long at = (long long)pos * (a.rope_dim >> 4) + rope_piece16(c, a.rope_dim);
            cp[i] = reinterpret_cast<const uint4*>(a.cos_table)[at];
            sp[i] = reinterpret_cast<const uint4*>(a.sin_table)[at];
        }
    }
#pragma unroll
    for (int i = 0; i < kProducerSteps; i++) {
        if (xform[i]) {                            // the same for the 16 lanes of a vector
            float x[8];
            unpack_halves(raw[i], x);
            if (a.norm) norm_head16(x, reinterpret_cast<const uint4*>(weight[i])[c], a.eps, a.biased);
            if (roped) rope_head16(x, cp[i], sp[i], c, a.rope_dim, a.single_order);
            raw[i] = pack_halves(x);
        }
        if (live[i]) reinterpret_cast<uint4*>(dst[i])[c] = raw[i];
    }
}

}  // namespace twkv
