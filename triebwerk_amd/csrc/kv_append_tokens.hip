// kv_append_tokens.hip -- the compressed append of a prompt's rows (turbo_kv_quantize_kernel, kernels.cu:1482-1559), with
// the producers of q and k on the way (qk_norm_batch, rope_batch, 880-961), in one launch (gfx950).
//
// rotate_kernel (kv_rotate.hip) gives every wave 16 output coordinates of its vectors and nothing to share: right for the
// few vectors of a decode step, but each vector is then fetched, transformed, measured and regrouped eight times.  Here a
// workgroup of four waves takes a tile of 16 vectors at a time, once:
//   - 16 lanes to a vector, 16 bytes each: RMSNorm and rotation (K), the norm, and the vector into LDS as the halves it is;
//     K goes back to its row as the producers leave it;
//   - wave w rotates the tile for output coordinates 16w .. 16w + 15 and 64 + 16w ... on v_mfma_f32_16x16x32_f16 (exact products, fp32
//     sums).  A code is taken from those sums where no boundary between buckets lies within their bound of error, which 16 of 17
//     blocks of 16 vectors are through with; the others repeat the sum as rotate_kernel's chain of v_mfma_f32_16x16x4_f32, hence its
//     bits.  Codes meet in LDS and leave 16 lanes to a vector.
// One barrier per tile: tile i is rotated while tile i + 1 is transformed and the codes of tile i - 1 are stored.
// The chain alone was bound by the matrix cores (32 of its steps take 16 of the fp16 form's time); now the issue of the transformation
// and of the buckets bounds it.  Launches without producers whose tiles all run at once, one to a workgroup, keep the chain: they wait for
// memory, and a repeated block costs more than the sums save.  Other workgroups of the same launch transform the queries, a matter of memory
// alone, beside them.
// The prompt step of 4111 tokens (4 layers, 16 heads over 8 KV heads, 4 bit, producers; attention included): 893 us with the
// chain, 858 with the sums; attention's own changes take it to 839.

#include <algorithm>
#include <type_traits>

#include "kv_common.hpp"
#include "kv_kernels.hpp"
#include "kv_mfma_util.hpp"
#include "kv_producer_rows.hpp"
#include "kv_rotate_util.hpp"

namespace twkv {

namespace {

constexpr int kTileVecs = 16;
constexpr int kAppendWaves = 4;
static_assert(kAppendWaves * kWave == kProducerThreads, "the workgroups of the queries");

}  // namespace

template <int BITS, bool PROD>
__global__ void __launch_bounds__(kAppendWaves* kWave, 3)
append_tokens_kernel(AppendTokensArgs a) {
    constexpr int kHeadBytes = kHeadDim * BITS / 8;
    constexpr int kCodeRow = kHeadBytes + 4;           // bytes per vector of codes in LDS
    // two tiles of vectors as halves; first a wave's 16 rows of R each
    __shared__ __attribute__((aligned(16))) uint4 x_s[kAppendWaves * kOperandTileDwords / 4];
    static_assert(sizeof(x_s) >= 2 * kTileVecs * kHeadDim * 2, "two tiles");
    __shared__ float inv_s[2][kTileVecs];
    __shared__ __attribute__((aligned(8))) float2 bucket_s[kBuckets];
    __shared__ __attribute__((aligned(16))) char code_s[2][kTileVecs][kCodeRow];

    // workgroups in turn: a tile run of K and V, a run of queries, until one kind is used up
    int b = (int)blockIdx.x;
    if (PROD) {
        const int both = min(a.kv_blocks, a.q_blocks);
        const bool is_q = b < 2 * both ? (b & 1) != 0 : a.q_blocks > a.kv_blocks;
        b = b < 2 * both ? b >> 1 : b - both;
        if (is_q) {
            producer_rows(a.p, (long long)b * kProducerVecs, a.p.num_heads);
            return;
        }
    }
    asm volatile("" :: "s"(a.p.k), "s"(a.p.v), "s"(a.p.positions), "s"(a.rotation), "s"(a.p.kv_stride), "s"(a.nper), "s"(a.nstreams), "s"(a.p.rows),
                 "s"(a.p.num_kv_heads), "s"(PROD ? a.p.k_weight : nullptr), "s"(PROD ? a.p.cos_table : nullptr), "s"(PROD ? a.p.sin_table : nullptr));
    const int tid = threadIdx.x;
    const int wave = uniform(tid / kWave), lane = tid % kWave;
    const int i16 = lane & 15, kk = lane >> 4;
    const int vl = tid >> 4, c = tid & 15;             // vector of the tile and piece of it this thread carries
    const int Hk = a.p.num_kv_heads;
    const unsigned per_row = (unsigned)(Hk * a.nstreams);
    const int nvec = a.p.rows * (int)per_row;
    const int tile0 = b * a.nper, ntiles = min(a.nper, (nvec + kTileVecs - 1) / kTileVecs - tile0);
    const bool normed = PROD && a.p.norm, roped = PROD && a.p.cos_table != nullptr;

    // The vector a thread carries, tile by tile: 16 vectors on is q16 rows and r16 heads on.  Past the end: the last row, not stored.
    struct Vec { int row, h, v; };
    const int q16 = kTileVecs / (int)per_row, r16 = kTileVecs % (int)per_row;
    auto advance = [&](const Vec& x) -> Vec {
        Vec r = {x.row + q16, x.h + r16, x.v + kTileVecs};
        if (r.h >= (int)per_row) { r.h -= (int)per_row; r.row++; }
        return r;
    };
    const int end_v = min(nvec, (tile0 + ntiles) * kTileVecs);
    auto row_of = [&](const Vec& x) -> int { return min(x.row, a.p.rows - 1); };
    // Requests run ahead of their use: the position three tiles, the vector and its table rows two.
    struct Request { uint4 x, cp, sp; };
    auto request_pos = [&](const Vec& x) -> int { return a.p.positions[row_of(x)]; };
    auto request = [&](const Vec& x, int pos) -> Request {
        Request q{};
        const half_t* src = (x.h >= Hk ? a.p.v - (long long)Hk * kHeadDim : a.p.k) + (long long)row_of(x) * a.p.kv_stride + x.h * kHeadDim;
        q.x = reinterpret_cast<const uint4*>(src)[c];
        if (PROD) {            // (no table: the rotation is read.  A load in a branch is waited for, with all before it, at the branch's end.)
            const long long at = roped ? (long long)pos * (a.p.rope_dim >> 4) + rope_piece16(c, a.p.rope_dim) : 0;
            q.cp = reinterpret_cast<const uint4*>(roped ? a.p.cos_table : a.rotation)[at];
            q.sp = reinterpret_cast<const uint4*>(roped ? a.p.sin_table : a.rotation)[at];
        }
        return q;
    };

    Vec x0;
    x0.v = tile0 * kTileVecs + vl;
    x0.row = (int)((unsigned)x0.v / per_row);
    x0.h = (int)((unsigned)x0.v - (unsigned)x0.row * per_row);
    Vec x1 = advance(x0), x2 = advance(x1);
    int pos0 = request_pos(x0), pos1 = request_pos(x1), pos2 = request_pos(x2);
    uint4 rraw[2][4];
#pragma unroll
    for (int d = 0; d < 2; d++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            rraw[d][j] = reinterpret_cast<const uint4*>(a.rotation + (wave + 4 * d) * 16 * kHeadDim)[j * kWave + lane];
    uint4 kw{};
    if (PROD) kw = reinterpret_cast<const uint4*>(normed ? a.p.k_weight : a.rotation)[c];
    Request cur = request(x0, pos0);
    Request next = request(x1, pos1);
    if (BITS == 4 && tid < kBuckets) bucket_s[tid] = bucket_entry(tid);
    uint4 rv[2][4];                                    // R[16 * (wave + 4 d) + i16][4s + kk], s = 8j .. 8j + 7
    float row_norm = a.row_norm;
    {
        uint32_t* mine = reinterpret_cast<uint32_t*>(x_s) + wave * kOperandTileDwords;      // this wave's own: no barrier in between
#pragma unroll
        for (int d = 0; d < 2; d++) {
            stage_operand_tile(mine, rraw[d], lane);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < 4; j++) rv[d][j] = *reinterpret_cast<const uint4*>(mine + operand_tile_dword(lane, 4 * j));
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            if (a.row_norm == 0.0f && !a.chains) row_norm = larger_norm(row_norm, operand_rows_norm(rv[d]));
        }
    }
    row_norm = __builtin_bit_cast(float, uniform(__builtin_bit_cast(int, row_norm)));      // (the same in every lane: no vector register)
    lds_barrier();                                     // every wave has its rows of R

    // coordinate 4s + kk of vector v in 16-byte piece 4kk + s / 8 of its row, which lies at that piece ^ 5v (no bank twice, written or read)
    auto vec_piece = [](int buf, int v, int p) -> int { return (buf * kTileVecs + v) * 16 + ((p ^ (5 * v)) & 15); };
    // transform, measure and regroup the vector piece of tile i
    auto fill = [&](int buf, const Vec& r, int pos, const Request& q) {
        float x[8], t[8];
        unpack_halves(q.x, x);
        const bool live = r.v < end_v, is_v = r.h >= Hk;
        if (PROD && !is_v) {                           // the same for the 16 lanes of a vector
            if (normed) norm_head16(x, kw, a.p.eps, a.p.biased);
            if (roped) rope_head16(x, q.cp, q.sp, c, a.p.rope_dim, 0);
            if (live) reinterpret_cast<uint4*>(a.p.k + (long long)r.row * a.p.kv_stride + r.h * kHeadDim)[c] = pack_halves(x);
        }
        const uint4 w = PROD ? pack_halves(x) : q.x;
        const uint32_t by_kk[4] = {(w.x & 0xffffu) | (w.z << 16), (w.x >> 16) | (w.z & 0xffff0000u),
                                   (w.y & 0xffffu) | (w.w << 16), (w.y >> 16) | (w.w & 0xffff0000u)};
#pragma unroll
        for (int k4 = 0; k4 < 4; k4++)
            reinterpret_cast<uint32_t*>(&x_s[vec_piece(buf, vl, 4 * k4 + (c >> 2))])[c & 3] = by_kk[k4];
#pragma unroll
        for (int e = 0; e < 8; e++) t[e] = x[e] * x[e];                // exact: fp16 values
        const float norm = sqrtf(head_tree_sum16(t) + 1e-12f);
        if (c == 0) {
            inv_s[buf][vl] = 1.0f / norm;
            if (live) {
                const long long crow = (long long)r.row * a.seq_stride_rows + pos;
                (is_v ? a.norms[1] : a.norms[0])[crow * Hk + (is_v ? r.h - Hk : r.h)] = (half_t)norm;
            }
        }
    };
    auto store_codes = [&](int buf, const Vec& r, int pos) {
        if (r.v >= end_v) return;
        const bool is_v = r.h >= Hk;
        const long long crow = (long long)r.row * a.seq_stride_rows + pos;
        uint8_t* dst = (is_v ? a.codes[1] : a.codes[0]) + (crow * Hk + (is_v ? r.h - Hk : r.h)) * kHeadBytes + c * BITS;
        const char* src = &code_s[buf][vl][c * BITS];
        if (BITS == 4) *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(src);
        else *reinterpret_cast<uint16_t*>(dst) = *reinterpret_cast<const uint16_t*>(src);
    };

    fill(0, x0, pos0, cur);
    Vec xs = x0, xf = x0;                              // whose codes are stored next; whose piece was filled in last
    int ps = pos0, pf = pos0;
    for (int i = 0;; i++) {
        lds_barrier();      // tile i and the codes of tile i - 1 are complete; tile i - 1 and the codes of i - 2 have been read
        if (i > 0) store_codes((i - 1) & 1, xs, ps);
        if (i == ntiles) break;
        xs = xf; ps = pf;
        if (i + 1 < ntiles) {
            const Request now = next;
            xf = x1; pf = pos1;
            next = request(x2, pos2);
            x1 = x2; pos1 = pos2;
            x2 = advance(x2);
            pos2 = request_pos(x2);
            fill((i + 1) & 1, xf, pf, now);
        }
        uint4 xv[4];
#pragma unroll
        for (int j = 0; j < 4; j++) xv[j] = x_s[vec_piece(i & 1, i16, 4 * kk + j)];
        const float inv = inv_s[i & 1][i16];
        uint32_t codes[2] = {0u, 0u};
        // the fp32 chain of blocks D0 .. D1, side by side
        auto chains = [&](auto first, auto last) {
            constexpr int D0 = decltype(first)::value, D1 = decltype(last)::value;
            float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float rf[2][8], uf[8];
#pragma unroll
                for (int d = D0; d <= D1; d++) {
                    uint4 rr = rv[d][j];
                    asm volatile("" : "+v"(rr.x), "+v"(rr.y), "+v"(rr.z), "+v"(rr.w));       // not expanded ahead of the loop: 64 registers
                    unpack_halves(rr, rf[d]);
                }
                unpack_halves(xv[j], uf);
#pragma unroll
                for (int e = 0; e < 8; e++)
#pragma unroll
                    for (int d = D0; d <= D1; d++) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(rf[d][e], uf[e] * inv, acc[d], 0, 0, 0);
            }
#pragma unroll
            for (int d = D0; d <= D1; d++) {
                codes[d] = 0;
#pragma unroll
                for (int r = 0; r < 4; r++) codes[d] |= bucket_quantize<BITS>(bucket_s, acc[d][r]) << (r * BITS);
            }
        };
        constexpr std::integral_constant<int, 0> d0{};
        constexpr std::integral_constant<int, 1> d1{};
        if (a.chains) {
            chains(d0, d1);
        } else {
            // Sums of the fp16 values times the fp16 matrix: every product exact, 8 matrix instructions where the chains take 64 of twice
            // the length.  The codes are those of the chain, by the sums unless one of a block's 256 is too near to a boundary
            // for them (kv_rotate_util.hpp; one block in 17).
            float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, sums[2][4];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int d = 0; d < 2; d++) {
                    acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, rv[d][j]), __builtin_bit_cast(half8_t, xv[j]), acc[d], 0, 0, 0);
                    sums[d][j] = acc[d];
                }
            bool doubt[2] = {false, false};
#pragma unroll
            for (int d = 0; d < 2; d++)                // lane: coordinates 16 (wave + 4d) + 4kk .. + 3 of vector i16
#pragma unroll
                for (int r = 0; r < 4; r++) codes[d] |= bucket_quantize_sure<BITS>(bucket_s, sums[d], r, inv, row_norm, doubt[d]) << (r * BITS);
            if (__any(doubt[0])) chains(d0, d0);
            if (__any(doubt[1])) chains(d1, d1);
        }
#pragma unroll
        for (int d = 0; d < 2; d++) {
            const uint32_t packed = codes[d];
            char* dst = &code_s[i & 1][i16][((wave + 4 * d) * 4 + kk) * (BITS / 2)];
            if (BITS == 4) *reinterpret_cast<uint16_t*>(dst) = (uint16_t)packed;
            else *reinterpret_cast<uint8_t*>(dst) = (uint8_t)packed;
        }
    }
}

bool append_tokens_usable(const AppendTokensArgs& a) {
    auto ok = [](const void* p, unsigned m) { return (reinterpret_cast<uintptr_t>(p) & m) == 0; };
    const bool prod = a.p.norm || a.p.cos_table;
    if (prod && !producer_rows_usable(a.p)) return false;
    for (int s = 0; s < a.nstreams; s++)
        if (!ok(a.codes[s], 3u) || !ok(a.norms[s], 1u)) return false;
    return ok(a.p.k, 15u) && (a.nstreams < 2 || ok(a.p.v, 15u)) && ok(a.rotation, 15u) && (a.p.kv_stride & 7) == 0 &&
           (long long)a.p.rows * a.p.num_kv_heads * a.nstreams < (1LL << 30) && (long long)a.p.rows * a.p.num_heads < (1LL << 31);
}

void launch_append_tokens(const AppendTokensArgs& args, int bits, hipStream_t s) {
    AppendTokensArgs a = args;
    const bool prod = a.p.norm || a.p.cos_table;
    const int tiles = (a.p.rows * a.p.num_kv_heads * a.nstreams + kTileVecs - 1) / kTileVecs;
    if (tiles <= 0) return;
    // Tiles per workgroup: a workgroup's start (R, the first loads) is worth a good part of a tile, but the compute units take the
    // workgroups in turns, and a turn begun for a few of them costs all of it.  With n tiles each a launch takes start[n] and
    // turn[n] for every turn of one workgroup per compute unit: within 7 % at 23 counts of 256 to 16384 tiles, and the n with
    // the smallest sum is the fastest or within 1.4 % of it in all of them (4 bit, us with 1, 2, 3, 4: 1024 tiles 9.4, 9.3, 12.1,
    // 10.6; 1536: 13.2, 12.0, 12.2, 15.5; 2300: 18.7, 18.2, 16.5, 20.4; 4096: 30.5, 27.1, 29.0, 26.0; 8192: 57.7, 50.1, 49.9, 47.8;
    // 6 each: 52.8).
    constexpr double kStart[] = {0.0, 3.3, 3.8, 4.4, 5.2}, kTurn[] = {0.0, 1.63, 2.8, 4.0, 5.2};
    double least = 0.0;
    for (int n = 1; n <= 4; n++) {
        const int groups = (tiles + n - 1) / n, turns = (groups + compute_units() - 1) / compute_units();
        const double us = kStart[n] + kTurn[n] * turns;
        if (n == 1 || us < least) { least = us; a.nper = n; }
    }
    a.kv_blocks = (tiles + a.nper - 1) / a.nper;
    // A launch whose workgroups run all at once, a tile each, lasts as long as the one that runs the chain besides the sums: there all of
    // them run it at once (256 tokens over 8 KV heads, 4 bit: 5.2 us with the sums, 4.4 without; beside producers, which take longer, the
    // sums are faster: 200 tokens 8.1 against 8.8).
    a.chains = !prod && a.kv_blocks <= compute_units() && a.nper == 1 ? 1 : 0;
    a.q_blocks = prod ? (int)(((long long)a.p.rows * a.p.num_heads + kProducerVecs - 1) / kProducerVecs) : 0;
    // queries beside the tiles while everything runs at once; beyond that the low occupancy of this kernel costs them more than
    // a launch of their own
    if (prod && a.kv_blocks + a.q_blocks > 3 * compute_units()) {
        ProducerArgs q = a.p;
        q.num_kv_heads = 0;
        launch_producer(q, s);
        a.q_blocks = 0;
    }
    const dim3 grid(a.kv_blocks + a.q_blocks), block(kAppendWaves * kWave);
    if (bits == 4) {
        if (prod) hipLaunchKernelGGL((append_tokens_kernel<4, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((append_tokens_kernel<4, false>), grid, block, 0, s, a);
    } else {
        if (prod) hipLaunchKernelGGL((append_tokens_kernel<2, true>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((append_tokens_kernel<2, false>), grid, block, 0, s, a);
    }
}

}  // namespace twkv
