// kv_decode_layers.hip -- the compressed decode step of EVERY layer in one launch (gfx950): what kv_decode_fused.hip does
// for one layer (append of K and V, query rotation, scan, merge, rotate-back; kernels.cu:880-961, 1563-1636, 1641-1776),
// for a caller that has the inputs of all layers at hand (tw_engine_decode_step, whose layers do not depend on each other).
//
// A workgroup owns one unit -- a sequence of a layer and HKW of its KV heads with their query heads.  Launched layer by
// layer a unit's start and end (the launch itself, trips to memory for the new token's vectors and the rotation, the merge, the
// drain) are paid by the whole chip at once, 11 us of a launch, and a batch of 4 leaves most of it idle besides.  Here
// thousands of units follow each other without a gap, and two workgroups of FOUR waves share a compute unit (a wave per
// SIMD each, 80 KB of LDS each), so that one's start and end run beside the other's scan.  That is why everything but the
// 64 KB table and the probabilities shares one LDS region, and why the rotation comes in operand order from a copy the engine
// keeps (rot_ops) instead of through an LDS tile.
//
// A unit's start and end were a third of the time of short contexts: arguments in one trip, loads without branches, K, V and q
// rotated on fp16 matrix instructions (codes from the fp32 chain where the sums leave a doubt), the parts merged behind one
// barrier, and no launch of its own to advance the positions.  28 layers of 4 x 613 tokens: 985 us a pass of 32 steps before, 697 to 714 now.
// MI355X, us per layer, layer by layer -> all at once (16 heads over 8 KV heads, 28 layers, 4 bit unless said), before those steps: 4 x 613
// tokens 13.8 -> 1.1 (now 0.8); 128 x 513 20.8 -> 13.8 (12.6); 64 x 8192 94.0 -> 83.2 (83 to 89 by the box, 6.2 to 6.7 TB/s); 2 bit 70.6 -> 61.1 (61 to 65);
// 64 ragged 512..8072 75 -> 61; 32 heads, 36 layers, 2 bit, 16 x 4097 23.8 -> 10.3 (9.6).  Over 500 random steps (2 to 36 layers, 1 to 192 sequences of 64 to 16000 tokens, even and
// ragged, both widths) 3.3 times faster in the geometric mean, the slowest 0.97.  Long contexts are bound by the streaming of the
// cache, short ones by the units' start and end.  One workgroup of eight waves per compute unit with kv_decode_fused.hip's LDS layout
// and all layers in its grid: 16.7 for 128 x 513, 85.1 for 64 x 8192, 6.4 against 5.2 at 36 layers of 12 x 2000 and 32 heads.  A table of
// 32 replicas (half the LDS): 3 to 6 % slower, two lanes to a bank.
#include <algorithm>
#include <cmath>

#include "kv_common.hpp"
#include "kv_kernels.hpp"
#include "kv_mfma_util.hpp"
#include "kv_pair_scan.hpp"
#include "kv_producer_util.hpp"
#include "kv_rotate_util.hpp"

namespace twkv {

namespace {
constexpr int kUnitRowFloats = kHeadDim + 4;          // LDS row of a vector: conflict-free 16-byte accesses
constexpr int kUnitVecs = 16;                         // vectors in LDS at a time; also the most query heads of a unit
}  // namespace

template <int R, int BITS, int HKW, int NW, bool PROD>
__global__ void __launch_bounds__(NW * kWave) __attribute__((amdgpu_waves_per_eu(2, 2)))
decode_layers_kernel(LayersArgs a) {
    constexpr uint32_t kHeadBytes = BITS * 16;
    constexpr float kAlpha = BITS == 4 ? kAlpha4 : kAlpha2;
    constexpr int NV = HKW * (2 + R), NQ = HKW * R;              // vectors of a unit: K heads, V heads, query heads
    constexpr int kPasses = (NV + kUnitVecs - 1) / kUnitVecs;    // of 16 vectors, 16 lanes each
    constexpr int kPairs = HKW / 2, kParts = NW / kPairs;
    constexpr int kBlocks = 8 / NW;                              // blocks of 16 output coordinates a wave rotates
    static_assert(NQ <= kUnitVecs && 2 * HKW <= kUnitVecs && kPairs * kParts == NW && kBlocks * NW == 8, "the unit fits its waves and LDS region");
    __shared__ __attribute__((aligned(16))) uint32_t tab_s[kTableWords];
    __shared__ __attribute__((aligned(16))) half_t p_s[NW][16][32];
    // in turn: the new token's vectors, the rotated queries, the parts' sums, the outputs
    __shared__ __attribute__((aligned(16))) float x_s[kUnitVecs][kUnitRowFloats];
    __shared__ __attribute__((aligned(8))) float2 bucket_s[kBuckets];
    __shared__ float inv_s[kUnitVecs];                           // 1 / |vector| of the K and V vectors
    uint4* qop_s = reinterpret_cast<uint4*>(&x_s[0][0]);
    static_assert(NV * 16 * sizeof(uint4) <= sizeof(x_s) && 2 * NQ * 16 * sizeof(uint4) <= sizeof(x_s), "the unit's vectors, and its queries, as halves");

    const int tid = threadIdx.x;
    const int wave = uniform(tid / kWave), lane = tid % kWave;
    const int ln = lane & 15, kg = lane >> 4;
    // the arguments in one trip: fetched where they are first used, the start is five of them one after the other
    asm volatile("" :: "s"(a.q), "s"(a.k), "s"(a.v), "s"(a.positions), "s"(a.rot_ops), "s"(a.q_layer), "s"(a.kv_layer), "s"(a.cache_layer),
                 "s"(a.rotation), "s"(PROD ? a.q_weight : nullptr), "s"(PROD ? a.k_weight : nullptr), "s"(PROD ? a.cos_table : nullptr),
                 "s"(PROD ? a.sin_table : nullptr), "s"(PROD ? a.rope_dim : 0), "s"(a.layers), "s"(a.G), "s"(a.nhg), "s"(a.g_magic), "s"(a.num_kv_heads), "s"(a.q_stride), "s"(a.kv_stride), "s"(a.seq_stride_rows));
    const int Hk = a.num_kv_heads;

    // ---- the unit: (layer, sequence) pairs in one row, eight of them side by side on the XCDs (workgroups are dealt to
    // those in turn), the units of a pair one after the other on its XCD: they share cache lines of codes and norms
    const int nhg = a.nhg;
    const int j8 = (int)blockIdx.x >> 3, group = (nhg & (nhg - 1)) == 0 ? j8 >> __builtin_ctz(nhg) : j8 / nhg;
    const int at = group * 8 + ((int)blockIdx.x & 7);
    if (at >= a.layers * a.G) return;
    const int hg = j8 - group * nhg, layer = a.g_magic ? (int)__umulhi((unsigned)at, a.g_magic) : at / a.G, g = at - layer * a.G;
    const half_t* q = a.q + layer * a.q_layer + (long long)g * a.q_stride + (long long)hg * NQ * kHeadDim;
    const long long kv_at = layer * a.kv_layer + (long long)g * a.kv_stride + (long long)hg * HKW * kHeadDim;
    const half_t *k_src = a.k + kv_at, *v_src = a.v + kv_at;
    const long long cache_at = layer * a.cache_layer;
    const long long row0 = (long long)g * a.seq_stride_rows;

    // ---- requests that do not depend on the position
    const int pos_request = a.positions[g];
    uint4 stage[kPasses], prod_w[kPasses] = {};
    const half_t* q_weight = PROD && a.q_weight ? a.q_weight + layer * kHeadDim : a.rotation;
    const half_t* k_weight = PROD && a.q_weight ? a.k_weight + layer * kHeadDim : a.rotation;
    const int piece = tid & 15;
    auto vec_kind = [&](int vc) -> int { return vc < HKW ? 0 : vc < 2 * HKW ? 1 : 2; };
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
        // (threads without a vector repeat one, and producers that are not there read the rotation: a load in a branch is waited for at
        // the branch's end, and these waits one after the other were 4 us of a unit's start)
        const int vc = min(kUnitVecs * p + ((tid >> 4) & (kUnitVecs - 1)), NV - 1), kind = vec_kind(vc);
        const half_t* src = kind == 2 ? q + (vc - 2 * HKW) * kHeadDim : (kind == 0 ? k_src : v_src) + (vc - kind * HKW) * kHeadDim;
        stage[p] = reinterpret_cast<const uint4*>(src)[piece];
        if (PROD) prod_w[p] = reinterpret_cast<const uint4*>((kind == 0 ? k_weight : q_weight))[piece];
    }
    // A operands of the rotation, dblk = wave and wave + NW: R[16 dblk + ln][4s + kg], s = 8j .. 8j + 7
    uint4 rraw[kBlocks][4];
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) rraw[i][j] = a.rot_ops[((wave + NW * i) * 4 + j) * kWave + lane];

    // ---- table and bucket table while the loads are under way
    {   // as kv_decode_fused.hip: a thread's entries share their low four bits, a wave's their upper four
        constexpr int kStep = NW * kWave * 4, kRounds = kTableWords / kStep;
        const float cent_lane = kAlpha * centroid_of<BITS>(lane);
        const int e0 = tid >> 4, hi0 = uniform(tid >> 8);
        auto cent_of = [&](int c) -> float {                // c uniform over the wave
            return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cent_lane), c));
        };
        if constexpr (BITS == 4) {
            const half_t lo = (half_t)__shfl(cent_lane, e0 & 15, 64);
#pragma unroll
            for (int k = 0; k < kRounds; k++) {
                half2_t p = {lo, (half_t)cent_of(hi0 + (NW / 4) * k)};
                const uint32_t w = *reinterpret_cast<uint32_t*>(&p);
                *reinterpret_cast<uint4*>(&tab_s[tid * 4 + k * kStep]) = uint4{w, w, w, w};
            }
        } else {
            const half_t c0 = (half_t)__shfl(cent_lane, e0 & 3, 64), c1 = (half_t)__shfl(cent_lane, (e0 >> 2) & 3, 64);
#pragma unroll
            for (int k = 0; k < kRounds; k++) {
                const int hi = hi0 + (NW / 4) * k;          // e >> 4
                half2_t p0 = {c0, c1}, p1 = {(half_t)cent_of(hi & 3), (half_t)cent_of(hi >> 2)};
                const uint32_t w0 = *reinterpret_cast<uint32_t*>(&p0), w1 = *reinterpret_cast<uint32_t*>(&p1);
                *reinterpret_cast<uint4*>(&tab_s[tid * 4 + k * kStep]) = uint4{w0, w1, w0, w1};
            }
        }
    }
    if (BITS == 4 && wave == NW - 1 && lane < kBuckets) bucket_s[lane] = bucket_entry(lane);

    const int pos = uniform(pos_request);
    const int n = pos + 1;
    uint4 prod_c = {0u, 0u, 0u, 0u}, prod_s = {0u, 0u, 0u, 0u};              // the same for every vector a thread carries
    if (PROD) {
        const long long at = a.cos_table ? (long long)pos * (a.rope_dim >> 4) + rope_piece16(piece, a.rope_dim) : 0;
        prod_c = reinterpret_cast<const uint4*>(a.cos_table ? a.cos_table : a.rotation)[at];
        prod_s = reinterpret_cast<const uint4*>(a.cos_table ? a.sin_table : a.rotation)[at];
    }

    // ---- the wave's tiles: part p of a pair takes tiles p, p + kParts, ...
    const int pair = wave % kPairs, part = wave / kPairs;
    const int hk_local = 2 * pair;
    const int ntile_seq = (n + 31) >> 5;
    const int ntiles = ntile_seq > part ? (ntile_seq - part + kParts - 1) / kParts : 0;
    int l2 = lane;
    asm volatile("" : "+v"(l2));
    PairLane<R, BITS> L;
    L.init(l2, p_s[wave], tab_s);
    const uint32_t kvp = (uint32_t)Hk * kHeadBytes, nrow = (uint32_t)Hk * 2u;
    const uint32_t koff = L.koff_rows * kvp + L.koff_bytes, voff = L.voff_rows * kvp + L.voff_bytes, noff = (uint32_t)L.tok0 * nrow;
    const int h = hg * HKW + hk_local;
    const char* kpair = reinterpret_cast<const char*>(a.k_codes) + cache_at + row0 * kvp + (long long)h * kHeadBytes;
    const char* vpair = reinterpret_cast<const char*>(a.v_codes) + cache_at + row0 * kvp + (long long)h * kHeadBytes;
    const char* knpair = reinterpret_cast<const char*>(a.k_norms) + cache_at + row0 * nrow + (long long)h * 2;
    const char* vnpair = reinterpret_cast<const char*>(a.v_norms) + cache_at + row0 * nrow + (long long)h * 2;
    int next_tile = 0, next_rows = 0;
    auto set_next = [&](int i) {
        next_tile = 32 * (i * kParts + part);
        next_rows = i < ntiles ? max(min(n - next_tile, 32), 0) : 0;
    };
    constexpr int kCodesAux = BITS == 4 ? kStreamCodes : 0;
    auto issue_k = [&](PairTileRegs<BITS>& t) {
        __amdgpu_buffer_rsrc_t r = make_rsrc(kpair + (long long)next_tile * kvp, next_rows * (int)kvp);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if constexpr (BITS == 4) t.k[c] = __builtin_amdgcn_raw_buffer_load_b128(r, (int)(koff + (uint32_t)(8 * c) * kvp), 0, kCodesAux);
            else t.k[c] = __builtin_amdgcn_raw_buffer_load_b64(r, (int)(koff + (uint32_t)(8 * c) * kvp), 0, kCodesAux);
        }
    };
    auto issue_v = [&](PairTileRegs<BITS>& t) {
        __amdgpu_buffer_rsrc_t r = make_rsrc(vpair + (long long)next_tile * kvp, next_rows * (int)kvp);
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (BITS == 4) t.v[sub][j] = __builtin_amdgcn_raw_buffer_load_b64(r, (int)(voff + (uint32_t)(16 * sub + j) * kvp), 0, kCodesAux);
                else t.v[sub][j] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(voff + (uint32_t)(16 * sub + j) * kvp), 0, kCodesAux);
            }
        }
    };
    auto issue_n = [&](PairTileRegs<BITS>& t) {
        __amdgpu_buffer_rsrc_t rk = make_rsrc(knpair + (long long)next_tile * nrow, next_rows * (int)nrow);
        __amdgpu_buffer_rsrc_t rv = make_rsrc(vnpair + (long long)next_tile * nrow, next_rows * (int)nrow);
        t.n[0][0] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)noff, 0, kStreamNorms);
        t.n[1][0] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)(noff + 16u * nrow), 0, kStreamNorms);
        t.n[0][1] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)noff, 0, kStreamNorms);
        t.n[1][1] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)(noff + 16u * nrow), 0, kStreamNorms);
    };

    // ---- the new token's vectors into LDS, 16 lanes to one, as the halves they are, regrouped for the matrix cores: coordinate 4s + kk of
    // vector v in 16-byte piece 4kk + s / 8 of its row, which lies at that piece ^ 5v (no bank twice, written or read)
    PairTileRegs<BITS> t;
    uint4 (*x_h)[16] = reinterpret_cast<uint4 (*)[16]>(&x_s[0][0]);
    auto piece_of = [&](int v, int p) -> int { return (p ^ (5 * v)) & 15; };
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
        const int vc = kUnitVecs * p + (tid >> 4), kind = vec_kind(vc);
        if (vc < NV && tid < kUnitVecs * 16) {             // the same for the 16 lanes of a vector
            float x[8], sq[8];
            unpack_halves(stage[p], x);
            if (PROD && kind != 1) {
                if (a.q_weight) norm_head16(x, prod_w[p], a.eps, a.biased);
                if (a.cos_table) rope_head16(x, prod_c, prod_s, piece, a.rope_dim, 0);
            }
            const uint4 w = PROD ? pack_halves(x) : stage[p];          // coordinates 8 piece .. 8 piece + 7
            const uint32_t by_kk[4] = {(w.x & 0xffffu) | (w.z << 16), (w.x >> 16) | (w.z & 0xffff0000u),
                                       (w.y & 0xffffu) | (w.w << 16), (w.y >> 16) | (w.w & 0xffff0000u)};
#pragma unroll
            for (int kk = 0; kk < 4; kk++)
                reinterpret_cast<uint32_t*>(&x_h[vc][piece_of(vc, 4 * kk + (piece >> 2))])[piece & 3] = by_kk[kk];
            if (kind != 2) {
#pragma unroll
                for (int e = 0; e < 8; e++) sq[e] = x[e] * x[e];       // exact: fp16 values
                const float norm = sqrtf(head_tree_sum16(sq) + 1e-12f);
                if (piece == 0) {
                    inv_s[vc] = 1.0f / norm;
                    half_t* norms = reinterpret_cast<half_t*>(reinterpret_cast<char*>(kind == 0 ? a.k_norms : a.v_norms) + cache_at);
                    norms[(row0 + pos) * Hk + hg * HKW + vc - kind * HKW] = (half_t)norm;
                }
            }
        }
    }
    lds_barrier();
    // the first tile, when all of its rows are older than the token this launch appends (whose own row is only there after the
    // barrier that ends the rotations)
    const bool first_early = ntiles > 0 && 32 * part + 32 <= pos;
    set_next(0);
    if (!first_early) next_rows = 0;         // (asked for without a branch: behind one, the rotation's operands would be waited for with the tile)
    issue_k(t); issue_n(t); issue_v(t);
    // ---- rotation of all of them on fp16 matrix instructions: fp16 values times an fp16 matrix, every product exact in the fp32
    // accumulator, 4 matrix instructions a block and 16 vectors
    float4_t y[kPasses][kBlocks], sums[kBlocks][4];         // sums: after each operand of the first 16 vectors
#pragma unroll
    for (int p = 0; p < kPasses; p++) {
        const int v = kUnitVecs * p + ln < NV ? kUnitVecs * p + ln : 0;
#pragma unroll
        for (int i = 0; i < kBlocks; i++) y[p][i] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            union { uint4 u; half8_t h; } xv, rv;
            xv.u = x_h[v][piece_of(v, 4 * kg + j)];
#pragma unroll
            for (int i = 0; i < kBlocks; i++) {
                rv.u = rraw[i][j];
                y[p][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(rv.h, xv.h, y[p][i], 0, 0, 0);
                if (p == 0) sums[i][j] = y[p][i];
            }
        }
    }
    {   // Codes of K and V.  They are those of the fp32 chain of kv_rotate.hip, which is 32 matrix instructions of twice the length a
        // block; the sums above decide every coordinate that is further from a boundary than the two can be apart (kv_rotate_util.hpp), and
        // a block with one that is not (one in 17 with 16 vectors, one in 66 with 4) runs the chain.
        const int v = ln, vk = vec_kind(v);                // this lane's vector
        const bool live = v < 2 * HKW;
        const float inv = inv_s[live ? v : 0];
#pragma unroll
        for (int i = 0; i < kBlocks; i++) {                  // lane: coordinates 16 dblk + 4 kg .. + 3 of vector v
            uint32_t packed = 0;
            bool doubt = false;
#pragma unroll
            for (int r = 0; r < 4; r++) packed |= bucket_quantize_sure<BITS>(bucket_s, sums[i], r, inv, kUnitRows, doubt) << (r * BITS);
            if (__any(live && doubt)) {
                float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s8 = 0; s8 < 4; s8++) {
                    float rv[8], uv[8];
                    unpack_halves(rraw[i][s8], rv);
                    unpack_halves(x_h[live ? v : 0][piece_of(live ? v : 0, 4 * kg + s8)], uv);
#pragma unroll
                    for (int e = 0; e < 8; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[e], uv[e] * inv, acc, 0, 0, 0);
                }
                packed = 0;
#pragma unroll
                for (int r = 0; r < 4; r++) packed |= bucket_quantize<BITS>(bucket_s, acc[r]) << (r * BITS);
            }
            if (live) {
                uint8_t* dst = (vk == 0 ? a.k_codes : a.v_codes) + cache_at + ((row0 + pos) * Hk + hg * HKW + v - vk * HKW) * kHeadBytes +
                               (4 * (wave + NW * i) + kg) * (BITS / 2);
                if (BITS == 4) *reinterpret_cast<uint16_t*>(dst) = (uint16_t)packed;
                else *dst = (uint8_t)packed;
            }
        }
    }
    lds_barrier();                                           // the vectors have been read
#pragma unroll
    for (int p = 0; p < kPasses; p++) {                      // the rotated queries, scaled
        const int v = kUnitVecs * p + ln - 2 * HKW;
        if (v >= 0 && v < NQ) {
#pragma unroll
            for (int i = 0; i < kBlocks; i++) store_query_operand(qop_s, v, wave + NW * i, kg, y[p][i], a.q_scale);
        }
    }
    *reinterpret_cast<uint4*>(&p_s[wave][0][0] + 8 * lane) = uint4{0u, 0u, 0u, 0u};       // the wave's probabilities start at zero
    __syncthreads();                                         // table, queries and the new row are in place
    if (!first_early) { set_next(0); issue_k(t); issue_n(t); issue_v(t); }
    // ---- B operands of the rotate-back: R[32 kg + s][16 dblk + ln] (behind the first tile's loads: the registers are there)
    uint4 rb[kBlocks][4];
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) rb[i][j] = a.rot_ops[2048 + ((wave + NW * i) * 4 + j) * kWave + lane];
    PairState<R> S;
    S.reset();
    S.load_query_operands(L, [&](int i, int part2, int p) { return &qop_s[query_piece(2 * (hk_local * R + i) + part2, p)]; });
    S.zero_repeated_queries(L);
    lds_barrier();                                           // the queries have been read
    // The step's last act, positions + 1 (engine.cpp:2394): every wave of this unit has used its sequence's position by now, and the unit
    // that draws a sequence's last ticket is behind all others in that, so it writes the next one.
    // (Every thread asks, all but the first out of range: drawn in a branch, the ticket is waited for at the branch's end.)
    const unsigned ticket = (unsigned)__builtin_amdgcn_raw_ptr_buffer_atomic_add_i32(
        1, make_rsrc(reinterpret_cast<const char*>(a.tickets + g), 4), tid == 0 ? 0 : 1 << 30, 0, kDeviceScope);
    for (int it = 0; it < ntiles; it++) {
        const int tile = next_tile;
        set_next(it + 1);
        pair_scan_tile<R>(L, S, t, tile, n, [&]() { issue_k(t); }, [&]() { issue_n(t); }, [&]() { issue_v(t); });
    }

    // ---- the parts meet in LDS: every wave leaves its sums, then 32 threads to an output merge them (in halves, the upper handed to the lower
    // until one is left, with two barriers each: 0.5 us of a unit's end)
    constexpr bool kInPlace = NW * 2 * R <= kUnitVecs;        // else where the table was, once every wave is through with it
    float (*sum_s)[kUnitRowFloats] = kInPlace ? x_s : reinterpret_cast<float (*)[kUnitRowFloats]>(tab_s);
    if (kParts > 1 && !kInPlace) lds_barrier();
    pair_scan_finish<R>(L, S, 1.0f / kAlpha, [&](int, int r, const float (&o)[16]) {     // dims 16 (pn % 8) .. of head hd
        float* row = kParts > 1 ? sum_s[(part * kPairs + pair) * 2 * R + L.hd * R + r] : x_s[pair * 2 * R + L.hd * R + r];
        const float inv = kParts > 1 ? 1.0f : kLowScale / (S.l_run[r] + 1e-8f);          // kernels.cu:1746, as split_scaled wants it
#pragma unroll
        for (int j4 = 0; j4 < 4; j4++)
            *reinterpret_cast<float4*>(row + 16 * (L.pn & 7) + 4 * j4) = float4{o[4 * j4] * inv, o[4 * j4 + 1] * inv, o[4 * j4 + 2] * inv, o[4 * j4 + 3] * inv};
        if (kParts > 1 && (L.pn & 7) == 0) *reinterpret_cast<float2*>(row + kHeadDim) = float2{S.m_run[r], S.l_run[r]};
    });
    lds_barrier();
    if constexpr (kParts > 1) {
        for (int v = tid >> 5; v < NQ; v += NW * kWave / 32) {                           // output: heads of the pairs, then query heads
            const int k4 = (tid & 31) * 4;
            float2 ml[kParts];
            float4 c[kParts];
            float m = kNegBig, l = 0.0f;
#pragma unroll
            for (int p = 0; p < kParts; p++) {
                const float* row = sum_s[p * kPairs * 2 * R + v];
                ml[p] = *reinterpret_cast<const float2*>(row + kHeadDim);
                c[p] = *reinterpret_cast<const float4*>(row + k4);
                m = fmaxf(m, ml[p].x);
            }
            float4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < kParts; p++) {
                const float fs = __builtin_amdgcn_exp2f(ml[p].x - m);
                l = __builtin_fmaf(ml[p].y, fs, l);
                o.x = __builtin_fmaf(c[p].x, fs, o.x); o.y = __builtin_fmaf(c[p].y, fs, o.y);
                o.z = __builtin_fmaf(c[p].z, fs, o.z); o.w = __builtin_fmaf(c[p].w, fs, o.w);
            }
            const float inv = kLowScale / (l + 1e-8f);       // kernels.cu:1746
            *reinterpret_cast<float4*>(&x_s[v][k4]) = float4{o.x * inv, o.y * inv, o.z * inv, o.w * inv};
        }
        lds_barrier();
    }

    // ---- rotate back (as kv_decode_fused.hip): o as fp16 value + enlarged remainder, R exact in fp16
    half_t* out = a.out + layer * a.q_layer + (long long)g * a.q_stride + (long long)hg * NQ * kHeadDim;
    half8_t ahi[4], alo[4];
    const float* orow = &x_s[ln < NQ ? ln : 0][32 * kg];
#pragma unroll
    for (int st = 0; st < 4; st++) {
        const float4 oa = *reinterpret_cast<const float4*>(orow + 8 * st), ob = *reinterpret_cast<const float4*>(orow + 8 * st + 4);
        const float o8[8] = {oa.x, oa.y, oa.z, oa.w, ob.x, ob.y, ob.z, ob.w};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            half_t hi, lo;
            split_scaled(o8[i], hi, lo);
            ahi[st][i] = hi; alo[st][i] = lo;
        }
    }
#pragma unroll
    for (int i = 0; i < kBlocks; i++) {
        float4_t acc = {0.f, 0.f, 0.f, 0.f}, low = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 4; st++) {
            union { uint4 u; half8_t h; } bm;
            bm.u = rb[i][st];
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[st], bm.h, acc, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[st], bm.h, low, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {                        // out[vector 4 kg + r][16 dblk + ln]
            const int vec = 4 * kg + r;
            if (vec < NQ) out[(long long)vec * kHeadDim + 16 * (wave + NW * i) + ln] = (half_t)__builtin_fmaf(low[r], 1.0f / kLowScale, acc[r]);
        }
    }
    if (tid == 0 && ticket == (unsigned)(a.layers * nhg) - 1u) {
        a.positions[g] = n;
        a.tickets[g] = 0u;                                   // for the next launch
    }
}

// The rotation's 128 x 128 halves in operand order: 8 KB-pieces ((dblk * 4 + j) * 64 + lane) of eight halves, first R[16 dblk +
// lane % 16][4 s + lane / 16], then R[32 (lane / 16) + s][16 dblk + lane % 16], s = 8 j .. 8 j + 7.
void order_rotation(const uint16_t* rot, uint16_t* ops) {
    for (int dblk = 0; dblk < 8; dblk++)
        for (int lane = 0; lane < kWave; lane++)
            for (int s = 0; s < 32; s++) {
                const int ln = lane & 15, kg = lane >> 4, at = ((dblk * 4 + s / 8) * kWave + lane) * 8 + s % 8;
                ops[at] = rot[(16 * dblk + ln) * kHeadDim + 4 * s + kg];
                ops[kHeadDim * kHeadDim + at] = rot[(32 * kg + s) * kHeadDim + 16 * dblk + ln];
            }
}

// Microseconds of the launch: rounds of workgroups as decode_fused_estimate_us counts them, with the cube-root sum taken over the
// whole launch (units end and start at different times), and no shorter than the longest sequence's unit.  Fitted on MI355X to all
// shapes at 1500 random steps of 4 to 36 layers, 1 to 192 sequences of 64 to 12000 tokens, even, ragged and with one long sequence:
// the choice is the fastest shape or within 3 % of it at 93 %, within 10 % at 98 %.
static double decode_layers_estimate_us(int layers, int G, int R, int Hk, int bits, int hkw, int waves, double ctx_max, double ctx_mean) {
    const PlanConstants& pc = plan_constants();
    const double cus = compute_units();
    const int w = bits == 4 ? 0 : 1, r = R >= 4 ? 2 : R >= 2 ? 1 : 0;
    const int parts = waves / (hkw / 2), per_cu = waves == 4 ? 2 : 1;
    const double units = (double)layers * G * (Hk / hkw);
    const double fixed = pc.layers_unit_us[per_cu == 2 ? 0 : 1] + pc.layers_vector_us * hkw * (2 + R);
    const double mean = fixed + std::ceil(ctx_mean / 32.0 / parts) * pc.layers_tile_us[w][r];
    double longest = fixed + std::ceil(ctx_max / 32.0 / parts) * pc.layers_tile_us[w][r];
    // rounds of per_cu workgroups a compute unit; a workgroup of the last round that shares its unit with none is faster
    const double full = std::floor(units / (per_cu * cus)), rest = units - full * per_cu * cus;
    double last = rest > 0.0 ? 1.0 : 0.0;
    if (per_cu == 2 && rest > 0.0) {
        last = rest <= cus ? pc.layers_alone : pc.layers_alone + (1.0 - pc.layers_alone) * (rest - cus) / cus;
        if (units <= cus) longest *= pc.layers_alone;
    }
    const double work = mean * (full + last);
    const double mem = (double)layers * G * ctx_mean * Hk * (bits == 4 ? 132.0 : 68.0) / pc.layers_bw[w][hkw == 2 ? 0 : hkw == 4 ? 1 : 2];
    const double body = std::cbrt(work * work * work + mem * mem * mem);
    return pc.layers_launch_us + std::max(longest, body) + pc.layers_both * std::min(longest, body);
}

LayersShape decode_layers_shape(int layers, int G, int num_heads, int Hk, int bits, double ctx_max, double ctx_mean) {
    const int R = Hk > 0 ? num_heads / Hk : 0;
    const int forced = decode_fused_forced_hkw();
    LayersShape best{0, 0, 0.0};
    if ((R != 1 && R != 2 && R != 4) || (bits != 4 && bits != 2)) return best;
    constexpr int kShapes[4][2] = {{2, 4}, {4, 4}, {8, 4}, {2, 8}};          // KV heads, waves
    for (const auto& c : kShapes) {
        if (Hk % c[0] != 0 || R * c[0] > kUnitVecs || (forced > 0 && c[0] != forced)) continue;
        const double us = decode_layers_estimate_us(layers, G, R, Hk, bits, c[0], c[1], ctx_max, ctx_mean);
        if (best.hkw == 0 || us < best.us) best = LayersShape{c[0], c[1], us};
    }
    return best;
}

void launch_decode_layers(const LayersArgs& args, int num_heads, int bits, int hkw, int waves, hipStream_t s) {
    LayersArgs a = args;
    a.nhg = a.num_kv_heads / hkw;
    const uint64_t G = (uint64_t)a.G, two32 = 1ull << 32;
    a.g_magic = G > 1 && ((uint64_t)a.layers * G + 8) * G < two32 ? (uint32_t)((two32 + G - 1) / G) : 0u;
    const int R = num_heads / a.num_kv_heads;
    const long long pairs = ((long long)a.layers * a.G + 7) / 8 * 8;
    const dim3 g3((unsigned)(pairs * (a.num_kv_heads / hkw))), b3(waves * kWave);
    note_scan_kernel(hkw == 8 ? "decode_layers_kernel, eight KV heads in four waves" : hkw == 4 ? "decode_layers_kernel, four KV heads in four waves"
                     : waves == 4 ? "decode_layers_kernel, two KV heads in four waves" : "decode_layers_kernel, two KV heads in eight waves");
    const bool prod = a.q_weight != nullptr || a.cos_table != nullptr;
#define TW_L(RR, BB, HH, WW) do { if (prod) launch_scan_kernel(decode_layers_kernel<RR, BB, HH, WW, true>, g3, b3, s, a); \
                                  else launch_scan_kernel(decode_layers_kernel<RR, BB, HH, WW, false>, g3, b3, s, a); } while (0)
#define TW_LB(RR, HH, WW) do { if (bits == 4) TW_L(RR, 4, HH, WW); else TW_L(RR, 2, HH, WW); } while (0)
#define TW_L2(RR) do { if (waves == 4) TW_LB(RR, 2, 4); else TW_LB(RR, 2, 8); } while (0)
    if (R == 1) { if (hkw == 8) TW_LB(1, 8, 4); else if (hkw == 4) TW_LB(1, 4, 4); else TW_L2(1); }
    else if (R == 2) { if (hkw == 8) TW_LB(2, 8, 4); else if (hkw == 4) TW_LB(2, 4, 4); else TW_L2(2); }
    else { if (hkw == 4) TW_LB(4, 4, 4); else TW_L2(4); }
#undef TW_L2
#undef TW_LB
#undef TW_L
}

}  // namespace twkv
