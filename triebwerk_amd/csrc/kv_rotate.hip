// kv_rotate.hip -- the 128x128 rotation on the matrix cores (gfx950), for
//   - the TurboQuant compressed append: y = R (x / |x|), bin search, pack, norm
//     (turbo_kv_quantize{,_batch}_kernel, kernels.cu:1482-1636), K and V rows, and
//   - the query rotation q_rot = R q of the compressed attention (kernels.cu:1671-1681),
// all in one launch (any subset); optionally with the producers of q and k applied on the way in
// (per-head RMSNorm and rotary embedding, kernels.cu:880-961), which saves their two launches and
// the round trip of the rows through memory.
//
// Bit-exactness of the append.  The reference accumulates each output coordinate as
// one fp32 fused-multiply-add chain over k = 0..127.  v_mfma_f32_16x16x4_f32 chained
// over k-blocks of 4 produces the same bits: inside one instruction the four k of the
// block are accumulated in ascending order with fused multiply-adds, and blocks chain
// through the accumulator (checked on hardware against a host fmaf chain: 0 of 4096
// outputs differ).  The sum of squares keeps the reference's reduction tree
// (kernels.cu:1509-1520): offsets 16, 8 and 4 of the 32-lane shuffle tree only combine
// coordinates that are congruent mod 4, which one lane owns; offsets 2 and 1 and the
// combination of the four 32-coordinate groups, (s0+s2)+(s1+s3), are done across lanes.
//
// Mapping.  One wave = one work unit = (16 vectors) x (16 output coordinates):
//   A operand = R rows   : lane (i = lane%16, kk = lane/16) holds R[d0+i][4s+kk], s = 0..31
//   B operand = vectors  : the same lane holds u[v0+i][4s+kk]
//   D[16 x 16]           : lane holds y[d0 + 4*(lane/16) + r][v0 + lane%16], r = 0..3
// A wave needs nothing from any other wave, so a launch is ceil(vectors/16) * 8 independent single-wave
// workgroups that spread over the chip; that matters because the launches of a decode step are small (a few
// thousand vectors) and latency-bound.  The 8 waves that share a tile of vectors are numbered so that they land
// on one XCD (workgroup b runs on XCD b % 8), whose L2 then serves 7 of their 8 reads of it.
//
// Operand loads.  In the MFMA layout a lane wants every fourth half of a 256-byte row, and 16 lanes want 16
// different rows: asked for directly that is 16 loads per lane of which a quarter is used, each touching 16
// cache lines, and the address path of the CU becomes the limit of a big launch.  So a tile (16 rows, 4 KB)
// comes in as 4 fully used 16-byte pieces per lane, is written to LDS with the halves regrouped
// ([kk][row][s], kv_rotate_util.hpp), and each lane reads back its 32 halves as 4 x 16 bytes.

//
// What bounds both launches of a step is the chain of trips to memory and the issue of one wave (a launch is few waves a SIMD).
// So the arguments come in one trip (an asm statement that wants them all), positions, rows and R are asked for before any is waited
// for, the buckets are a table of pairs instead of a search, queries for attention_pair_kernel leave as the operands of
// its matrix instructions, and the merge asks for as many slots as there can be before it knows their number and rotates back on
// fp16 matrix instructions (value + remainder).  With the scan's own start: 8 layers of the launchers' step, 47 ragged sequences at
// 2 bit, 397 -> 346 us; the paged step of 64 ragged sequences 580 -> 539.

#include <algorithm>
#include <type_traits>

#include "kv_common.hpp"
#include "kv_kernels.hpp"
#include "kv_mfma_util.hpp"
#include "kv_rotate_util.hpp"

namespace twkv {

namespace {

// Rotary embedding of a vector held as xv[s] = coordinate 4s + kk: coordinate d < HALF pairs with d + HALF
// (same lane, HALF4 = HALF / 4 registers further on); fp16 rounding as in rope_batch_kernel
// (kernels.cu:927-961).  The table rows hold HALF entries and arrive as 16-byte pieces.
template <int HALF4>
__device__ __forceinline__ void rope_registers(float (&xv)[32], const uint4 (&cp)[8], const uint4 (&sp)[8], int kk) {
#pragma clang fp contract(off)      // products rounded to fp32 first, as rope_batch_kernel's are
#pragma unroll
    for (int s = 0; s < HALF4; s++) {
        const float c = pick_half(cp[s >> 1], s & 1, kk), sn = pick_half(sp[s >> 1], s & 1, kk);
        const float x0 = xv[s], x1 = xv[s + HALF4];
        xv[s] = as_half_value(__builtin_fmaf(x0, c, -(x1 * sn)));
        xv[s + HALF4] = as_half_value(__builtin_fmaf(x0, sn, x1 * c));
    }
}

}  // namespace

// PROD: the producers of q and k may be switched on (their operands cost 64 registers and a third of the
// occupancy, which only the big launches of a prompt notice).
template <int BITS, bool PROD>
__global__ void __launch_bounds__(kWave)
rotate_kernel(RotArgs a) {
    __shared__ __attribute__((aligned(16))) uint32_t x_s[kOperandTileDwords];
    __shared__ __attribute__((aligned(8))) float2 bucket_s[kBuckets];
    const int lane = threadIdx.x;
    const int i16 = lane & 15, kk = lane >> 4;

    // ---- which unit: (segment, group of a.nper vector tiles, block of 16 output coordinates)
    asm volatile("" :: "s"(a.seg[0].units), "s"(a.seg[1].units), "s"(a.nseg), "s"(a.nper), "s"(a.rotation), "s"(a.positions), "s"(a.block_table),
                 "s"(a.seq_stride_rows), "s"(a.token_list));
    int unit = blockIdx.x;
    const int after0 = unit - a.seg[0].units, after1 = after0 - a.seg[1].units;
    const int seg = a.nseg > 1 && after0 >= 0 ? (a.nseg > 2 && after1 >= 0 ? 2 : 1) : 0;
    unit = seg == 0 ? unit : seg == 1 ? after0 : after1;
    const RotArgs::Segment& sg = a.seg[seg];
    asm volatile("" :: "s"(sg.src), "s"(sg.stride), "s"(sg.heads), "s"(sg.nvec), "s"(sg.kind), "s"(sg.units));
    // Units of a segment in blocks of 64 = 8 tile groups x 8 coordinate blocks, the coordinate blocks of one
    // tile group 8 workgroups apart (same XCD; every segment starts at a multiple of 8); what is left over at the
    // end of the segment is numbered plainly.
    int dblk = unit & 7, vgroup = unit >> 3;
    if (unit < (sg.units >> 6) << 6) {
        vgroup = (unit >> 6) * 8 + (unit & 7);
        dblk = (unit >> 3) & 7;
    }
    const int nvec = sg.nvec;
    const int heads = sg.heads;               // head vectors per source row
    const bool is_query = sg.kind != 0;
    const bool roped = PROD && sg.rope != 0;
    const half_t* weight = PROD ? sg.weight : nullptr;
    uint8_t* codes = sg.codes;
    half_t* norms = sg.norms;
    const bool heads_pow2 = (heads & (heads - 1)) == 0;  // (else a division: twenty instructions)
    const int heads_log2 = __builtin_ctz(heads);
    auto row_of = [&](int v) -> int { return heads_pow2 ? v >> heads_log2 : v / heads; };

    // ---- A operand, once per wave: R rows d0 .. d0 + 15 (4 KB in a row); requested now, staged after the
    // first tile of vectors has been requested too
    uint4 raw[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
        raw[j] = reinterpret_cast<const uint4*>(a.rotation + dblk * 16 * kHeadDim)[j * kWave + lane];

    // 16-byte piece j * 64 + lane of a tile of vectors: piece lane % 16 of vector 4j + lane / 16
    const half_t* src = sg.src;
    const long long stride = sg.stride;
    auto request_tile = [&](int vtile, uint4 (&dst)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int vi = min(vtile * 16 + 4 * j + (lane >> 4), nvec - 1);
            const int ri = row_of(vi), hi = vi - ri * heads;
            dst[j] = reinterpret_cast<const uint4*>(src + (long long)ri * stride + (long long)hi * kHeadDim)[lane & 15];
        }
    };
    const int vtile0 = vgroup * a.nper;
    if (vtile0 * 16 >= nvec) return;
    uint4 xraw[4];
    request_tile(vtile0, xraw);
    // The position of a vector's row: needed for the cache row and for the rotary table row.  Asked for without a branch (at whose end it
    // would be waited for, with all requests before it): where neither is wanted a word of R is read.
    const bool want_pos = !is_query || roped;
    auto request_pos = [&](int vtile) -> int {
        const int row = row_of(min(vtile * 16 + i16, nvec - 1));
        return (want_pos ? a.positions : reinterpret_cast<const int*>(a.rotation))[want_pos ? row : 0];
    };
    int next_pos = request_pos(vtile0);
    if (BITS == 4 && lane < kBuckets) bucket_s[lane] = bucket_entry(lane);

    float rv[32];
    stage_operand_tile(x_s, raw, lane);
    lds_barrier();
    read_operand_tile(x_s, lane, rv);

    // Small launches (decode) give every wave one tile of 16 vectors; large ones (prompts) let a wave keep
    // its rows of R and walk a.nper tiles, the next tile requested while this one is worked on.
    for (int it = 0; it < a.nper; it++) {
    const int vtile = vtile0 + it;
    if (vtile * 16 >= nvec) break;
    const int v = vtile * 16 + i16;
    const int vc = v < nvec ? v : nvec - 1;              // clamp loads, mask stores
    const int row = row_of(vc), head = vc - row * heads;

    // everything that depends on the position is requested before the operands are used
    const int pos_row = next_pos;
    const bool paged = !is_query && !a.token_list && a.block_table != nullptr;
    const int page = (paged ? a.block_table : reinterpret_cast<const int*>(a.rotation))[paged ? (long long)row * a.bt_stride + pos_row / kPageTokens : 0];
    // ---- B operand: the tile's vectors through LDS
    lds_barrier();                                        // the reads of the previous tile (or of R) are done
    stage_operand_tile(x_s, xraw, lane);
    if (it + 1 < a.nper) {                                // clamped to the last vector: never out of bounds
        request_tile(vtile + 1, xraw);
        next_pos = request_pos(vtile + 1);
    }
    lds_barrier();
    float xv[32];
    read_operand_tile(x_s, lane, xv);

    // rotary table row of this position: rope_dim / 2 halves = rope_dim / 16 pieces
    uint4 cpiece[8], spiece[8];
    if (roped) {
        const int pieces = a.rope_dim >> 4;
        const uint4* cr = reinterpret_cast<const uint4*>(a.cos_table + (long long)pos_row * (a.rope_dim >> 1));
        const uint4* sr = reinterpret_cast<const uint4*>(a.sin_table + (long long)pos_row * (a.rope_dim >> 1));
#pragma unroll
        for (int q = 0; q < 8; q++) {
            if (q < pieces) { cpiece[q] = cr[q]; spiece[q] = sr[q]; }
        }
    }

    // ---- optional producers: per-head RMSNorm (kernels.cu:880-923), then rotary embedding (927-961),
    // each rounded to fp16 as the in-place kernels of the reference leave it
    if (PROD && weight) {
#pragma clang fp contract(off)      // (x * rms) * w: two fp32 roundings, then the one to fp16
        const float rms = 1.0f / sqrtf(rotation_tree_sum_sq(xv) / (float)kHeadDim + a.eps);
        const uint4* wsrc = reinterpret_cast<const uint4*>(weight);
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const uint4 wp = wsrc[q];
            float w0 = pick_half(wp, 0, kk), w1 = pick_half(wp, 1, kk);
            if (a.biased) { w0 += 1.0f; w1 += 1.0f; }
            xv[2 * q] = as_half_value((xv[2 * q] * rms) * w0);
            xv[2 * q + 1] = as_half_value((xv[2 * q + 1] * rms) * w1);
        }
    }
    if (roped) {
        switch (a.rope_dim >> 1) {                               // rope_dim: 128, or a multiple of 16 up to 64
            case 64: rope_registers<16>(xv, cpiece, spiece, kk); break;
            case 32: rope_registers<8>(xv, cpiece, spiece, kk); break;
            case 24: rope_registers<6>(xv, cpiece, spiece, kk); break;
            case 16: rope_registers<4>(xv, cpiece, spiece, kk); break;
            default: rope_registers<2>(xv, cpiece, spiece, kk); break;
        }
    }

    float n2 = 0.0f;
    if (!is_query) {
        n2 = rotation_tree_sum_sq(xv);
        const float inv = 1.0f / sqrtf(n2 + 1e-12f);
#pragma unroll
        for (int s = 0; s < 32; s++) xv[s] *= inv;
    }

    // ---- y[d][v] = sum_k R[d][k] u[v][k], k ascending
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 32; s++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[s], xv[s], acc, 0, 0, 0);

    if (is_query) {
        if (v < nvec) {
            float* dst = a.qrot + (long long)v * a.qrot_stride;
            const float o[4] = {acc[0] * a.q_scale, acc[1] * a.q_scale, acc[2] * a.q_scale, acc[3] * a.q_scale};
            if (a.q_operands) {
                half4_t hi, lo;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    hi[r] = (half_t)o[r];
                    lo[r] = (half_t)(o[r] - (float)hi[r]);
                }
                half4_t* ops = reinterpret_cast<half4_t*>(dst) + dblk * 4 + kk;
                ops[0] = hi;
                ops[kHeadDim / 4] = lo;
            } else {
                *reinterpret_cast<float4*>(dst + dblk * 16 + 4 * kk) = float4{o[0], o[1], o[2], o[3]};
            }
        }
        continue;
    }

    // ---- quantize the lane's 4 consecutive coordinates d0 + 4kk .. +3, pack (low field first) and store them
    uint32_t packed = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) packed |= bucket_quantize<BITS>(bucket_s, acc[r]) << (r * BITS);
    if (v < nvec) {
        const long long crow = a.token_list ? pos_row                                   // sequence 0, kernels.cu:1499, 1553
                               : paged ? (long long)page * kPageTokens + pos_row % kPageTokens : (long long)row * a.seq_stride_rows + pos_row;
        constexpr int BPH = kHeadDim * BITS / 8;                  // bytes per head: 64 or 32
        uint8_t* dst = codes + (crow * a.num_kv_heads + head) * BPH + dblk * (2 * BITS) + kk * (BITS / 2);
        if (BITS == 4) *reinterpret_cast<uint16_t*>(dst) = (uint16_t)packed;
        else *dst = (uint8_t)packed;
        if (dblk == 0 && kk == 0) norms[crow * a.num_kv_heads + head] = (half_t)sqrtf(n2 + 1e-12f);
    }
    }   // tiles of this wave
}

void launch_rotate(const RotArgs& args, int bits, hipStream_t s) {
    RotArgs a = args;
    // tiles of 16 vectors per wave: one while the launch is small, more once there are far more tiles than
    // the GPU holds waves
    long long tiles = 0;
    for (int i = 0; i < a.nseg; i++) tiles += (a.seg[i].nvec + 15) / 16;
    constexpr long long kWantUnits = 16384;               // 64 single-wave workgroups per CU
    int nper = (int)((tiles * 8 + kWantUnits - 1) / kWantUnits);
    if (nper < 1) nper = 1;
    if (nper > 32) nper = 32;
    a.nper = nper;
    int units = 0;
    for (int i = 0; i < a.nseg; i++) {
        const int t = (a.seg[i].nvec + 15) / 16;
        a.seg[i].units = (t + nper - 1) / nper * 8;
        units += a.seg[i].units;
    }
    if (units <= 0) return;
    bool prod = false;
    for (int i = 0; i < a.nseg; i++) prod = prod || a.seg[i].weight != nullptr || a.seg[i].rope != 0;
    if (bits == 4) {
        if (prod) hipLaunchKernelGGL((rotate_kernel<4, true>), dim3(units), dim3(kWave), 0, s, a);
        else hipLaunchKernelGGL((rotate_kernel<4, false>), dim3(units), dim3(kWave), 0, s, a);
    } else {
        if (prod) hipLaunchKernelGGL((rotate_kernel<2, true>), dim3(units), dim3(kWave), 0, s, a);
        else hipLaunchKernelGGL((rotate_kernel<2, false>), dim3(units), dim3(kWave), 0, s, a);
    }
}

// The sums that bucket_quantize_sure decides codes from, for a test of its bound: a wave per 16 vectors and 16 coordinates, operands as
// append_tokens_kernel and the one-launch steps hold them (operand j of a lane: coordinates 4s + kk, s = 8j .. 8j + 7).
__global__ void __launch_bounds__(kWave)
rotation_sums_kernel(const half_t* __restrict__ x, int n, const half_t* __restrict__ rotation, float* __restrict__ sums, float* __restrict__ row_norms) {
    const int lane = threadIdx.x, i16 = lane & 15, kk = lane >> 4, dblk = blockIdx.y, v = blockIdx.x * 16 + i16;
    const half_t* row = rotation + (dblk * 16 + i16) * kHeadDim + kk;
    const half_t* vec = x + (long long)min(v, n - 1) * kHeadDim + kk;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    uint4 rows[4];
    for (int j = 0; j < 4; j++) {
        half8_t r, u;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            r[e] = row[4 * (8 * j + e)];
            u[e] = vec[4 * (8 * j + e)];
        }
        rows[j] = __builtin_bit_cast(uint4, r);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(r, u, acc, 0, 0, 0);
    }
    if (v < n) {                                       // lane: coordinates 16 dblk + 4kk .. + 3 of vector v
#pragma unroll
        for (int r = 0; r < 4; r++) sums[(long long)v * kHeadDim + dblk * 16 + 4 * kk + r] = acc[r];
    }
    const float norm = operand_rows_norm(rows);
    if (blockIdx.x == 0 && lane == 0) row_norms[dblk] = norm;
}
void launch_rotation_sums(const half_t* x, int n, const half_t* rotation, float* sums, float* row_norms, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(rotation_sums_kernel, dim3((n + 15) / 16, 8), dim3(kWave), 0, s, x, n, rotation, sums, row_norms);
}

// ---------------------------------------------------------------- split merge + rotate-back
// out[g][head][d] = sum_k R[k][d] * o[k],  o = (sum_c f_c acc_c) / (sum_c f_c l_c + 1e-8),
// f_c = exp(m_c - max_c m_c): the log-sum-exp merge of the split partials, the
// normalisation of kernels.cu:1746 and the rotate-back of kernels.cu:1769-1775.
// A workgroup of 8 waves takes 16 (sequence, head) vectors: all threads merge into LDS,
// then wave w produces output coordinates [16w, 16w+16) with 8 fp16 MFMAs (A = merged vectors from LDS, B = a column block of R).
// R lies in LDS as in memory and a wave's columns of it come out by transposing reads (four rows of 16 halves, four lanes to a row, lane ln
// gets column ln).  The merged vectors enter as fp16 value and enlarged remainder (kLowScale), every product exact in the fp32 accumulators.
constexpr int kMergeVecs = 16;
constexpr int kMergeRow = 2 * kHeadDim + 16;   // bytes per LDS row of merged halves: no bank twice in 16-byte reads
constexpr int kMergeRot = 2 * kHeadDim + 32;   // and of R

__global__ void __launch_bounds__(8 * kWave)
merge_rotate_kernel(AttnArgs a, int nper) {
    __shared__ __attribute__((aligned(16))) char o_s[2][kMergeVecs * kMergeRow];
    __shared__ __attribute__((aligned(16))) char r_s[kHeadDim * kMergeRot];
    asm volatile("" :: "s"(a.rotation), "s"(a.positions), "s"(a.ws), "s"(a.ws_stride), "s"(a.num_heads), "s"(a.G), "s"(a.nsplit), "s"(a.max_slots),
                 "s"(a.pos_mode), "s"(a.pos_scalar), "s"(a.slots_from_ws), "s"(a.m_log2), "s"(nper), "s"(a.out), "s"(a.q_stride));
    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid % kWave;
    const int i16 = lane & 15, kk = lane >> 4;
    const int total = a.G * a.num_heads;
    uint32x4_t rot[4];
#pragma unroll
    for (int r = 0; r < 4; r++) rot[r] = reinterpret_cast<const uint32x4_t*>(a.rotation)[tid + 512 * r];
    const int room = max(a.max_slots, a.nsplit);
    const bool heads_pow2 = (a.num_heads & (a.num_heads - 1)) == 0;
    const int heads_log2 = __builtin_ctz(a.num_heads);
    auto row_of = [&](int v) -> int { return heads_pow2 ? v >> heads_log2 : v / a.num_heads; };

    // A workgroup keeps its block of R and walks nper tiles of 16 vectors (1 in a decode step, more for a prompt).
    for (int it = 0; it < nper; it++) {
    const int v0 = (blockIdx.x * nper + it) * kMergeVecs;
    if (v0 >= total) break;
    if (it > 0) lds_barrier();                        // the previous tile's vectors have been read

    // ---- merge: thread -> (vector tid/32, coordinates 4*(tid%32) .. +3)
    {
        const int vl = tid >> 5, k4 = (tid & 31) * 4;
        const int vv = min(v0 + vl, total - 1);
        const int g = row_of(vv);
        // (both loads without a branch, at whose end they would be waited for: a word of R where there is no array of positions)
        const bool array = a.pos_mode == kPosArray;
        const int pos_read = (array ? a.positions : reinterpret_cast<const int*>(a.rotation))[array ? g : 0];
        const float* part = a.ws + (long long)vv * a.ws_stride;
        const int nseg_read = reinterpret_cast<const int*>(part)[kHeadDim + 2];
        // Slots in blocks with every load of a block issued before the first use, so a block costs one memory
        // latency rather than one per slot; the running maximum is carried across blocks as in an online softmax.
        float mg = -1e30f, lsum = 0.0f;
        float4 av = {0.f, 0.f, 0.f, 0.f};
        int n = 0, nslots = room;
        // (a sequence of at least nsplit tiles has a token in every slot; only shorter ones are asked slot by slot, a division each)
        bool some_empty = false, any_empty = false;
        const float to_log2 = a.m_log2 ? 1.0f : kLog2e;
        auto merge_block = [&](int c0, auto width) {
            constexpr int W = decltype(width)::value;
            float mc[W], lc[W];
            float4 pc4[W];
#pragma unroll
            for (int j = 0; j < W; j++) {
                const int c = c0 + j;
                // (perhaps no workgroup wrote this slot.)  The address does not wait for that answer, which needs the position or the
                // workspace's own count, a load in front of these: every slot the workspace has room for may be read, and what it
                // holds is dropped below.
                const float* pc = part + (long long)(c < room ? c : 0) * kPartialFloats;
                const float2 ml = *reinterpret_cast<const float2*>(pc + kHeadDim);
                mc[j] = ml.x;
                lc[j] = ml.y;
                pc4[j] = *reinterpret_cast<const float4*>(pc + k4);
            }
            if (c0 == 0) {
                n = (array ? pos_read : a.pos_mode == kPosScalar ? a.pos_scalar : g) + 1;
                const int nseg = a.slots_from_ws ? nseg_read : 0;
                nslots = nseg > 0 ? nseg : a.nsplit;
                some_empty = nseg == 0 && ((unsigned)(n + 31) >> 5) < (unsigned)a.nsplit;
                any_empty = __any(some_empty);
            }
            unsigned live = nslots >= c0 + W ? (1u << W) - 1u : nslots > c0 ? (1u << (nslots - c0)) - 1u : 0u;
            if (any_empty) {
#pragma unroll 1
                for (int j = 0; j < W; j++)
                    if (some_empty && c0 + j < nslots && !chunk_nonempty(n, c0 + j, a.nsplit)) live &= ~(1u << j);
            }
#pragma unroll
            for (int j = 0; j < W; j++)
                if (!(live >> j & 1u)) { mc[j] = -1e30f; lc[j] = 0.0f; pc4[j] = float4{0.f, 0.f, 0.f, 0.f}; }
            float mb = mg;
#pragma unroll
            for (int j = 0; j < W; j++) mb = fmaxf(mb, mc[j]);
            const float fo = __builtin_amdgcn_exp2f((mg - mb) * to_log2);
            lsum *= fo; av.x *= fo; av.y *= fo; av.z *= fo; av.w *= fo;
            mg = mb;
#pragma unroll
            for (int j = 0; j < W; j++) {
                float f = __builtin_amdgcn_exp2f((mc[j] - mg) * to_log2);
                lsum = __builtin_fmaf(lc[j], f, lsum);
                av.x = __builtin_fmaf(pc4[j].x, f, av.x);
                av.y = __builtin_fmaf(pc4[j].y, f, av.y);
                av.z = __builtin_fmaf(pc4[j].z, f, av.z);
                av.w = __builtin_fmaf(pc4[j].w, f, av.w);
            }
        };
        // blocks of 8 (the first one before anything is known of the count); room for 1 or 2 (a prompt) is not padded to 8 loads
        if (room <= 2) {
            merge_block(0, std::integral_constant<int, 2>{});
        } else {
            merge_block(0, std::integral_constant<int, 8>{});
            for (int c0 = 8; c0 < nslots; c0 += 8) merge_block(c0, std::integral_constant<int, 8>{});
        }
        const float inv = kLowScale / (lsum + 1e-8f);
        const float o4[4] = {av.x * inv, av.y * inv, av.z * inv, av.w * inv};
        half4_t hi, lo;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            half_t h, l;
            split_scaled(o4[i], h, l);
            hi[i] = h; lo[i] = l;
        }
        *reinterpret_cast<half4_t*>(&o_s[0][vl * kMergeRow + 2 * k4]) = hi;
        *reinterpret_cast<half4_t*>(&o_s[1][vl * kMergeRow + 2 * k4]) = lo;
    }
    if (it == 0) {
#pragma unroll
        for (int r = 0; r < 4; r++) *reinterpret_cast<uint32x4_t*>(&r_s[((tid >> 4) + 32 * r) * kMergeRot + 16 * (tid & 15)]) = rot[r];
    }
    lds_barrier();

    // ---- out[vector][d] = sum_k o[vector][k] R[k][d]; lane group kk owns k = 32 t + 8 kk ..
    float4_t acc = {0.f, 0.f, 0.f, 0.f}, low = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const half8_t hi = *reinterpret_cast<const half8_t*>(&o_s[0][i16 * kMergeRow + 64 * t + 16 * kk]);
        const half8_t lo = *reinterpret_cast<const half8_t*>(&o_s[1][i16 * kMergeRow + 64 * t + 16 * kk]);
        typedef __fp16 __attribute__((ext_vector_type(4))) fp16x4_t;
        typedef __attribute__((address_space(3))) fp16x4_t* lds_fp16x4_t;
        const char* at = &r_s[(32 * t + 8 * kk + (i16 >> 2)) * kMergeRot + 32 * wave + 8 * (i16 & 3)];
        union { fp16x4_t q[2]; half8_t h; } rt;
        rt.q[0] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_fp16x4_t)at);
        rt.q[1] = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_fp16x4_t)(at + 4 * kMergeRot));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, rt.h, acc, 0, 0, 0);
        low = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, rt.h, low, 0, 0, 0);
    }
    // lane holds out[vector 4kk + r][d = 16*wave + i16]
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int vv = v0 + 4 * kk + r;
        if (vv < total) {
            const int g = row_of(vv), head = vv - g * a.num_heads;
            const long long col = (long long)head * kHeadDim + 16 * wave + i16;
            half_t h = (half_t)__builtin_fmaf(low[r], 1.0f / kLowScale, acc[r]);
            if (a.gate) h = gated(h, a.gate[(long long)g * a.gate_stride + col]);
            a.out[(long long)g * a.q_stride + col] = h;
        }
    }
    }   // tiles of this workgroup
}

bool launch_merge_rotate(const AttnArgs& a, hipStream_t s) {
    if (a.bits == 0 || !a.ws) return false;
    if ((reinterpret_cast<uintptr_t>(a.ws) & 15u) != 0 || (a.ws_stride & 3) != 0) return false;
    const int total = a.G * a.num_heads;
    if (total <= 0) return true;
    // one tile per workgroup until there are 8 workgroups per CU, then up to 8
    const int tiles = (total + kMergeVecs - 1) / kMergeVecs;
    const int nper = std::max(1, std::min(8, tiles / 2048));
    hipLaunchKernelGGL(merge_rotate_kernel, dim3((tiles + nper - 1) / nper), dim3(8 * kWave), 0, s, a, nper);
    return true;
}

}  // namespace twkv
