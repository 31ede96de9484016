// kv_decode_fused.hip -- one decode step of one layer over the compressed cache in ONE launch (gfx950):
// append K and V of the new token (turbo_kv_quantize_batch_kernel, kernels.cu:1563-1636), rotate the query
// (1671-1681), scan the context (1688-1766), merge the parts of the context, normalise and rotate back
// (1746, 1769-1775).  forward_layer_batch does this with three launches (engine.cpp:1985-2006) and the
// three-kernel path of this library (rotate_kernel, attention_pair_kernel or attention_mfma_kernel,
// merge_rotate_kernel) does too;
// each of those small launches costs ~4.5 us before it does anything and the scan another ~6 us to start
// and drain, which is a third of a layer at contexts of a few hundred tokens.
//
// A workgroup owns one sequence and HKW of its KV heads (HKW = 1, 2, 4 or 8) together with their query heads, so
// nothing is handed from one workgroup to another.  Two forms: PAIR (HKW even) -- 8 waves, each scanning two KV heads
// with the tile of kv_pair_scan.hpp (256 registers per wave, two waves per SIMD either way); otherwise 16 waves with
// one KV head each, described here:
//   1. all threads fetch the unit's vectors (K heads, V heads, query heads of the new token), 16 lanes to a vector, and
//      fill the centroid table meanwhile; the 16 lanes apply the producers' RMSNorm and rotary embedding
//      (kernels.cu:880-961), measure the vector and leave it in LDS as halves.  Waves 0-7 (all 16 when the unit has more than 16
//      vectors) then rotate them -- lane i16 = vector, wave = block of 16 output coordinates -- on v_mfma_f32_16x16x32_f16; codes
//      come from those sums where their bound of error allows no other, and from rotate_kernel's v_mfma_f32_16x16x4_f32
//      chain otherwise, so they have its bits -- and store the codes in the cache, the scaled q_rot in LDS as the scan's operands;
//   2. after the barrier wave w scans every SPLIT-th tile of the context (SPLIT = 16 / HKW, starting at tile
//      w / HKW) for head w % HKW with the loop of attention_mfma_kernel (the table look-ups, MFMA tiling,
//      online softmax are described there).  All its loads are issued after the barrier: the new token's row
//      was stored by this workgroup (same CU, same L1), which a workgroup-scope barrier makes visible;
//   3. the partial results meet in LDS: merge (log-sum-exp), "+1e-8" normalisation, and R^T on fp16 MFMAs (value +
//      remainder of the normalised output; the output tolerates a different order of additions, the codes did
//      not); output gate as in merge_rotate_kernel.
// The waves in the upper wave slots of a CU run ~5 % slower (see kv_common.hpp: kPairShare), so the parts
// of the upper eight waves get 31/64 of the tiles.
//
// One sequence is one workgroup's work whatever its length: right for batches of similar lengths (a
// rollout's decode steps) and for short contexts; the three-kernel path with its balanced walk stays the
// choice for ragged long contexts, and the only one for the paged layout.
// (Tried at batch 64: workgroups of all 8 KV heads, four per sequence with a quarter of the context each, so that a
// workgroup's waves read whole cache rows side by side -- a plain read of the cache in that pattern runs at 6.8
// instead of 6.4 TB/s -- and the quarters' sums meeting in a workspace, finished by whichever workgroup takes the
// last arrival ticket.  The agent-scope release and acquire fences around that hand-over, each a write-back or an
// invalidation of the XCD's L2, cost 34 us per launch; with no fence at all, which is not correct, the launch took
// 99 us against 97: the scan is not held up by the access pattern.)

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>

#include "kv_common.hpp"
#include "kv_kernels.hpp"
#include "kv_mfma_util.hpp"
#include "kv_pair_scan.hpp"
#include "kv_producer_util.hpp"
#include "kv_rotate_util.hpp"

namespace twkv {

namespace {

constexpr int kFusedWaves = 16;
constexpr int kPairWaves = 8;                  // waves of a workgroup whose waves scan two KV heads each
constexpr unsigned kFusedShare = 33;           // 64ths of a sequence's tiles that go to the lower eight waves
constexpr unsigned kPairTileShare = 32;        // the same with eight waves in all: two per SIMD, no upper slots
constexpr int kFusedMaxQ = 32;                 // query heads of a unit: HKW * R <= 8 * 4
constexpr int kRowFloats = kHeadDim + 4;       // LDS row of a vector: conflict-free 16-byte accesses
constexpr int kMaxShares = 64;                 // workgroups that may share one sequence's context
enum { kStep = 0, kAttend = 1, kPaged = 2 };

}  // namespace

// EARLY (PAIR only): waves ask for their first tile in the middle of the prologue; for launches whose waves have few
// tiles (the host decides from what it knows of the context lengths).  A template parameter because the mere presence
// of that path, never taken, made the long-context launch 2 us slower.
// SHARES: f.shares (a power of two up to 64) workgroups share the context of a unit -- for batches whose units alone leave
// compute units idle.  Share c scans the c-th of f.shares even runs of the sequence's tiles; the last share appends the new row.  Each
// leaves its unnormalised sums in memory, draws a ticket, and the workgroup with the last ticket merges all of them (in
// share order, all read back from memory: the result does not depend on who was last) and finishes the unit.  The
// hand-over uses device-scope accesses only where they are needed -- the partial sums and the ticket -- and no
// cache-wide fence: stores with device scope are written through to where every compute unit's device-scope loads look
// (a release / acquire pair at device scope writes back and invalidates a whole L2 and costs 20 us per launch; this costs
// 2 to 4 us, which is what 1 sequence of 16001 tokens, 4 bit, 16 heads over 8 KV heads, pays to have 128 workgroups and
// more instead of 64 single chunks, a merge launch and a rotation launch -- 16 us per layer against 27).
// A share's waves have few tiles: SHARES asks for the first one in the prologue as EARLY does.  (While the prologue still waited for
// its loads one after the other that cost 5 % at 2 bit.)  The start and end bound a step of short contexts: every argument
// fetched in one trip, loads without branches, fp16 sums, parts merged four at a time.  28 layers of one sequence of 16001 tokens: 18.4 us
// a layer before, 15.8 with them (300 tokens 12.0 -> 10.2).
// MODE (PAIR, no SHARES): kAttend is attention alone, over a cache that holds the new token already (the reference's attention
// launcher): the unit's vectors are its queries, and the first tile is asked for in the prologue, nothing being appended.  kPaged
// is the whole step over the paged cache: a tile is two pages, whose block-table entries are fetched a tile ahead.
template <int R, int BITS, bool PROD, bool PAIR, bool EARLY, bool SHARES = false, int MODE = kStep>
__global__ void __launch_bounds__((PAIR ? kPairWaves : kFusedWaves) * kWave)
decode_fused_kernel(AttnArgs a, FusedArgs f) {
    static_assert(MODE == kStep || (PAIR && !SHARES && !EARLY && (MODE == kPaged || !PROD)), "modes of the pair kernel");
    constexpr bool kAppends = MODE != kAttend, kEarly = EARLY || SHARES || MODE != kStep;
    constexpr int NW = PAIR ? kPairWaves : kFusedWaves;        // waves of the workgroup
    constexpr int KW = BITS, VW = BITS;
    constexpr uint32_t kHeadBytes = BITS * 16;
    constexpr float kAlpha = BITS == 4 ? kAlpha4 : kAlpha2;
    __shared__ __attribute__((aligned(16))) uint32_t tab_s[kTableWords];
    // the scan's probabilities and partials; before the scan the same space holds R as 8 operand tiles, then the unit's vectors
    constexpr int kParts = PAIR ? 2 * NW : NW;                 // (part, head) partials: a wave leaves one per head it scans
    constexpr int kRotGroups = NW / 8;                         // groups of eight waves that rotate (a wave = 16 output coordinates)
    constexpr int kPBytes = NW * 16 * 32 * 2, kPartBytes = kParts * R * kRowFloats * 4;
    constexpr int kRotBytes = 8 * kOperandTileDwords * 4;
    constexpr int kMaxVecs = PAIR ? 4 * NW : 8 * (2 + R);      // vectors of a unit: a thread group of 16 each
    static_assert(kMaxVecs <= 4 * NW, "a vector per 16 threads");
    constexpr int kPrologueBytes = kRotBytes + kMaxVecs * kHeadDim * 2;
    __shared__ __attribute__((aligned(16))) char scan_s[kPBytes + kPartBytes > kPrologueBytes ? kPBytes + kPartBytes : kPrologueBytes];
    half_t (*p_s)[16][32] = reinterpret_cast<half_t (*)[16][32]>(scan_s);
    float (*part_s)[R][kRowFloats] = reinterpret_cast<float (*)[R][kRowFloats]>(scan_s + kPBytes);
    uint32_t* rot_s = reinterpret_cast<uint32_t*>(scan_s);
    uint4 (*x_s)[16] = reinterpret_cast<uint4 (*)[16]>(scan_s + kRotBytes);
    auto piece_of = [](int v, int p) -> int { return (p ^ (5 * v)) & 15; };
    __shared__ float inv_s[16];                                // 1 / |vector| of the K and V vectors
    // the rotated queries: floats, or (PAIR, at most 16 of them) operands of the score MFMAs
    __shared__ __attribute__((aligned(16))) char q_buf[PAIR ? 2 * 16 * 256 : kFusedMaxQ * kHeadDim * 4];
    float (*qrot_s)[kHeadDim] = reinterpret_cast<float (*)[kHeadDim]>(q_buf);
    uint4* qop_s = reinterpret_cast<uint4*>(q_buf);
    __shared__ __attribute__((aligned(16))) float o_s[kFusedMaxQ][kRowFloats];
    __shared__ __attribute__((aligned(8))) float2 bucket_s[kBuckets];

    const int tid = threadIdx.x;
    const int wave = uniform(tid / kWave), lane = tid % kWave;
    const int ln = lane & 15, kg = lane >> 4;          // names of the scan; the rotations call them i16, kk
    // the arguments in one trip: fetched where they are first used, the start is several of them one after the other
    asm volatile("" :: "s"(a.q), "s"(f.k_src), "s"(f.v_src), "s"(a.rotation), "s"(a.positions), "s"(a.num_kv_heads), "s"(f.hkw), "s"(f.nhg), "s"(f.shares),
                 "s"(f.by_xcd), "s"(a.G), "s"(a.q_stride), "s"(f.kv_stride), "s"(a.seq_stride_rows), "s"(PROD ? f.q_weight : nullptr),
                 "s"(PROD ? f.k_weight : nullptr), "s"(PROD ? f.cos_table : nullptr), "s"(PROD ? f.sin_table : nullptr), "s"(PROD ? f.rope_dim : 0), "s"(f.row_norm));
    const int Hk = a.num_kv_heads;
    const int HKW = f.hkw, hkw_log2 = __builtin_ctz(HKW);      // (powers of two: a division is fifty instructions here)
    const int nhg = f.nhg;                             // Hk / HKW
    const int SPLIT = kParts >> hkw_log2;              // parts of the context per head

    // ---- unit of this workgroup.  Workgroups are dealt to the 8 XCDs in turn; the units of one sequence
    // go to one XCD so that the norm rows they all read (16 bytes per token for 8 heads) come out of one L2.
    int g, hg, share = 0;
    const int nshares = SHARES ? f.shares : 1, share_log2 = SHARES ? __builtin_ctz(f.shares) : 0;
    {
        int b = (int)blockIdx.x >> (f.by_xcd ? 3 : 0);
        if (SHARES) { share = b & (nshares - 1); b >>= share_log2; }      // the shares of a unit on one XCD as well
        if ((nhg & (nhg - 1)) == 0) { g = b >> __builtin_ctz(nhg); hg = b & (nhg - 1); }
        else { g = b / nhg; hg = b - g * nhg; }
        if (f.by_xcd) {
            g = g * 8 + ((int)blockIdx.x & 7);
            if (g >= a.G) return;                                   // (the grid covers whole eights of sequences)
        }
    }
    const bool appends = kAppends && (!SHARES || share == nshares - 1);   // the share that holds the sequence's last tile
    // ---- operands of the rotations first: nothing about them depends on the position.  The unit's vectors
    // (K heads, V heads, query heads) are fetched once by all threads, 16 lanes to a vector, 16 bytes each;
    // waves 0-7 fetch 16 rows of R each.
    const int first_q = kAppends ? 2 * HKW : 0;            // the queries come behind the K and V heads
    const int nvec = first_q + HKW * R;
    const int rot_dblk = wave & 7;
    const bool rotating = wave < 8 * kRotGroups && (wave >> 3) * 16 < nvec;
    auto unit_vector = [&](int vc, int& kind, int& head) -> const half_t* {    // vc < nvec
        if (kAppends && vc < HKW) {
            kind = 0; head = hg * HKW + vc;
            return f.k_src + (long long)g * f.kv_stride + (long long)head * kHeadDim;
        }
        if (kAppends && vc < 2 * HKW) {
            kind = 1; head = hg * HKW + vc - HKW;
            return f.v_src + (long long)g * f.kv_stride + (long long)head * kHeadDim;
        }
        kind = 2; head = hg * HKW * R + (vc - first_q);
        return a.q + (long long)g * a.q_stride + (long long)head * kHeadDim;
    };
    // (Threads without a vector repeat one, waves without rows of R repeat some, and producers that are not there read the rotation: a load
    // in a branch is waited for, with all before it, at the branch's end.)
    const int my_vec = tid >> 4, my_piece = tid & 15;  // what this thread carries of the unit's vectors
    const bool carries = my_vec < nvec;
    int my_kind, my_head;
    const half_t* my_src = unit_vector(min(my_vec, nvec - 1), my_kind, my_head);
    const int pos_request = a.positions[g];
    const uint4 stage = reinterpret_cast<const uint4*>(my_src)[my_piece];
    uint4 prod_w = {0u, 0u, 0u, 0u};
    const bool normed = PROD && f.q_weight != nullptr, roped = PROD && f.cos_table != nullptr;
    if (PROD) prod_w = reinterpret_cast<const uint4*>(normed ? (my_kind == 0 ? f.k_weight : f.q_weight) : a.rotation)[my_piece];
    // R: wave w < 8 fetches rows 16w .. 16w + 15 (4 KB in a row, 4 fully used pieces per lane) and stages them
    // as an operand tile; the rotating waves read their operand from there
    uint4 rraw[4];
#pragma unroll
    for (int j = 0; j < 4; j++) rraw[j] = reinterpret_cast<const uint4*>(a.rotation + (wave & 7) * 16 * kHeadDim)[j * kWave + lane];

    // ---- the centroid table while the loads are under way: entry e fills 256 bytes with replicas.  A thread writes
    // entries e0 + 4 NW k, k = 0, 1, ...: the low four bits of e are the thread's own in every round (their
    // centroids come out of a register by wave shuffle, once: lane c holds centroid c; indexing the constant array
    // with a per-lane index is a dependent memory load per look-up, several microseconds for this loop), the
    // upper four are the same for the whole wave (v_readlane).
    {
        const float cent_lane = kAlpha * centroid_of<BITS>(lane);
        constexpr int kStep = NW * kWave * 4, kRounds = kTableWords / kStep;
        static_assert(kRounds * kStep == kTableWords && kStep % 1024 == 0, "a round advances e by a multiple of 16");
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
            // a byte's four codes in the order 0, 2, 1, 3 (one head per wave: what its lane-pair exchange wants) or
            // in their own order (two heads per wave)
            const half_t c0 = (half_t)__shfl(cent_lane, e0 & 3, 64), c1 = (half_t)__shfl(cent_lane, (e0 >> 2) & 3, 64);
#pragma unroll
            for (int k = 0; k < kRounds; k++) {
                const int hi = hi0 + (NW / 4) * k;          // e >> 4
                const half_t c2 = (half_t)cent_of(hi & 3), c3 = (half_t)cent_of(hi >> 2);
                half2_t p0 = {c0, PAIR ? c1 : c2};
                half2_t p1 = {PAIR ? c2 : c1, c3};
                const uint32_t w0 = *reinterpret_cast<uint32_t*>(&p0), w1 = *reinterpret_cast<uint32_t*>(&p1);
                *reinterpret_cast<uint4*>(&tab_s[tid * 4 + k * kStep]) = uint4{w0, w1, w0, w1};
            }
        }
    }
    if (BITS == 4 && wave == NW - 1 && lane < kBuckets) bucket_s[lane] = bucket_entry(lane);

    const int pos = uniform(pos_request);
    const int n = pos + 1;
    const int* bt = MODE == kPaged ? a.block_table + (long long)g * a.bt_stride : nullptr;
    // producers: the pieces of the table rows of this sequence's position that go with this thread's coordinates
    uint4 prod_c = {0u, 0u, 0u, 0u}, prod_s = {0u, 0u, 0u, 0u};
    if (PROD) {
        const long long at = roped ? (long long)pos * (f.rope_dim >> 4) + rope_piece16(my_piece, f.rope_dim) : 0;
        prod_c = reinterpret_cast<const uint4*>(roped ? f.cos_table : a.rotation)[at];
        prod_s = reinterpret_cast<const uint4*>(roped ? f.sin_table : a.rotation)[at];
    }
    // the sequence's first cache row.  (For long contexts in scalar registers by force, as is h: the new row's address is made on the vector
    // ALU, and with it the compiler put the base addresses of the scan there too, 8 to 12 instructions more per tile to make its
    // descriptors.  Where waves have few tiles the start's two trips to the scalar side cost as much.)
    const long long row0 = MODE == kPaged ? 0 : (long long)g * a.seq_stride_rows, seq_row0 = kEarly ? row0 : uniform(row0);
    // the new token's cache row
    const long long new_row = MODE == kPaged ? (long long)uniform(bt[pos / kPageTokens]) * kPageTokens + pos % kPageTokens
                                             : seq_row0 + pos;
    // PAIR: wave = part * (HKW / 2) + pair; hk_local is the first head of the pair
    const int hk_local = PAIR ? 2 * (wave & ((HKW >> 1) - 1)) : wave & (HKW - 1), part = PAIR ? 2 * wave >> hkw_log2 : wave >> hkw_log2;
    const int h = kEarly ? hg * HKW + hk_local : uniform(hg * HKW + hk_local);                 // (first) KV head of this wave

    // ---- tiles of 32 tokens this wave scans.  They are dealt round by round: in round r part p takes tile
    // r * SPLIT + p, so that at any moment the workgroup -- and with it the other workgroups of the sequence,
    // which started together -- reads one window of consecutive rows (1.2 % faster at 8192 tokens than giving
    // every part one contiguous run).  The parts of the upper eight waves stop after `rounds` rounds (31/64 of
    // the tiles); what is left goes round the lower waves' parts.
    const int ntile_seq = (n + 31) >> 5;
    // SHARES: this workgroup's run of the sequence's tiles (even runs, the last one ends with the sequence)
    const int tile_lo = SHARES ? (int)((unsigned)(share * ntile_seq) >> share_log2) : 0;
    const int ntile = SHARES ? (int)((unsigned)((share + 1) * ntile_seq) >> share_log2) - tile_lo : ntile_seq;
    const int halfparts = SPLIT >> 1;                      // SPLIT is 2, 4, 8 or 16
    const int lower = min(ntile, (int)((ntile * (PAIR ? kPairTileShare : kFusedShare) + 63u) / 64u));
    const int split_log2 = 31 - __builtin_clz(SPLIT), half_log2 = split_log2 - 1;
    const int rounds = (ntile - lower) >> half_log2;
    const int tail0 = rounds * SPLIT;                      // tail tiles tail0 + part + j * halfparts, lower parts only
    const int left = ntile - tail0 - part;
    const int ntiles = rounds + ((part < halfparts && left > 0) ? (left + halfparts - 1) >> half_log2 : 0);
    auto tile_at = [&](int i) -> int {                     // first token of this wave's i-th tile
        return 32 * (tile_lo + (i < rounds ? i * SPLIT + part : tail0 + part + (i - rounds) * halfparts));
    };
    const int first_tile = tile_at(0);

    // ---- scan set-up (as attention_mfma_kernel, contiguous layout)
    // Per-lane offsets and selectors.  They are derived after the rotations from a laundered copy of the lane
    // number: computed from the lane number itself they are hoisted to the top of the kernel, stay live across
    // the rotations, and the allocator spills some of them there and reloads them inside the scan loop, where a
    // reload waits for every load in flight.
    const char* tab_lane = reinterpret_cast<const char*>(tab_s);
    const uint32_t kvp = (uint32_t)Hk * kHeadBytes;
    const uint32_t nrow = (uint32_t)Hk * 2u;
    const uint32_t vstep = BITS == 4 ? kvp : 2u * kvp;  // V: dword i of a lane sits vstep bytes after dword 0 (one register for the four)
    const uint32_t sub_bytes = 16u * kvp;
    uint32_t lane_rep, koff, voff0, noff, sel_keep, sel_send;
    int ksrc, my_sub;
    bool odd, useful;
    half_t* p_w;
    const uint4* p_r;
    auto derive_lane = [&](int l) {
        const int ln_ = l & 15, kg_ = l >> 4;
        lane_rep = BITS == 4 ? (uint32_t)l * 4u : (uint32_t)(l & 31) * 8u;
        koff = (uint32_t)(l >> 2) * kvp + (kHeadBytes / 4) * (uint32_t)(l & 3);
        ksrc = 4 * (4 * ln_ + kg_);
        voff0 = BITS == 4 ? (uint32_t)(4 * kg_) * kvp + 4u * (uint32_t)ln_
                          : (uint32_t)(4 * kg_ + (ln_ & 1)) * kvp + 4u * (uint32_t)(ln_ >> 1);
        odd = (ln_ & 1) != 0;
        sel_keep = odd ? 0x07060302u : 0x05040100u;
        sel_send = odd ? 0x05040100u : 0x07060302u;
        my_sub = kg_ >> 1;
        useful = (kg_ & 1) == 0;
        noff = (uint32_t)ln_ * nrow + (uint32_t)my_sub * 16u * nrow;
        p_w = &p_s[wave][0][8 * (ln_ >> 2) + 4 * my_sub + (ln_ & 3)];
        p_r = reinterpret_cast<const uint4*>(&p_s[wave][ln_][8 * kg_]);
    };
    constexpr float kRaise = 5.0f;

    auto lut32 = [&](uint32_t addr) -> uint32_t { return *reinterpret_cast<const uint32_t*>(tab_lane + addr); };
    auto lut64 = [&](uint32_t addr) -> uint2 { return *reinterpret_cast<const uint2*>(tab_lane + addr); };

    const char* kseq = reinterpret_cast<const char*>(a.k) + (long long)h * kHeadBytes;
    const char* vseq = reinterpret_cast<const char*>(a.v) + (long long)h * kHeadBytes;
    const char* knseq = reinterpret_cast<const char*>(a.k_norms) + (long long)h * 2;
    const char* vnseq = reinterpret_cast<const char*>(a.v_norms) + (long long)h * 2;

    auto load_k = [&](__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t (&dst)[KW]) {
        if constexpr (BITS == 4) {
            uint32x4_t q = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
            dst[0] = q[0]; dst[1] = q[1]; dst[2] = q[2]; dst[3] = q[3];
        } else {
            uint32x2_t q = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
            dst[0] = q[0]; dst[1] = q[1];
        }
    };
    // Descriptors span the rows of the tile that exist (rows past the sequence's end read as zeros).
    auto issue_k = [&](uint32_t (&kreg)[2][KW], int tile) {
        __amdgpu_buffer_rsrc_t r = make_rsrc(kseq + (seq_row0 + tile) * kvp, max(min(n - tile, 32), 0) * (int)kvp);
        load_k(r, koff, kreg[0]);
        load_k(r, koff + sub_bytes, kreg[1]);
    };
    auto issue_v = [&](uint32_t (&vreg)[2][VW], int tile) {
        __amdgpu_buffer_rsrc_t r = make_rsrc(vseq + (seq_row0 + tile) * kvp, max(min(n - tile, 32), 0) * (int)kvp);
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
#pragma unroll
            for (int i = 0; i < VW; i++)
                vreg[sub][i] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(voff0 + i * vstep + sub * sub_bytes), 0, 0);
        }
    };
    auto pick = [&](const uint32x4_t& q) -> uint32_t {
        const int dw = (h & 7) >> 1;
        uint32_t w = dw == 0 ? q[0] : dw == 1 ? q[1] : dw == 2 ? q[2] : q[3];
        return (h & 1) ? (w >> 16) : (w & 0xffffu);
    };
    auto issue_n = [&](int tile) -> uint32_t {        // fp16 bits of kn (low) and vn (high) of this lane's token
        const bool wide = (nrow & 15u) == 0;
        const uint32_t hgrp = (uint32_t)(h >> 3) * 16u;
        const long long row = seq_row0 + tile;
        const int rows = max(min(n - tile, 32), 0);
        if (wide) {
            __amdgpu_buffer_rsrc_t rk = make_rsrc(reinterpret_cast<const char*>(a.k_norms) + row * nrow, rows * (int)nrow);
            __amdgpu_buffer_rsrc_t rv = make_rsrc(reinterpret_cast<const char*>(a.v_norms) + row * nrow, rows * (int)nrow);
            uint32x4_t kq = {0, 0, 0, 0}, vq = {0, 0, 0, 0};
            if (useful) {
                kq = __builtin_amdgcn_raw_buffer_load_b128(rk, (int)(noff + hgrp), 0, 0);
                vq = __builtin_amdgcn_raw_buffer_load_b128(rv, (int)(noff + hgrp), 0, 0);
            }
            return pick(kq) | (pick(vq) << 16);
        }
        __amdgpu_buffer_rsrc_t rk = make_rsrc(knseq + row * nrow, rows * (int)nrow);
        __amdgpu_buffer_rsrc_t rv = make_rsrc(vnseq + row * nrow, rows * (int)nrow);
        uint32_t kk = __builtin_amdgcn_raw_buffer_load_b16(rk, (int)noff, 0, 0);
        uint32_t vv = __builtin_amdgcn_raw_buffer_load_b16(rv, (int)noff, 0, 0);
        return kk | (vv << 16);
    };

    uint32_t kreg[2][KW];
    uint32_t vreg[2][VW];
    uint32_t nreg = 0;
    // (One head per wave: tiles are only requested after the rotations.  Asking for the first one up front, without the
    // row this workgroup is about to store, made launches 0.4 to 0.9 us slower at every context length, also with R
    // arriving in 4 coalesced pieces per lane, and no faster when only the waves without a rotation to do ask;
    // pulling further tiles towards the caches during the prologue cost 2 us per tile: what the prologue waits
    // for then queues behind them.)

    // ---- 1. rotations of the unit's vectors
    // early(): called once the staged vectors and R are in LDS, before the rotations -- where the scan asks for its
    // first tile when that tile lies wholly before the new token
    auto rotate_unit = [&](auto early) {
        const int i16 = ln, kk = kg;
        const int dblk = rot_dblk;
        if (wave < 8) stage_operand_tile(rot_s + wave * kOperandTileDwords, rraw, lane);
        // This thread's piece of its vector: the optional producers (K and queries; each step rounded to fp16 as the
        // reference's in-place kernels leave it), the norm in the reference's order, and the halves into LDS, once for
        // all waves, regrouped for the matrix cores: coordinate 4s + kk of vector v in 16-byte piece 4kk + s / 8 of its row, which lies at
        // that piece ^ 5v (no bank twice, written or read).
        if (carries) {                                     // the same for the 16 lanes of a vector
            float x[8], t[8];
            unpack_halves(stage, x);
            if (PROD && my_kind != 1) {
                if (normed) norm_head16(x, prod_w, f.eps, f.biased);
                if (roped) rope_head16(x, prod_c, prod_s, my_piece, f.rope_dim, 0);
            }
            const uint4 w = PROD ? pack_halves(x) : stage;
            const uint32_t by_kk[4] = {(w.x & 0xffffu) | (w.z << 16), (w.x >> 16) | (w.z & 0xffff0000u),
                                       (w.y & 0xffffu) | (w.w << 16), (w.y >> 16) | (w.w & 0xffff0000u)};
#pragma unroll
            for (int k4 = 0; k4 < 4; k4++)
                reinterpret_cast<uint32_t*>(&x_s[my_vec][piece_of(my_vec, 4 * k4 + (my_piece >> 2))])[my_piece & 3] = by_kk[k4];
            if (kAppends && my_kind != 2) {
#pragma unroll
                for (int e = 0; e < 8; e++) t[e] = x[e] * x[e];            // exact: fp16 values
                const float norm = sqrtf(head_tree_sum16(t) + 1e-12f);
                if (my_piece == 0) {
                    inv_s[my_vec] = 1.0f / norm;
                    if (appends) (my_kind == 0 ? f.k_norms : f.v_norms)[new_row * Hk + my_head] = (half_t)norm;
                }
            }
        }
        lds_barrier();
        early();
        uint4 rv[4];                                       // R[16 * rot_dblk + ln][4s + kg], s = 8j .. 8j + 7
        float row_norm = f.row_norm;
        if (rotating) {
#pragma unroll
            for (int j = 0; j < 4; j++) rv[j] = *reinterpret_cast<const uint4*>(rot_s + rot_dblk * kOperandTileDwords + operand_tile_dword(lane, 4 * j));
            if (appends && row_norm == 0.0f) row_norm = operand_rows_norm(rv);
        }
        for (int vt = wave >> 3; rotating && vt * 16 < nvec; vt += kRotGroups) {  // uniform over the wave
            const int vi = vt * 16 + i16;
            const int vc = vi < nvec ? vi : nvec - 1;              // clamp reads, mask stores
            int kind, head;
            (void)unit_vector(vc, kind, head);
            const bool is_query = kind == 2;
            // fp16 values times an fp16 matrix: every product exact, the sums in fp32
            float4_t acc = {0.f, 0.f, 0.f, 0.f}, sums[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                union { uint4 u; half8_t h; } xv, rm;
                xv.u = x_s[vc][piece_of(vc, 4 * kk + j)];
                rm.u = rv[j];
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(rm.h, xv.h, acc, 0, 0, 0);
                sums[j] = acc;
            }
            if (is_query && vi < nvec) {
                float4 o = {acc[0] * f.q_scale, acc[1] * f.q_scale, acc[2] * f.q_scale, acc[3] * f.q_scale};
                if (PAIR) store_query_operand(qop_s, vc - first_q, dblk, kk, acc, f.q_scale);
                else *reinterpret_cast<float4*>(&qrot_s[vc - first_q][dblk * 16 + 4 * kk]) = o;
            }
            if (appends && vt * 16 < first_q) {                    // lane: coordinates 16 dblk + 4kk .. + 3
                // codes: those of the fp32 chain, by the sums above unless one of the block's is too near to a boundary
                // for them (kv_rotate_util.hpp; one block in 17 with 16 vectors, one in 66 with 4)
                const bool live = vi < nvec && !is_query;
                const float inv = live ? inv_s[vc] : 0.0f;
                uint32_t packed = 0;
                bool doubt = false;
#pragma unroll
                for (int r = 0; r < 4; r++) packed |= bucket_quantize_sure<BITS>(bucket_s, sums, r, inv, row_norm, doubt) << (r * BITS);
                if (__any(live && doubt)) {
                    acc = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        float rf[8], uf[8];
                        unpack_halves(rv[j], rf);
                        unpack_halves(x_s[vc][piece_of(vc, 4 * kk + j)], uf);
#pragma unroll
                        for (int e = 0; e < 8; e++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(rf[e], uf[e] * inv, acc, 0, 0, 0);
                    }
                    packed = 0;
#pragma unroll
                    for (int r = 0; r < 4; r++) packed |= bucket_quantize<BITS>(bucket_s, acc[r]) << (r * BITS);
                }
                if (live) {
                    uint8_t* dst = (kind == 0 ? f.k_codes : f.v_codes) + (new_row * Hk + head) * kHeadBytes + (4 * dblk + kk) * (BITS / 2);
                    if (BITS == 4) *reinterpret_cast<uint16_t*>(dst) = (uint16_t)packed;
                    else *dst = (uint8_t)packed;
                }
            }
        }
        if (appends) __syncthreads();         // table, q_rot and the new cache row are in place; R has been read
        else lds_barrier();                   // (no new row: the first tile stays in flight)
        // the wave's slice of the probabilities starts at zero (no other wave touches it)
        *reinterpret_cast<uint4*>(&p_s[wave][0][0] + 8 * lane) = uint4{0u, 0u, 0u, 0u};
    };
    // ---- 3. the parts meet in LDS.  B operand of the rotate-back first (its loads run under the merge, and stay
    // hidden there: R brought in coalesced and passed through LDS instead was 0.25 us slower per launch):
    // R[32kk + s][16*dblk + i16], s = 0..31
    const int nv = HKW * R;                                  // output vectors of this unit
    const int dblk = wave & 7;
    const bool back = wave < 8 * kRotGroups && (wave >> 3) * 16 < nv;
    uint16_t rb[32];
    auto load_rb = [&]() {
    if (PAIR || back) {          // (PAIR: eight waves, every one of them rotates back)
        const uint16_t* rp = reinterpret_cast<const uint16_t*>(a.rotation) + (32 * kg) * kHeadDim + 16 * dblk + ln;
#pragma unroll
        for (int s = 0; s < 32; s++) rb[s] = rp[s * kHeadDim];
    }
    };
    if constexpr (PAIR) {
        // ---- 2 (PAIR). scan of this wave's part, two KV heads per wave (kv_pair_scan.hpp has the tile and why)
        int l2 = lane;
        asm volatile("" : "+v"(l2));
        PairLane<R, BITS> L;
        L.init(l2, p_s[wave], tab_s);
        const uint32_t kvp = (uint32_t)Hk * kHeadBytes;
        const uint32_t nrow = (uint32_t)Hk * 2u;
        const uint32_t koff = L.koff_rows * kvp + L.koff_bytes;
        const uint32_t voff = L.voff_rows * kvp + L.voff_bytes;
        const uint32_t noff = (uint32_t)L.tok0 * nrow;
        // the sequence's rows of this pair: a tile is one multiplication per array away
        const char* kpair = reinterpret_cast<const char*>(a.k) + seq_row0 * kvp + (long long)h * kHeadBytes;
        const char* vpair = reinterpret_cast<const char*>(a.v) + seq_row0 * kvp + (long long)h * kHeadBytes;
        const char* knpair = reinterpret_cast<const char*>(a.k_norms) + seq_row0 * nrow + (long long)h * 2;
        const char* vnpair = reinterpret_cast<const char*>(a.v_norms) + seq_row0 * nrow + (long long)h * 2;
        // The tile whose loads are issued during the current one: first token and rows that exist.  (Loads of a tile
        // past the wave's last one get an empty extent: they return zeros without touching memory.)
        int next_tile = 0, next_rows = 0;
        // (paged: the tile's two block-table entries, in the even and odd lanes, and those of the tile after it on the way; past the
        // end the last page again, its tokens masked)
        int pages = 0, pages_after = 0;
        auto fetch_pages = [&](int i) -> int { return bt[min(tile_at(i) + kPageTokens * (lane & 1), pos) / kPageTokens]; };
        auto page_row = [&](int sub) -> long long { return (long long)__builtin_amdgcn_readlane(pages, sub) * kPageTokens; };
        auto set_next = [&](int i) {
            next_tile = tile_at(i);
            next_rows = i < ntiles ? max(min(n - next_tile, 32), 0) : 0;
            if (MODE == kPaged) {
                pages = pages_after;
                pages_after = fetch_pages(i + 1);
            }
        };
        auto page_bytes = [&](uint32_t row) -> int { return next_rows > 0 ? kPageTokens * (int)row : 0; };
        // (4 bit: every load instruction covers whole lines, non-temporal; 2 bit: half lines, the ordinary policy)
        constexpr int kCodesAux = BITS == 4 ? kStreamCodes : 0;
        auto load_k = [&](__amdgpu_buffer_rsrc_t r, uint32_t off) {
            if constexpr (BITS == 4) return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, kCodesAux);
            else return __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, kCodesAux);
        };
        auto load_v = [&](__amdgpu_buffer_rsrc_t r, uint32_t off) {
            if constexpr (BITS == 4) return __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, kCodesAux);
            else return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, kCodesAux);
        };
        auto issue_k = [&](PairTileRegs<BITS>& t) {
            if constexpr (MODE == kPaged) {
#pragma unroll
                for (int sub = 0; sub < 2; sub++) {
                    __amdgpu_buffer_rsrc_t r = make_rsrc(kpair + page_row(sub) * kvp, page_bytes(kvp));
                    t.k[2 * sub] = load_k(r, koff);
                    t.k[2 * sub + 1] = load_k(r, koff + 8u * kvp);
                }
            } else {
                __amdgpu_buffer_rsrc_t r = make_rsrc(kpair + (long long)next_tile * kvp, next_rows * (int)kvp);
#pragma unroll
                for (int c = 0; c < 4; c++) t.k[c] = load_k(r, koff + (uint32_t)(8 * c) * kvp);
            }
        };
        auto issue_v = [&](PairTileRegs<BITS>& t) {
            if constexpr (MODE == kPaged) {
#pragma unroll
                for (int sub = 0; sub < 2; sub++) {
                    __amdgpu_buffer_rsrc_t r = make_rsrc(vpair + page_row(sub) * kvp, page_bytes(kvp));
#pragma unroll
                    for (int j = 0; j < 4; j++) t.v[sub][j] = load_v(r, voff + (uint32_t)j * kvp);
                }
            } else {
                __amdgpu_buffer_rsrc_t r = make_rsrc(vpair + (long long)next_tile * kvp, next_rows * (int)kvp);
#pragma unroll
                for (int sub = 0; sub < 2; sub++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) t.v[sub][j] = load_v(r, voff + (uint32_t)(16 * sub + j) * kvp);
                }
            }
        };
        // (every lane asks, also those that own no token: they repeat a neighbour's address, which costs nothing, and
        // the loop has no branch here)
        auto issue_n = [&](PairTileRegs<BITS>& t) {
            if constexpr (MODE == kPaged) {
                // (the rows that exist and no more: an unwritten slot's norm may be a NaN or an infinity, which a probability of
                // zero does not take out; codes of any bits are finite values)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int bytes = min(max(next_rows - kPageTokens * i, 0), kPageTokens) * (int)nrow;
                    __amdgpu_buffer_rsrc_t rk = make_rsrc(knpair + page_row(i) * nrow, bytes);
                    __amdgpu_buffer_rsrc_t rv = make_rsrc(vnpair + page_row(i) * nrow, bytes);
                    t.n[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)noff, 0, kStreamNorms);
                    t.n[i][1] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)noff, 0, kStreamNorms);
                }
                return;
            }
            __amdgpu_buffer_rsrc_t rk = make_rsrc(knpair + (long long)next_tile * nrow, next_rows * (int)nrow);
            __amdgpu_buffer_rsrc_t rv = make_rsrc(vnpair + (long long)next_tile * nrow, next_rows * (int)nrow);
            t.n[0][0] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)noff, 0, kStreamNorms);
            t.n[1][0] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)(noff + 16u * nrow), 0, kStreamNorms);
            t.n[0][1] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)noff, 0, kStreamNorms);
            t.n[1][1] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)(noff + 16u * nrow), 0, kStreamNorms);
        };

        PairState<R> S;
        S.reset();
        // One tile of loads in flight per wave.  (Tried: two tiles, 2 % slower; a second register set for K alone, whose
        // loads otherwise have only the softmax and P.V of one tile to arrive in, 6 % slower -- more requests in flight
        // make the memory slower here, not faster; the first tile asked for before the rotations, 0.4 us slower, as
        // with one head per wave; the scores of tile i + 1 placed beside the P.V of tile i for the scheduler to
        // interleave, 3 % slower.)
        PairTileRegs<BITS> t;
        // (EARLY) a wave asks for its first tile in the middle of the prologue, behind the prologue's own loads
        // and ahead of the rotations, when all of its rows are older than the token this launch appends (the launch's
        // own row only exists after the barrier that ends the rotations).  Rollouts of a few hundred tokens gain
        // 4.5 % (128 sequences at 257..768 tokens: 21.6 against 22.6 us per launch); with 8 tiles per wave it makes no
        // difference, and with 16 and more the launch gets slower (64 x 4096 tokens: + 0.6 us, x 8192: + 2.2 us), as
        // with every other way of putting more requests in flight at the start that was tried.  (A second register set
        // in this short-context form, so that the tile after next is in flight too -- the memory is far from busy there:
        // 22.9 against 21.2 us per launch on the rollout, 24.7 against 23.5 at 64 x 1024 tokens, 8 % and 5 % slower; with
        // four query heads per KV head it does not fit the registers.  A wave's tile time at these sizes is the tile's
        // own chain of look-ups and matrix instructions, not the wait for its loads.)
        const bool first_early = kEarly && ntiles > 0 && (MODE == kAttend || tile_at(0) + 32 <= pos);      // uniform over the wave
        pages_after = MODE == kPaged ? fetch_pages(0) : 0;
        rotate_unit([&]() {
            set_next(0);
            if (kEarly) {                    // (asked for without a branch: behind one, the next wait of the prologue takes the tile with it)
                const int rows = next_rows;
                if (!first_early) next_rows = 0;
                issue_k(t); issue_n(t); issue_v(t);
                next_rows = rows;
            }
        });
        if (!first_early) { issue_k(t); issue_n(t); issue_v(t); }
        if (kEarly && !SHARES) load_rb();    // behind the first tile's loads; the registers are there, and the epilogue need not wait
        if (ntiles > 0) {
            S.load_query_operands(L, [&](int i, int part2, int p) { return &qop_s[query_piece(2 * (hk_local * R + i) + part2, p)]; });
            if (!kEarly) S.zero_repeated_queries(L);
            for (int it = 0; it < ntiles; it++) {
                const int tile = next_tile;
                set_next(it + 1);
                pair_scan_tile<R>(L, S, t, tile, n, [&]() { issue_k(t); }, [&]() { issue_n(t); }, [&]() { issue_v(t); });
            }
        }
        // (Long contexts ask at the end: at the start these 32 two-byte loads a wave hold up the second tile.  With the scalar addresses
        // above 64 x 8192 tokens 94.0 -> 92.7 us, 96 x 4096 79.1 -> 77.7, 112 x 8192 167.2 -> 164.5.)
        if (!kEarly) load_rb();
        pair_scan_finish<R>(L, S, 1.0f / kAlpha, [&](int hd, int r, const float (&ov)[16]) {
            float* pr = &part_s[part * HKW + hk_local + hd][r][0];
#pragma unroll
            for (int j4 = 0; j4 < 4; j4++)
                *reinterpret_cast<float4*>(pr + 16 * (L.pn & 7) + 4 * j4) = float4{ov[4 * j4], ov[4 * j4 + 1], ov[4 * j4 + 2], ov[4 * j4 + 3]};
            if ((L.pn & 7) == 0) { pr[kHeadDim] = S.m_run[r]; pr[kHeadDim + 1] = S.l_run[r]; }
        });
    } else {
        rotate_unit([]() {});
        {
            int l2 = lane;
            asm volatile("" : "+v"(l2));
            derive_lane(l2);
        }

        // ---- 2. scan of this wave's part
        float4_t o[8];
    #pragma unroll
        for (int j = 0; j < 8; j++) o[j] = float4_t{0.f, 0.f, 0.f, 0.f};
        float m_run[R], l_run[R];
    #pragma unroll
        for (int r = 0; r < R; r++) { m_run[r] = kNegBig; l_run[r] = 0.0f; }

        if (ntiles > 0) {
            issue_k(kreg, first_tile);
            nreg = issue_n(first_tile);
            issue_v(vreg, first_tile);
            // A operand of the score MFMAs: q_rot[head][32kg + 8j + i], row m = fp16 value of head m, row m + 8
            // its rounding remainder; the 2-bit table returns the codes of a byte in the order 0,2,1,3
            half8_t aq[4];
            {
                const int hq = ln & 7;
                const bool lo_part = (ln & 8) != 0;
                const float* qr = &qrot_s[hk_local * R + (hq < R ? hq : 0)][32 * kg];
    #pragma unroll
                for (int j = 0; j < 4; j++) {
                    float4 v0 = *reinterpret_cast<const float4*>(qr + 8 * j);
                    float4 v1 = *reinterpret_cast<const float4*>(qr + 8 * j + 4);
                    float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
    #pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const int src = BITS == 4 ? i : ((i & 4) | ((i & 1) << 1) | ((i & 2) >> 1));
                        float x = (hq < R) ? v[src] : 0.0f;
                        half_t hi = (half_t)x;
                        half_t lo = (half_t)(x - (float)hi);
                        aq[j][i] = lo_part ? lo : hi;
                    }
                }
            }

            for (int it = 0; it < ntiles; it++) {
                const int tile = tile_at(it);
                const int next_tile = tile_at(it + 1);
                const bool more = it + 1 < ntiles;

                // ---- scores S[head][token] for both sub-tiles
                float4_t s[2];
    #pragma unroll
                for (int sub = 0; sub < 2; sub++) {
                    uint32_t kw[KW];
    #pragma unroll
                    for (int i = 0; i < KW; i++) kw[i] = (uint32_t)__builtin_amdgcn_ds_bpermute(ksrc, (int)kreg[sub][i]);
                    union { uint32_t u[4]; half8_t h; } kv[4];
    #pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if constexpr (BITS == 4) {
                            const uint32_t w = kw[j];
                            kv[j].u[0] = lut32(__builtin_amdgcn_perm(w, lane_rep, 0x0c0c0400u));
                            kv[j].u[1] = lut32(__builtin_amdgcn_perm(w, lane_rep, 0x0c0c0500u));
                            kv[j].u[2] = lut32(__builtin_amdgcn_perm(w, lane_rep, 0x0c0c0600u));
                            kv[j].u[3] = lut32(__builtin_amdgcn_perm(w, lane_rep, 0x0c0c0700u));
                        } else {
                            const uint32_t w = kw[j >> 1];
                            const uint32_t sel = (j & 1) ? 0x0c0c0600u : 0x0c0c0400u;
                            uint2 l0 = lut64(__builtin_amdgcn_perm(w, lane_rep, sel));
                            uint2 l1 = lut64(__builtin_amdgcn_perm(w, lane_rep, sel + 0x100u));
                            kv[j].u[0] = l0.x; kv[j].u[1] = l0.y; kv[j].u[2] = l1.x; kv[j].u[3] = l1.y;
                        }
                    }
                    s[sub] = float4_t{0.f, 0.f, 0.f, 0.f};
    #pragma unroll
                    for (int j = 0; j < 4; j++) s[sub] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aq[j], kv[j].h, s[sub], 0, 0, 0);
                }
                if (more) issue_k(kreg, next_tile);

                // ---- online softmax (base 2): this lane owns token ln of sub-tile my_sub
                const float kn = h2f_bits(nreg & 0xffffu), vn = h2f_bits(nreg >> 16);
                if (more) nreg = issue_n(next_tile);
                const bool valid = useful && (tile + 16 * my_sub + ln < n);
                float raw[R], x[R];
                bool raise = false;
    #pragma unroll
                for (int r = 0; r < R; r++) {
                    uint32x2_t sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(s[0][r]), __float_as_uint(s[1][r]), false, false);
                    raw[r] = (__uint_as_float(sw[0]) + __uint_as_float(sw[1])) * kn;    // kernels.cu:1707
                    x[r] = valid ? raw[r] - m_run[r] : kNegBig;
                    raise = raise || (x[r] > kRaise);
                }
                if (__any(raise)) {
    #pragma unroll
                    for (int r = 0; r < R; r++) {
                        float m_new = fmaxf(m_run[r], wave_max(valid ? raw[r] : kNegBig));
                        float alpha = __builtin_amdgcn_exp2f(m_run[r] - m_new);
                        m_run[r] = m_new;
                        l_run[r] *= alpha;
                        x[r] = valid ? raw[r] - m_new : kNegBig;
    #pragma unroll
                        for (int j = 0; j < 8; j++) o[j][r] *= alpha;
                    }
                }
    #pragma unroll
                for (int r = 0; r < R; r++) {
                    float p = __builtin_amdgcn_exp2f(x[r]);
                    l_run[r] += p;
                    float pf = p * vn;                                      // (s * vn) * centroid, kernels.cu:1765
                    half_t hi = (half_t)pf;
                    half_t lo = (half_t)(pf - (float)hi);
                    if (useful) {
                        p_w[r * 32] = hi;
                        p_w[(r + 8) * 32] = lo;
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                union { uint4 q; half8_t h; } pa;
                pa.q = *p_r;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                __builtin_amdgcn_wave_barrier();

                // ---- O[head][dim 8ln + j] += P[head][token] V[token][dim]
                if constexpr (BITS == 4) {
                    uint32_t xe[4], xo[4];
    #pragma unroll
                    for (int sub = 0; sub < 2; sub++) {
    #pragma unroll
                        for (int pr = 0; pr < 2; pr++) {
                            uint32_t wa = vreg[sub][2 * pr], wb = vreg[sub][2 * pr + 1];
                            xe[2 * sub + pr] = (wa & 0x0f0f0f0fu) | ((wb << 4) & 0xf0f0f0f0u);
                            xo[2 * sub + pr] = ((wa >> 4) & 0x0f0f0f0fu) | (wb & 0xf0f0f0f0u);
                        }
                    }
                    if (more) issue_v(vreg, next_tile);
    #pragma unroll
                    for (int jp = 0; jp < 4; jp++) {
                        const uint32_t sel = 0x0c0c0400u + ((uint32_t)jp << 8);
                        union { uint32_t u[4]; half8_t h; } be, bo;
    #pragma unroll
                        for (int q4 = 0; q4 < 4; q4++) {
                            be.u[q4] = lut32(__builtin_amdgcn_perm(xe[q4], lane_rep, sel));
                            bo.u[q4] = lut32(__builtin_amdgcn_perm(xo[q4], lane_rep, sel));
                        }
                        o[2 * jp] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa.h, be.h, o[2 * jp], 0, 0, 0);
                        o[2 * jp + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa.h, bo.h, o[2 * jp + 1], 0, 0, 0);
                    }
                } else {
                    uint32_t ie[2], io[2];
    #pragma unroll
                    for (int sub = 0; sub < 2; sub++) {
                        const uint32_t keep = __builtin_amdgcn_perm(vreg[sub][1], vreg[sub][0], sel_keep);
                        const uint32_t send = __builtin_amdgcn_perm(vreg[sub][1], vreg[sub][0], sel_send);
                        const uint32_t recv = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send, 0xB1, 0xf, 0xf, false);  // lane ^ 1
                        const uint32_t wa = odd ? recv : keep, wb = odd ? keep : recv;
                        ie[sub] = (wa & 0x0f0f0f0fu) | ((wb << 4) & 0xf0f0f0f0u);
                        io[sub] = ((wa >> 4) & 0x0f0f0f0fu) | (wb & 0xf0f0f0f0u);
                    }
                    if (more) issue_v(vreg, next_tile);
    #pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const uint32_t x0 = (q & 1) ? io[0] : ie[0], x1 = (q & 1) ? io[1] : ie[1];
                        const uint32_t sel = 0x0c0c0400u + ((uint32_t)(q >> 1) << 8);
                        uint2 l00 = lut64(__builtin_amdgcn_perm(x0, lane_rep, sel));
                        uint2 l01 = lut64(__builtin_amdgcn_perm(x0, lane_rep, sel + 0x200u));
                        uint2 l10 = lut64(__builtin_amdgcn_perm(x1, lane_rep, sel));
                        uint2 l11 = lut64(__builtin_amdgcn_perm(x1, lane_rep, sel + 0x200u));
                        union { uint32_t u[4]; half8_t h; } be, bo;
                        be.u[0] = l00.x; be.u[1] = l01.x; be.u[2] = l10.x; be.u[3] = l11.x;
                        bo.u[0] = l00.y; bo.u[1] = l01.y; bo.u[2] = l10.y; bo.u[3] = l11.y;
                        o[2 * q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa.h, be.h, o[2 * q], 0, 0, 0);
                        o[2 * q + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa.h, bo.h, o[2 * q + 1], 0, 0, 0);
                    }
                }
            }
        }

    if (!SHARES) load_rb();
    #pragma unroll
        for (int r = 0; r < R; r++) {
            l_run[r] = wave_sum(l_run[r]);
    #pragma unroll
            for (int j = 0; j < 8; j++) o[j][r] += __shfl_xor(o[j][r], 32, 64);   // row r + row r+8 (lo part of P)
        }
        if (kg == 0) {
    #pragma unroll
            for (int r = 0; r < R; r++) {
                float* pr = &part_s[wave][r][0];
                float4 lo4 = {o[0][r] * (1.0f / kAlpha), o[1][r] * (1.0f / kAlpha), o[2][r] * (1.0f / kAlpha), o[3][r] * (1.0f / kAlpha)};
                float4 hi4 = {o[4][r] * (1.0f / kAlpha), o[5][r] * (1.0f / kAlpha), o[6][r] * (1.0f / kAlpha), o[7][r] * (1.0f / kAlpha)};
                *reinterpret_cast<float4*>(pr + 8 * ln) = lo4;
                *reinterpret_cast<float4*>(pr + 8 * ln + 4) = hi4;
                if (ln == 0) { pr[kHeadDim] = m_run[r]; pr[kHeadDim + 1] = l_run[r]; }
            }
        }
    }
    lds_barrier();                 // the loads of R above stay in flight

    {   // merge: thread -> (vector tid / 32, coordinates 4 * (tid % 32) .. +3); vector = (local KV head, query head)
        const int vec = tid >> 5, k4 = (tid & 31) * 4;
        float4 o4 = {0.f, 0.f, 0.f, 0.f};
        float mg = kNegBig, lsum = 0.0f;
        float4 av = {0.f, 0.f, 0.f, 0.f};
        if (vec < nv) {
            const int hk_l = vec / R, r = vec - hk_l * R;
            // (four parts' reads at a time: one after the other each is a trip through LDS)
            for (int p0 = 0; p0 < SPLIT; p0 += 4) {
                float2 ml[4];
                float4 c[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float* pr = &part_s[min(p0 + j, SPLIT - 1) * HKW + hk_l][r][0];
                    ml[j] = *reinterpret_cast<const float2*>(pr + kHeadDim);
                    c[j] = *reinterpret_cast<const float4*>(pr + k4);
                }
                const float m0 = mg;
#pragma unroll
                for (int j = 0; j < 4; j++) mg = fmaxf(mg, ml[j].x);
                const float f0 = __builtin_amdgcn_exp2f(m0 - mg);
                lsum *= f0; av.x *= f0; av.y *= f0; av.z *= f0; av.w *= f0;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float fs = p0 + j < SPLIT ? __builtin_amdgcn_exp2f(ml[j].x - mg) : 0.0f;
                    lsum = __builtin_fmaf(ml[j].y, fs, lsum);
                    av.x = __builtin_fmaf(c[j].x, fs, av.x);
                    av.y = __builtin_fmaf(c[j].y, fs, av.y);
                    av.z = __builtin_fmaf(c[j].z, fs, av.z);
                    av.w = __builtin_fmaf(c[j].w, fs, av.w);
                }
            }
        }
        if constexpr (SHARES) {
            // this share's sums to memory (device scope: written through), then the ticket.  16-byte accesses with the sc1
            // bit of device scope; a row of the sums is 128 values, then maximum and sum (and two spare words).
            __shared__ unsigned last_s;
            const long long unit = (long long)g * nhg + hg;
            const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<const char*>(f.share_ws + unit * nshares * nv * kRowFloats),
                                                        nshares * nv * kRowFloats * 4);
            auto row_bytes = [&](int sh, int v) -> int { return (sh * nv + v) * (kRowFloats * 4); };
            auto bits4 = [](const float4& x) -> uint32x4_t {
                return uint32x4_t{__float_as_uint(x.x), __float_as_uint(x.y), __float_as_uint(x.z), __float_as_uint(x.w)};
            };
            if (vec < nv) {
                __builtin_amdgcn_raw_buffer_store_b128(bits4(av), rs, row_bytes(share, vec) + 4 * k4, 0, kDeviceScope);
                if (k4 == 0)
                    __builtin_amdgcn_raw_buffer_store_b128(bits4(float4{mg, lsum, 0.f, 0.f}), rs, row_bytes(share, vec) + 4 * kHeadDim, 0, kDeviceScope);
            }
            __builtin_amdgcn_s_waitcnt(0);          // every store of this wave has been acknowledged
            __syncthreads();
            if (tid == 0) {
                const unsigned old = __hip_atomic_fetch_add(f.tickets + unit, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last_s = old == (unsigned)nshares - 1u ? 1u : 0u;
            }
            __syncthreads();
            if (!last_s) return;                    // uniform over the workgroup: the last share finishes the unit
            load_rb();                              // (by every share beside its scan, these 32 loads a wave hold the second tile up)
            if (tid == 0) __hip_atomic_store(f.tickets + unit, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
            // The slots of 32 threads that the unit's vectors leave free take a part of the shares each (slot = (part, vector),
            // shares part, part + nsub, ...), eight shares' loads in flight at a time -- one share after the other costs
            // a trip to memory each -- and the parts meet in LDS, where the waves' partial sums were.  All orders
            // are fixed by the shape alone.
            constexpr int kSlots = NW * kWave / 32;
            const int nv_log2 = 31 - __builtin_clz(nv);                    // nv is a power of two, at most both
            const int nsub = min(kSlots, kParts * R) >> nv_log2;
            const int mv = vec & (nv - 1), msub = vec >> nv_log2;
            float (*sum_s)[kRowFloats] = &part_s[0][0];
            if (msub < nsub) {
                float m = kNegBig, l = 0.0f;
                float4 acc = {0.f, 0.f, 0.f, 0.f};
                for (int s0 = msub; s0 < nshares; s0 += 8 * nsub) {
                    uint32x4_t ml[8], x[8];
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int at = row_bytes(min(s0 + j * nsub, nshares - 1), mv);
                        ml[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, at + 4 * kHeadDim, 0, kDeviceScope);
                        x[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, at + 4 * k4, 0, kDeviceScope);
                    }
                    float mb = m;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        if (s0 + j * nsub >= nshares) ml[j] = uint32x4_t{__float_as_uint(kNegBig), 0u, 0u, 0u};
                        mb = fmaxf(mb, __uint_as_float(ml[j][0]));
                    }
                    const float fo = __builtin_amdgcn_exp2f(m - mb);
                    l *= fo; acc.x *= fo; acc.y *= fo; acc.z *= fo; acc.w *= fo;
                    m = mb;
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const float fs = s0 + j * nsub < nshares ? __builtin_amdgcn_exp2f(__uint_as_float(ml[j][0]) - m) : 0.0f;
                        l = __builtin_fmaf(__uint_as_float(ml[j][1]), fs, l);
                        acc.x = __builtin_fmaf(__uint_as_float(x[j][0]), fs, acc.x);
                        acc.y = __builtin_fmaf(__uint_as_float(x[j][1]), fs, acc.y);
                        acc.z = __builtin_fmaf(__uint_as_float(x[j][2]), fs, acc.z);
                        acc.w = __builtin_fmaf(__uint_as_float(x[j][3]), fs, acc.w);
                    }
                }
                *reinterpret_cast<float4*>(&sum_s[vec][k4]) = acc;
                if (k4 == 0) { sum_s[vec][kHeadDim] = m; sum_s[vec][kHeadDim + 1] = l; }
            }
            lds_barrier();
            if (vec < nv) {
                mg = kNegBig; lsum = 0.0f;
                av = float4{0.f, 0.f, 0.f, 0.f};
                for (int u = 0; u < nsub; u++) mg = fmaxf(mg, sum_s[u * nv + vec][kHeadDim]);
                for (int u = 0; u < nsub; u++) {
                    const float* pr = &sum_s[u * nv + vec][0];
                    const float fs = __builtin_amdgcn_exp2f(pr[kHeadDim] - mg);
                    const float4 c = *reinterpret_cast<const float4*>(pr + k4);
                    lsum = __builtin_fmaf(pr[kHeadDim + 1], fs, lsum);
                    av.x = __builtin_fmaf(c.x, fs, av.x);
                    av.y = __builtin_fmaf(c.y, fs, av.y);
                    av.z = __builtin_fmaf(c.z, fs, av.z);
                    av.w = __builtin_fmaf(c.w, fs, av.w);
                }
            }
        }
        if (vec < nv) {
            const float inv = kLowScale / (lsum + 1e-8f);        // kernels.cu:1746, as split_scaled wants it
            o4 = float4{av.x * inv, av.y * inv, av.z * inv, av.w * inv};
        }
        *reinterpret_cast<float4*>(&o_s[vec][k4]) = o4;
    }
    lds_barrier();

    // ---- out[vector][d] = sum_k o[vector][k] R[k][d]; lane group kk owns k in [32kk, 32kk+32).  On fp16 MFMAs: R is
    // exact in fp16, o enters as fp16 value + enlarged rounding remainder, every product is exact in the fp32 accumulators --
    // only the order of the additions differs from the reference's chain (kernels.cu:1769-1775), far inside what the
    // fp16 result resolves -- and the chain is 8 MFMAs instead of 32.
    for (int vt = wave >> 3; back && vt * 16 < nv; vt += kRotGroups) {
        float4_t acc = {0.f, 0.f, 0.f, 0.f}, low = {0.f, 0.f, 0.f, 0.f};
        const float* orow = &o_s[vt * 16 + ln][32 * kg];
#pragma unroll
        for (int st = 0; st < 4; st++) {
            float4 oa = *reinterpret_cast<const float4*>(orow + 8 * st);
            float4 ob = *reinterpret_cast<const float4*>(orow + 8 * st + 4);
            const float ov[8] = {oa.x, oa.y, oa.z, oa.w, ob.x, ob.y, ob.z, ob.w};
            half8_t ahi, alo;
            union { uint16_t u[8]; half8_t h; } bm;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                half_t hi, lo;
                split_scaled(ov[i], hi, lo);
                ahi[i] = hi; alo[i] = lo;
                bm.u[i] = rb[8 * st + i];
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi, bm.h, acc, 0, 0, 0);
            low = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo, bm.h, low, 0, 0, 0);
        }
        // lane holds out[vector vt*16 + 4kk + r][d = 16*dblk + i16]
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int vec = vt * 16 + 4 * kg + r;
            if (vec < nv) {
                const int head = hg * HKW * R + vec;
                const long long col = (long long)head * kHeadDim + 16 * dblk + ln;
                half_t hv = (half_t)__builtin_fmaf(low[r], 1.0f / kLowScale, acc[r]);
                if (a.gate) hv = gated(hv, a.gate[(long long)g * a.gate_stride + col]);
                a.out[(long long)g * a.q_stride + col] = hv;
            }
        }
    }
}

// Two KV heads per wave (PAIR) when the workgroup's heads come in pairs: eight waves, every cache line of the 4-bit
// cache fetched by one instruction.  The workgroup's HKW * (2 + R) vectors must fit its staging slots (a vector per
// 16 threads) and its HKW * R outputs its merge slots (one per 32 threads).
static bool pairs_fit(int bits, int R, int hkw) {
    return (bits == 4 || bits == 2) && (hkw & 1) == 0 && (2 * kPairWaves) % hkw == 0 && hkw * (2 + R) <= 4 * kPairWaves && hkw * R <= 2 * kPairWaves;
}
bool decode_fused_pairs(const AttnArgs& a, int hkw) { return pairs_fit(a.bits, a.num_heads / a.num_kv_heads, hkw); }

// The measured figures behind the estimates below, fitted on MI355X.  One launch or three: 1870 steps of 1 to 256 sequences, 64 to
// 16000 tokens, 1 to 16 KV heads, GQA groups of 1, 2 and 4, both widths, each in every shape of a launch with 1 to 32 shares and in
// three launches, over as many layers as the last cache level does not hold (12 at most).  What counts is the choice, not the single
// estimate: it is the fastest of the forms or within 3 % of it at 90 % of the sizes and within 10 % at 99 %; fitted to 70 % of them,
// at 88 and 99 % of the other 30 %.  (Before the launches' starts and ends were made shorter, with the figures of then and a tile for
// every wave of a share: 71 % and 93 %.)  A rate above what the memory gives is one the last
// cache level helped with.  Every layer in one
// launch: 11100 steps of 4 to 36 layers in each of the four shapes, choice within 3 % of the fastest at 91 %, 10 % at 98 %
// of the sizes that were not fitted to (85 and 95 % before).  64 shares and ragged batches keep figures from earlier fits.
// (A vector of sixteen waves was fitted as 0.222 us, which kept eight KV heads of four query heads from batches of one round: 2 bit, 129 x 231
// tokens 23.0 us with four heads in two rounds, 19.2 with eight. As 0.208, of 4300 sizes 20 change their form, 19 of them to a faster one.)
namespace {
// Batches past 256 sequences, every one of which takes rounds of workgroups: figures of their own, since the first ones, fitted without
// such batches and with rates above the memory's, counted a further round of eight waves too high and one of sixteen too low. Fitted to 2129
// steps of 100 to 1000 sequences of 64 to 16000 tokens, without shares, no rate above the 7.0 TB/s of the best reader: past 256 sequences
// the choice is within 3 % of the fastest form at 97 % of the sizes and within 10 % at 99.5 %, with the first ones at 65 and
// 78 %. us a layer, 4 bit: 300 x 600 tokens, 32 heads over 16 123 -> 94; 300 x 300, 16 over 8 42.1 -> 37.6; 292 x 377, 2 over 2 27.1 -> 20.3.
// (One table for all of them, fitted to 5699 sizes, is 1.6 % faster in the mean, but 15 to 20 % slower at a few sizes of few long sequences.)
constexpr int kFittedBatch = 256;
constexpr PlanConstants kPlanTable[][2] = {{
    {"gfx950", {2.85, 4.16}, {0.178, 0.208}, {9.47, 3.73},
     {{{2.88, 2.11, 2.92}, {1.83, 1.99, 2.39}}, {{3.1, 1.91, 3.32}, {2.65, 2.11, 3.08}}},
     {{{3.39e6, 7.95e6, 9e6, 9e6}, {2.2e6, 4.12e6, 5.74e6, 9e6}},
      {{2.93e6, 5.64e6, 9e6, 8.9e6}, {1.38e6, 3.05e6, 4.88e6, 9e6}}}, {0, 4.39, 6, 2.49, 2.53, 2.59, 4.7},
     {{17.7, 20.2, 20.1}, {18.9, 15.2, 23}}, {{7.02e6, 8e6, 8e6}, {6.97e6, 4.5e6, 3.8e6}}, {{3.08, 1.54, 2.62}, {1.94, 1.8, 1.79}}, {2.39, 2.66}, 0.000465, 16.2, 0.774e-3, 0.629,
     2.5, {8.81, 7.67}, 0.01, {{1.39, 1.42, 1.29}, {1.08, 1.1, 1.09}}, 0.80, {{7.91e6, 8.52e6, 8.41e6}, {7.93e6, 8.41e6, 9.97e6}}, 0.112, false},
    {"gfx950", {9.03, 6.96}, {0.0236, 0.0398}, {6.24, 6.28},
     {{{1.49, 1.72, 2.37}, {0.927, 1.21, 1.54}}, {{2.35, 2.98, 3.01}, {1.99, 1.9, 2.51}}},
     {{{6.7e6, 7e6, 7e6, 6.9e6}, {5.83e6, 5.22e6, 5.37e6, 5.34e6}},
      {{6.11e6, 6.72e6, 6.9e6, 6.66e6}, {4.16e6, 4.58e6, 5.84e6, 5.61e6}}}, {0, 4.39, 6, 2.49, 2.53, 2.59, 4.7},
     {{14.9, 9.65, 6.55}, {12.8, 10.6, 9.25}}, {{5.37e6, 6.72e6, 7e6}, {5.86e6, 5.04e6, 6.7e6}}, {{1.52, 1.75, 1.91}, {1.61, 1.36, 1.26}}, {2.25, 1.54}, 0.00223, 16.2, 0.774e-3, 0.629,
     2.5, {8.81, 7.67}, 0.01, {{1.39, 1.42, 1.29}, {1.08, 1.1, 1.09}}, 0.80, {{7.91e6, 8.52e6, 8.41e6}, {7.93e6, 8.41e6, 9.97e6}}, 0.112, false},
}};
// Where scratch has no room for partials: fitted when both forms took longer, kept with the count of tiles they were fitted with, because
// the line that they draw decides which steps stay in fp32.
constexpr PlanConstants kWithoutRoom = {
    "", {7.45, 9.43}, {0.144, 0.125}, {8.37, 8.19},
    {{{1.88, 2.05, 2.48}, {1.35, 1.48, 1.93}}, {{1.99, 2, 2.81}, {1.69, 1.77, 2.23}}},
    {{{5.02e6, 7.61e6, 7.92e6, 7.69e6}, {3.62e6, 5.33e6, 5.91e6, 6.37e6}}, {{3.39e6, 7.65e6, 6.64e6, 7.18e6}, {1.83e6, 3.96e6, 5.99e6, 5.26e6}}},
    {}, {{19.7, 21.1, 24.9}, {19.1, 20, 22.6}}, {{6.67e6, 6.96e6, 6.32e6}, {5.91e6, 5.02e6, 4.94e6}},
    {{1.16, 1.27, 0.588}, {1.12, 0.672, 1.14}}, {1.74, 1.51}, 0.000277, 0, 0, 0, 0, {}, 0, {}, 0, {}, 0, true};
}  // namespace
const PlanConstants& plan_constants(int G) {
    static const PlanConstants* chosen = nullptr;
    if (!chosen) {
        const PlanConstants* pick = kPlanTable[0];
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) {
            for (const auto& c : kPlanTable)
                if (strstr(prop.gcnArchName, c[0].device)) { pick = c; break; }
        } else {
            (void)hipGetLastError();           // no device (a host-only process asking for the plan): the first entry
        }
        chosen = pick;
    }
    return chosen[G > kFittedBatch ? 1 : 0];
}

const PlanConstants& plan_constants_without_room() { return kWithoutRoom; }

// Microseconds one launch takes: the workgroups run in rounds of one per CU.  A round costs the cube-root sum of its waves'
// tiles of the longest sequence, one after the other, and of its bytes at the rate the chip streams them in this pattern: a
// workgroup with one KV head reads half lines, and unless the batch is a multiple of 8 the other half may be fetched
// again on another XCD.  A share is a sequence of its own of ctx / shares tokens, plus what the hand-over costs at the end.
// (The rates of other batches were fitted before units_by_xcd placed them.  With it, over 700 steps of 2 to 63 sequences, 64 to
// 16000 tokens, six shapes of heads: the choice is the fastest or within 3 % of it at 95 % of the batches of 8 or more that are no
// multiple of 8, at 94 % of the smaller ones and at 96 % of the multiples, 0.5 % from the fastest in the geometric mean of each.)
static int group_index(int R) { return R >= 4 ? 2 : R >= 2 ? 1 : 0; }
static double bytes_per_token(int bits) { return bits == 4 ? 132.0 : 68.0; }       // and KV head: K and V codes and norms
static double cube_sum(double x, double y) { return std::cbrt(x * x * x + y * y * y); }
static int log2_of(int x) { int n = 0; while (x > 1) { x >>= 1; n++; } return n; }

double decode_fused_estimate_us(int G, int num_heads, int Hk, int bits, bool allow_pairs, int hkw, int shares, double ctx, double fill,
                                const PlanConstants& pc) {
    const double cus = compute_units();
    const int R = Hk > 0 ? num_heads / Hk : 1;
    const int w = bits == 4 ? 0 : 1;
    const bool pair = allow_pairs && pairs_fit(bits, R, hkw);
    const int p = pair ? 0 : 1;
    const int parts = (pair ? 2 * kPairWaves : kFusedWaves) / hkw;          // waves that share a head's tiles
    const double units = (double)G * (Hk / hkw) * shares, full = std::floor(units / cus), rest = units - full * cus;
    const double share_tiles = std::ceil(ctx / shares / 32.0);            // fewer than waves: the ones that have a tile are faster
    const double tiles = (share_tiles >= parts || pc.whole_tiles ? std::ceil(share_tiles / parts) : 0.5 + 0.5 * share_tiles / parts) * pc.tile_us[p][w][group_index(R)];
    const double unit_bytes = hkw * bytes_per_token(bits) * ctx / shares * fill / pc.one_bw[G % 8 == 0 ? 0 : 1][w][log2_of(hkw)];
    double us = pc.one_fixed_us[p] + pc.one_vector_us[p] * hkw * (2 + R) + pc.handover_us[log2_of(shares)];
    us += full * cube_sum(tiles, cus * unit_bytes);
    if (rest > 0.0) us += cube_sum(tiles, rest * unit_bytes);
    return us + pc.one_round_us[p] * (full + (rest > 0.0 ? 0.0 : -1.0));
}

// Three launches (rotation, scan, merge) for the same step: what they cost before the scan and after it, the scan's bytes
// at its rate or the tiles of one piece of a sequence, one after the other, and the pieces through the merge.
double decode_three_estimate_us(int G, int num_heads, int Hk, int bits, double ctx, const PlanConstants& pc) {
    const int w = bits == 4 ? 0 : 1, r = group_index(num_heads / Hk);
    const bool odd = (Hk & 1) != 0;
    // as plan_splits and the scans' launches cut it: 512 (sequence, chunk) items, a group of waves each
    int waves = odd ? std::min(Hk, 8) : std::min(Hk / 2, 4);
    while (waves > 1 && (odd ? Hk : Hk / 2) % waves != 0) waves--;
    const int groups = (odd ? 16 : 8) / waves, per_item = odd ? waves : 2 * waves;
    const double base = (double)G * ((Hk + 7) / 8);
    const double pieces = std::max(1.0, std::min({std::floor(512.0 / base), 64.0, std::ceil(ctx / 128.0)}));
    const double rounds = std::ceil(G * pieces * (Hk / per_item) / ((double)compute_units() * groups));
    const double tiles = std::ceil(ctx / pieces / 32.0) * rounds * (odd ? pc.three_tile_odd_us[w] : pc.three_tile_us[w][r]);
    return pc.three_fixed_us[w][r] + cube_sum(tiles, (double)G * Hk * bytes_per_token(bits) * ctx / pc.three_bw[w][r]) +
           pc.three_partial_us * G * num_heads * pieces;
}

// KV heads per workgroup (8, 4, 2 or 1) and shares with the smallest estimate; among equals without shares the larger number
// of heads, whose workgroups read longer contiguous pieces of a cache row.  Shares are only taken while all workgroups
// fit the compute units in one round and a share still has a tile for every fourth wave (for every wave: 4 bit, 4 query heads over
// one KV head, one sequence of 2935 tokens: 16.6 us a layer with 4 shares, 14.2 with 16).
namespace {
std::atomic<int> g_force_hkw{0}, g_force_shares{0};
}  // namespace
void decode_fused_force_shape(int hkw, int shares) { g_force_hkw.store(hkw); g_force_shares.store(shares); }
int decode_fused_forced_hkw() { return g_force_hkw.load(); }

FusedShape decode_fused_shape(int G, int num_heads, int Hk, int bits, bool allow_pairs, int max_shares, double ctx, const PlanConstants& pc) {
    const int R = Hk > 0 ? num_heads / Hk : 1;
    const double cus = compute_units();
    FusedShape best{1, 1, 0.0};
    for (int c = 1; c <= 8; c <<= 1) {
        if (Hk % c != 0) continue;
        const double us = decode_fused_estimate_us(G, num_heads, Hk, bits, allow_pairs, c, 1, ctx, 1.0, pc);
        if (c == 1 || us <= best.us) best = FusedShape{c, 1, us};
    }
    for (int c = 1; c <= 8 && max_shares >= 2; c <<= 1) {
        if (Hk % c != 0) continue;
        const bool pair = allow_pairs && pairs_fit(bits, R, c);
        const int parts = (pair ? 2 * kPairWaves : kFusedWaves) / c;          // waves (parts of the context) per head
        for (int sh = 2; sh <= kMaxShares && sh <= max_shares; sh <<= 1) {
            if ((double)G * (Hk / c) * sh > cus) continue;
            if (ctx < 8.0 * parts * sh) continue;
            const double us = decode_fused_estimate_us(G, num_heads, Hk, bits, allow_pairs, c, sh, ctx, 1.0, pc);
            if (us < best.us) best = FusedShape{c, sh, us};
        }
    }
    const int fh = g_force_hkw.load(), fs = g_force_shares.load();
    if (fh > 0 && Hk % fh == 0) best.hkw = fh;
    if (fs > 0) best.shares = fs <= max_shares && fs <= kMaxShares ? fs : 1;
    return best;
}

bool decode_fused_usable(const AttnArgs& a, const FusedArgs& f) {
    const int R = a.num_kv_heads > 0 ? a.num_heads / a.num_kv_heads : 0;
    if (a.bits != 4 && a.bits != 2) return false;
    if (R != 1 && R != 2 && R != 4) return false;
    if (a.pos_mode != kPosArray || !a.positions || a.G <= 0) return false;
    if (!a.block_table && a.seq_stride_rows <= 0) return false;
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (!al16(a.q) || !al16(f.k_src) || !al16(f.v_src) || !al16(a.rotation)) return false;
    if ((a.q_stride & 7) != 0 || (f.kv_stride & 7) != 0) return false;
    if (!al16(a.k) || !al16(a.v)) return false;
    if ((f.q_weight == nullptr) != (f.k_weight == nullptr) || (f.cos_table == nullptr) != (f.sin_table == nullptr)) return false;
    if (!al16(f.q_weight) || !al16(f.k_weight) || !al16(f.cos_table) || !al16(f.sin_table)) return false;
    if (f.cos_table && !(f.rope_dim == 128 || (f.rope_dim > 0 && f.rope_dim <= 64 && f.rope_dim % 16 == 0))) return false;
    // the scan addresses a tile through a 32-bit buffer offset from the tile's first row: always small
    return true;
}

bool decode_fused_early(int num_heads, int Hk, int bits, bool allow_pairs, int hkw, int shares, int ctx_bound) {
    // when no wave gets more than 8 tiles of 32 tokens (two heads per wave: 16 / hkw parts per head)
    return allow_pairs && pairs_fit(bits, num_heads / Hk, hkw) && shares == 1 && ctx_bound > 0 && ctx_bound <= 8 * 32 * (2 * kPairWaves / hkw);
}

// May the units of a sequence go to one XCD each (sequence g to XCD g % 8)?  Where that needs no more rounds of workgroups than any other
// order, and does not leave two or more XCDs idle while the others stream shared contexts.  MI355X, us per layer, by XCD against
// in any order: 8 over 8 heads, 4 bit, 5 x 16001 tokens 33.7 and 32.9, 6 x 8192 22.7 and 22.2, 2 x 2048 14.8 and 14.3; 7 x 4096 17.5 and
// 18.1.  One workgroup a unit: 5 x 613 12.7 and 13.0.  16 over 8 heads: 11 x 4096 22.6 and 23.3.
static bool units_by_xcd(int G, int units, int shares) {
    const int cus = compute_units(), per_xcd = std::max(1, cus / 8);
    if (shares > 1 && G < 7) return false;
    units *= shares;
    return (G & 7) == 0 || ((long long)(G + 7) / 8 * units + per_xcd - 1) / per_xcd <= ((long long)G * units + cus - 1) / cus;
}

void launch_decode_fused(const AttnArgs& a, const FusedArgs& f_in, hipStream_t s, bool allow_pairs, const StepPlan& plan) {
    FusedArgs f = f_in;
    f.hkw = plan.hkw;
    f.nhg = a.num_kv_heads / f.hkw;
    f.shares = plan.shares;
    f.q_scale = attention_mfma_q_scale(a.bits);
    const int R = a.num_heads / a.num_kv_heads;
    const bool pair = allow_pairs && decode_fused_pairs(a, f.hkw);
    f.by_xcd = units_by_xcd(a.G, a.num_kv_heads / f.hkw, f.shares) ? 1 : 0;
    const dim3 g3((unsigned)((f.by_xcd ? (a.G + 7) / 8 * 8 : a.G) * (a.num_kv_heads / f.hkw) * f.shares)), b3((pair ? kPairWaves : kFusedWaves) * kWave);
    const bool prod = f.q_weight != nullptr || f.cos_table != nullptr;
    const bool early = plan.early;
    note_scan_kernel(pair ? (f.shares > 1 ? "decode_fused_kernel, two KV heads per wave, context shared by workgroups"
                                          : "decode_fused_kernel, two KV heads per wave")
                          : (f.shares > 1 ? "decode_fused_kernel, one KV head per wave, context shared by workgroups"
                                          : "decode_fused_kernel, one KV head per wave"));
#define TW_FUSED_E(RR, BB, PP, EE, SS) \
    do { if (prod) launch_scan_kernel(decode_fused_kernel<RR, BB, true, PP, EE, SS>, g3, b3, s, a, f); \
         else launch_scan_kernel(decode_fused_kernel<RR, BB, false, PP, EE, SS>, g3, b3, s, a, f); } while (0)
#define TW_FUSED(RR, BB, PP) do { if (f.shares > 1) TW_FUSED_E(RR, BB, PP, false, true); else if (PP && early) TW_FUSED_E(RR, BB, PP, PP, false); else TW_FUSED_E(RR, BB, PP, false, false); } while (0)
#define TW_FUSED_R(BB, PP) do { if (R == 1) TW_FUSED(1, BB, PP); else if (R == 2) TW_FUSED(2, BB, PP); else TW_FUSED(4, BB, PP); } while (0)
    if (a.bits == 4) { if (pair) TW_FUSED_R(4, true); else TW_FUSED_R(4, false); }
    else { if (pair) TW_FUSED_R(2, true); else TW_FUSED_R(2, false); }
#undef TW_FUSED_R
#undef TW_FUSED
#undef TW_FUSED_E
}

// The lengths are in device memory, so the line lies by what bounds them: one launch takes as long as its longest sequence, taken as long
// as the bound, and streams 0.55 of it; the three launches take their fixed cost and what a batch of 0.4 of the bound takes, or
// longer.  Paged steps besides must win 3 us by the estimates (the pages' entries cost the longest sequence's waves 5 to 10 % per tile).
// MI355X, 700 random batches each, 1 to 160 sequences of 3 to 12000 tokens, even, ragged and with one long sequence, the room up to
// twice the longest: 1.38 times faster than three launches always in the geometric mean for attention alone, one batch of the 700
// slower (0.95), 4 % from the faster form on average; paged steps 1.35 times, none slower.  2 bit, 16 heads over 8, 27 x 440 tokens: 24.8 us
// in three launches, 12.9 in one; paged 27.5 and 14.0; 13 x 350..2071: 29.5 and 22.8; 18 x 6700 at 4 bit: 45.6 and 63.7.
int decode_fused_mode_shape(int G, int num_heads, int Hk, int bits, int ctx_bound, bool paged) {
    const int R = Hk > 0 ? num_heads / Hk : 0;
    if ((R != 1 && R != 2 && R != 4) || ctx_bound < 1) return 0;
    const int forced = g_force_hkw.load();
    if (forced > 0) return Hk % forced == 0 && pairs_fit(bits, R, forced) ? forced : 0;
    int best = 0;
    double best_us = 0.0;
    for (int hkw = 2; hkw <= 8; hkw <<= 1) {
        if (Hk % hkw != 0 || !pairs_fit(bits, R, hkw)) continue;
        double us = decode_fused_estimate_us(G, num_heads, Hk, bits, true, hkw, 1, ctx_bound, 0.55);
        if (!paged) us -= plan_constants().one_vector_us[0] * 2 * hkw;         // no K and V vectors
        if (best == 0 || us < best_us) { best = hkw; best_us = us; }
    }
    return best > 0 && best_us + (paged ? 3.0 : 0.5) <= decode_three_estimate_us(G, num_heads, Hk, bits, 0.4 * ctx_bound) ? best : 0;
}

void launch_decode_fused_mode(const AttnArgs& a, const FusedArgs& f_in, hipStream_t s, int hkw) {
    FusedArgs f = f_in;
    f.hkw = hkw;
    f.nhg = a.num_kv_heads / hkw;
    f.shares = 1;
    f.q_scale = attention_mfma_q_scale(a.bits);
    const int R = a.num_heads / a.num_kv_heads;
    f.by_xcd = units_by_xcd(a.G, a.num_kv_heads / hkw, 1) ? 1 : 0;
    const dim3 g3((unsigned)((f.by_xcd ? (a.G + 7) / 8 * 8 : a.G) * (a.num_kv_heads / hkw))), b3(kPairWaves * kWave);
    note_scan_kernel(a.block_table ? "decode_fused_kernel, two KV heads per wave, paged" : "decode_fused_kernel, two KV heads per wave, attention alone");
#define TW_MODE(RR, BB) do { if (a.block_table) launch_scan_kernel(decode_fused_kernel<RR, BB, false, true, false, false, kPaged>, g3, b3, s, a, f); \
                             else launch_scan_kernel(decode_fused_kernel<RR, BB, false, true, false, false, kAttend>, g3, b3, s, a, f); } while (0)
#define TW_MODE_R(BB) do { if (R == 1) TW_MODE(1, BB); else if (R == 2) TW_MODE(2, BB); else TW_MODE(4, BB); } while (0)
    if (a.bits == 4) TW_MODE_R(4); else TW_MODE_R(2);
#undef TW_MODE_R
#undef TW_MODE
}

}  // namespace twkv
