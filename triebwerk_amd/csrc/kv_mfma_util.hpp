// kv_mfma_util.hpp -- constants and helpers shared by the MFMA attention kernels
// (kv_attention_mfma.hip: decode scan, kv_prefill_mfma.hip: causal prefill).
#pragma once

#include "kv_common.hpp"
#include "kv_kernels.hpp"

namespace twkv {

constexpr int kGroupWaves = 8;        // KV heads (waves) that walk one item together
constexpr int kMaxWaves = 16;         // waves per workgroup: one workgroup per CU, two groups
constexpr int kMaxBalanceSeqs = 4096; // sequences (blocks) the balanced walk can index (16 KB of LDS)
constexpr int kTableWords = 256 * 64; // 64 KB
constexpr float kNegBig = -1e30f;
// fp16(kAlpha4 * c) has max relative rounding error 1.05e-4 over the 4-bit table
// (exhaustive search over the fp32 values of one octave).
constexpr float kAlpha4 = 19.391284942626953f;
// the same for the 2-bit table: 1.1e-7
constexpr float kAlpha2 = 25.46918296813965f;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kInvSqrtD = 0.08838834764831845f;

__device__ __forceinline__ int seq_pos(const AttnArgs& a, int g) {
    if (a.pos_mode == kPosArray) return a.positions[g];
    if (a.pos_mode == kPosScalar) return a.pos_scalar;
    return g;
}

__device__ __forceinline__ float h2f_bits(uint32_t bits16) {
    union { uint16_t u; half_t h; } cv;
    cv.u = (uint16_t)bits16;
    return (float)cv.h;
}

// Centroid number c % 16 (4 bit) or c % 4 (2 bit) by selections between immediates: the values are in a register while the
// first loads of a kernel are still under way, where a per-lane index into the constant array is one more load to wait for.
template <int BITS>
__host__ __device__ __forceinline__ constexpr float centroid_of(int c) {
    if constexpr (BITS == 4) {
        const int k = (c & 7) ^ ((c & 8) ? 0 : 7);                  // the tables are symmetric
        const float m01 = (k & 1) ? 0.03432f : 0.01135f, m23 = (k & 1) ? 0.08330f : 0.05806f;
        const float m45 = (k & 1) ? 0.14304f : 0.11099f, m67 = (k & 1) ? 0.24155f : 0.18293f;
        const float m = (k & 4) ? ((k & 2) ? m67 : m45) : ((k & 2) ? m23 : m01);
        return (c & 8) ? m : -m;
    } else {
        const float m = ((c ^ (c >> 1)) & 1) ? 0.04003f : 0.13351f;
        return (c & 2) ? m : -m;
    }
}

constexpr bool centroids_agree() {
    for (int c = 0; c < 16; c++)
        if (centroid_of<4>(c) != kCentroids4[c] || centroid_of<2>(c) != kCentroids2[c & 3]) return false;
    return true;
}
static_assert(centroids_agree(), "the selections give the tables' values");

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long long uniform(long long x) {
    return (long long)((unsigned long long)(unsigned)uniform((int)(x >> 32)) << 32 | (unsigned)uniform((int)x));
}

typedef uint32_t uint32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint32x2_t __attribute__((ext_vector_type(2)));

// Buffer descriptor over [base, base + bytes).  Every input is forced into scalar
// registers: a descriptor held in vector registers makes each load a serialising loop.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const char* base, int bytes) {
    uint64_t p = reinterpret_cast<uint64_t>(base);
    uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32));
    char* q = reinterpret_cast<char*>(((uint64_t)hi << 32) | lo);
    return __builtin_amdgcn_make_buffer_rsrc(q, 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// Cache policy (the aux operand of the raw buffer loads) of the loads that stream the cache: bit 1 = nt,
// "non-temporal".  A decode scan reads every cache byte once per launch and a layer's cache is far larger than
// any cache level, so nothing is gained by keeping the lines; with the hint a launch that only reads 554 MB
// takes 78-82 us instead of 88-90 us on MI355X (7.0 instead of 6.2 TB/s).
// Only for lines that one load instruction of one wave covers in full: a line touched by two instructions (two
// waves, or two half-line loads of one wave) is fetched twice, and the launch gets slower than without the hint.
constexpr int kStreamCodes = 2;
constexpr int kDeviceScope = 16;               // the sc1 bit of a raw buffer access: device scope
// the norm rows (16 bytes per token for 8 heads) are shared by the workgroups of a sequence: kept in the caches
constexpr int kStreamNorms = 0;

// The forms of the two flash prefill kernels, and the rule that picks one.  A workgroup of `waves` waves in `groups` groups takes
// 16 * nq * (waves / groups) / R query tokens of one KV head; the groups take turns with the context's tiles.
// With causal rows the last block's chain of tiles is twice the average, so what a launch takes is the larger of its longest
// chain (at the pace of a workgroup that has its compute unit for itself) and of the steps all workgroups make (at the pace of
// a full compute unit): estimate = fixed + max(alone * longest, loaded * steps per unit) + per_wg * workgroups per unit
//                                 + both * min(longest, steps per unit), in us.
// Measured on MI355X (256 compute units) as launches back to back in a graph, 2 to 32 heads over 1 to 16 KV heads.  fp16: fitted
// to all forms at 371 sizes of 1 to 16384 tokens; the choice is the fastest form or within 3 % of it at 362, within 10 % at all
// but 2 (18 %: 8500 tokens, 16 heads over 4).  (With figures fitted from 31 tokens up, launch gaps in them, prompts up to 80
// tokens took the eight-wave forms: 16 heads over 8, 33 tokens 5.8 us against 4.7 in four waves; and 3000 tokens 66 us
// against 53.)  The compressed kernel's figures are from 66 launches of 33 to 5500 tokens at 4 and 2 bit, 8, 16 and 32 heads
// over 8; at 410 sizes of 1 to 8192 tokens and 1 to 16 KV heads the choice is the fastest form or within 3 % at 361, within
// 7 % at all.
struct PrefillForm { int id, waves, nq, groups; double fixed, alone, loaded, per_wg, both; };
struct PrefillChoice { int id, waves, nq, groups; bool mirror; int blocks; };

inline PrefillChoice choose_prefill_form(const PrefillForm* forms, int nforms, double mirror_fill, int T, int R, int num_kv_heads, int forced) {
    const double cus = compute_units();
    PrefillChoice best{};
    double best_us = 0.0;
    for (int i = 0; i < nforms; i++) {
        const PrefillForm& f = forms[i];
        const int tpw = 16 * f.nq * (f.waves / f.groups) / R, blocks = (T + tpw - 1) / tpw;
        const double longest = ((T + 31) / 32 + f.groups - 1) / f.groups;
        const double shortest = (tpw + 31) / 32 > f.groups ? (double)((tpw + 31) / 32) / f.groups : 1.0;
        const double per_unit = blocks * (longest + shortest) * 0.5 * num_kv_heads / cus;
        double us = f.fixed + (f.alone * longest > f.loaded * per_unit ? f.alone * longest : f.loaded * per_unit) +
                    f.per_wg * blocks * num_kv_heads / cus + f.both * (longest < per_unit ? longest : per_unit);
        // Blocks in pairs, each with its mirror image from the other end, when the pairs fill whole rounds of one workgroup
        // per compute unit (a single round: by mirror_fill): every workgroup then does the same work and none starts late
        // (8192 tokens: 0.266 against 0.271 ms on the fp16 cache, 0.498 against 0.511 at 4 bit; 6400 tokens, a round 3/4 full: 0.186
        // against 0.192, but 0.392 against 0.364 at 4 bit).  A pair too many costs a second round (8200 tokens: 0.310 against
        // 0.275 and 0.605 against 0.524), so otherwise the blocks are workgroups of their own, longest first: a compute
        // unit that is done takes the next shorter one, which pairs them just as well.
        const double pairs = (double)((blocks + 1) / 2) * num_kv_heads, rounds = (double)(long long)((pairs + cus - 1) / cus);
        bool mirror = f.waves == 8 && f.groups == 1 && pairs >= (rounds > 1.0 ? 0.97 : mirror_fill) * rounds * cus;
        if (mirror) us *= 0.97;
        // forced by a test: 5 and 6 in pairs, 7 and 8 the same forms unpaired, 1 to 3 (never in pairs) as they are
        if (f.id == forced || f.id + 2 == forced) {
            if (f.id >= 5) { us = -1.0; mirror = f.id == forced; }
            else if (f.id == forced) us = -1.0;
        }
        if (i == 0 || us < best_us) { best_us = us; best = PrefillChoice{f.id, f.waves, f.nq, f.groups, mirror, blocks}; }
    }
    return best;
}

// The dequantization table of the MFMA scans, built by the nthreads threads of a workgroup: entry e (a cache byte)
// fills 256 bytes with replicas of its centroids as fp16 -- 4 bit: 64 replicas of (low code, high code); 2 bit: 32
// replicas of the byte's four codes, in their own order (NATURAL) or as 0, 2, 1, 3.  nthreads: whole waves.  The four entries a
// wave fills in a round share their upper four bits and start at a multiple of four: the upper centroids come out of a register by
// v_readlane (lane c holds centroid c, scaled), the lower ones out of four shuffles made once.  (Indexing the constant arrays with
// a per-lane index is a dependent memory load per look-up, a shuffle per entry and round a trip through LDS each.)
template <int BITS, bool NATURAL>
__device__ __forceinline__ void build_centroid_table(uint32_t* tab_s, float alpha, int tid, int nthreads) {
    const int lane = tid & 63, wave = uniform(tid >> 6), nwaves = nthreads >> 6;
    const float cent_lane = alpha * centroid_of<BITS>(lane);
    auto cent_of = [&](int c) -> half_t {                    // c uniform over the wave
        return (half_t)__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cent_lane), c));
    };
    if constexpr (BITS == 4) {
        half_t lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) lo[j] = (half_t)__shfl(cent_lane, 4 * j + (lane >> 4), 64);
        for (int e = 4 * wave; e < 256; e += 4 * nwaves) {   // this thread: entry e + lane / 16, 16 bytes of it
            const int j = (e >> 2) & 3;
            half2_t p = {j == 0 ? lo[0] : j == 1 ? lo[1] : j == 2 ? lo[2] : lo[3], cent_of(e >> 4)};
            const uint32_t w = *reinterpret_cast<uint32_t*>(&p);
            *reinterpret_cast<uint4*>(&tab_s[e * 64 + lane * 4]) = uint4{w, w, w, w};
        }
    } else {
        const half_t c0 = (half_t)__shfl(cent_lane, lane >> 4, 64);
        for (int e = 4 * wave; e < 256; e += 4 * nwaves) {
            const half_t c1 = cent_of((e >> 2) & 3), c2 = cent_of((e >> 4) & 3), c3 = cent_of(e >> 6);
            half2_t p0 = {c0, NATURAL ? c1 : c2}, p1 = {NATURAL ? c2 : c1, c3};
            const uint32_t w0 = *reinterpret_cast<uint32_t*>(&p0), w1 = *reinterpret_cast<uint32_t*>(&p1);
            *reinterpret_cast<uint4*>(&tab_s[e * 64 + lane * 4]) = uint4{w0, w1, w0, w1};
        }
    }
}

}  // namespace twkv
