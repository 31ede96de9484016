// kv_kernels.hpp -- internal launch interface between the C ABI (kv_capi.hip)
// and the kernel files.  Nothing here is exported.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stdint.h>

#include "kv_common.hpp"

struct tw_layer_step_args;          // include/triebwerk_kv.h

namespace twkv {

// ---------------------------------------------------------------- timing the context-scanning kernel
// When the profiler is on, kv_capi.hip hands the scan launch a pair of events; the launch attaches them
// to the kernel itself (start = the kernel begins, stop = it ends), so their distance is the kernel's
// duration without the gaps an event recorded before and after a launch would add.
extern thread_local hipEvent_t t_scan_start;
extern thread_local hipEvent_t t_scan_stop;
// Name of the kernel the last attention launch of this process used for the context (tw_kv_debug_last_scan_kernel):
// every launch function below records its own.
extern const char* volatile g_last_scan_kernel;
inline void note_scan_kernel(const char* name) { g_last_scan_kernel = name; }
template <typename... Args, typename F = void (*)(Args...)>
inline void launch_scan_kernel(F kernel, dim3 grid, dim3 block, hipStream_t s, Args... args) {
    if (t_scan_start) hipExtLaunchKernelGGL(kernel, grid, block, 0, s, t_scan_start, t_scan_stop, 0, args...);
    else hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
}

// ---------------------------------------------------------------- append
struct QuantArgs {
    // One or two streams (K, V) quantized by the same launch.
    uint8_t* codes[2];
    half_t* norms[2];
    const half_t* src[2];   // (nrows, kv_dim) fp16
    int nstreams;
    const half_t* rotation; // (128,128) fp16 row major
    const int* positions;   // device int32[nrows]
    const int* block_table; // NULL = contiguous cache
    int bt_stride;
    long long seq_stride_rows;  // max_seq_len for the contiguous batch layout
    int token_list;         // 1: row r goes to cache row positions[r] of sequence 0
    int nrows;              // G, or num_tokens
    int num_kv_heads;
    int kv_dim;
};

void launch_kv_write(half_t* ck, half_t* cv, const half_t* k, const half_t* v,
                     const int* positions, const int* block_table, int bt_stride,
                     long long seq_stride_rows, int G, int kv_dim, hipStream_t s);
void launch_turbo_quantize(const QuantArgs& a, int bits, hipStream_t s);
void launch_increment(int* positions, int G, hipStream_t s);

// Rows [0, T) of sequence `src` copied to sequences [dst_begin, dst_end) (src itself skipped) in up to four
// arrays that are laid out (sequence, row, ...): bytes = T * row bytes, seq_bytes = rows per sequence * row bytes.
// The same for `layers` layers whose arrays lie layer_bytes apart (one layer: any distance).
struct BroadcastArgs {
    char* base[4];
    size_t seq_bytes[4];
    size_t bytes[4];
    int layers;
    size_t layer_bytes;
    int narrays;
    int src, dst_begin, dst_end;
};
// checks the range, launches and notes what went wrong in the library's error state under fn's name (kv_capi.hip);
// 0, -1 for a bad range, -2 for a launch that failed
int broadcast_rows(const char* fn, const BroadcastArgs& a, hipStream_t s);
void launch_broadcast_rows(const BroadcastArgs& a, hipStream_t s);

// ---------------------------------------------------------------- producers of q and k (kv_producer.hip)
struct ProducerArgs {
    half_t* q;               // (rows, q_stride), transformed in place
    half_t* k;               // (rows, kv_stride)
    half_t* v;               // write_cache only
    long long q_stride, kv_stride;
    int rows, num_heads, num_kv_heads;
    int norm;                // per-head RMSNorm with q_weight / k_weight
    const half_t* q_weight;  // (128)
    const half_t* k_weight;
    float eps;
    int biased;              // weight + 1
    const half_t* cos_table; // NULL: no rotation; (positions, rope_dim / 2)
    const half_t* sin_table;
    int rope_dim;
    int single_order;        // operand order of the single-sequence rope kernel
    const int* positions;    // device int32[rows], or NULL: pos_scalar
    int pos_scalar;
    int write_cache;         // K (transformed) and V rows go to their fp16 cache rows instead of back
    half_t* cache_k;
    half_t* cache_v;
    int kv_dim;              // halves per cache row
    const int* block_table;
    int bt_stride;
    long long seq_stride_rows;
};
// Several layers in one launch: what layer l's pointers lie further on, l times each -- q and out, k and v in halves, the cache arrays
// in bytes, norm weights kHeadDim halves; workspace blocks are those of sequences l * G + g.  (A parameter of its own: the kernels
// without it keep their short argument blocks.)
struct LayerStrides {
    int layers = 1;
    long long q = 0, kv = 0, cache = 0;
};
void launch_producer(const ProducerArgs& a, hipStream_t s, const LayerStrides& layers = LayerStrides{});
bool producer_rows_usable(const ProducerArgs& a);   // pointers and strides admit 16-byte accesses

// Compressed append of many rows, optionally with the producers of q and k (kv_append_tokens.hip)
struct AppendTokensArgs {
    ProducerArgs p;          // p.k, p.v: the rows of streams 0 and 1; p.norm / p.cos_table: q and k transformed in place
    int nstreams;
    uint8_t* codes[2];
    half_t* norms[2];
    const half_t* rotation;
    long long seq_stride_rows;   // row r goes to cache row r * seq_stride_rows + positions[r]
    float row_norm;              // as FusedArgs has it
    int nper, kv_blocks, q_blocks, chains;   // launch_append_tokens fills these in
};
bool append_tokens_usable(const AppendTokensArgs& a);
// While one of these lives the calls of this thread have the engine's rotation, whose rows are of norm 1: the kernels need not measure them
// (FusedArgs::row_norm).
constexpr float kUnitRows = 1.001f;
struct KnownRotation {
    KnownRotation();
    ~KnownRotation();
};
void launch_append_tokens(const AppendTokensArgs& a, int bits, hipStream_t s);
// data[r][i] = half(data[r][i] / (1 + exp(-gate[r][i]))), rows of `dim` halves with their own strides
void launch_sigmoid_gate(half_t* data, long long data_stride, const half_t* gate, long long gate_stride, int dim,
                         int rows, hipStream_t s);

// ---------------------------------------------------------------- rotation on the matrix cores
// test hook (tw_kv_debug_rotation_sums)
void launch_rotation_sums(const half_t* x, int n, const half_t* rotation, float* sums, float* row_norms, hipStream_t s);
struct RotArgs {
    // up to 3 segments: K rows, V rows (quantize), Q rows (rotate only); each 64 bytes, one scalar load of a kernel
    struct alignas(64) Segment {
        const half_t* src;       // fp16 source, row r at src + r * stride
        long long stride;        // halves per source row
        uint8_t* codes;
        half_t* norms;
        const half_t* weight;    // optional producers applied to the vectors before anything else (kv_producer.hip has the rules): RMSNorm weight (128), NULL = none
        int heads;               // head vectors per source row
        int nvec;                // rows * heads
        int kind;                // 0 = quantize into the cache, 1 = query rotation
        int rope;                // rotate with the tables below at positions[row]
        int units;               // work units = ceil(tiles / nper) * 8 (launch_rotate fills this in)
    } seg[3];
    int nseg;
    int nper;                    // tiles of 16 vectors a wave walks (launch_rotate fills this in)
    const half_t* rotation;
    const int* positions;
    const int* block_table;
    int bt_stride;
    long long seq_stride_rows;
    int token_list;              // 1: source row r goes to cache row positions[r] of sequence 0
    int num_kv_heads;
    float* qrot;                 // query output: vector v at qrot + v * qrot_stride (fp32)
    int q_operands;              // instead of the floats 128 halves of fp16 values and 128 of what rounding left over (attention_takes_operands)
    long long qrot_stride;
    float q_scale;
    // producers of the segments that have them
    float eps;
    int biased;
    const half_t* cos_table;     // (positions, rope_dim / 2)
    const half_t* sin_table;
    int rope_dim;                // multiple of 16
};

void launch_rotate(const RotArgs& a, int bits, hipStream_t s);

// ---------------------------------------------------------------- attention
enum PosMode { kPosArray = 0, kPosScalar = 1, kPosIota = 2 };

struct AttnArgs {
    const half_t* q;        // (G, q_stride)
    half_t* out;            // (G, q_stride)
    int q_stride;
    const void* k;          // fp16 rows (kv_bits 0) or packed codes
    const void* v;
    const half_t* k_norms;  // compressed only: (rows, num_kv_heads)
    const half_t* v_norms;
    const half_t* rotation; // compressed only
    const int* positions;   // kPosArray
    int pos_scalar;         // kPosScalar
    int pos_mode;           // kPosIota: sequence g attends rows 0..g (causal prefill)
    const int* block_table; // NULL = contiguous
    int bt_stride;
    long long seq_stride_rows;  // msl (batch), 0 (single sequence / prefill)
    int G, num_heads, num_kv_heads;
    int bits;               // 0, 2, 4
    float* ws;              // split workspace: per (g, head) block, nsplit partials then q_rot
    long long ws_stride;    // floats per (g, head) block
    float* qrot;            // ws + offset of q_rot inside a block (128 floats), or NULL
    int nsplit;             // >= 1; 1 = no workspace, one workgroup walks the sequence
    int force_merge;        // the scan kernel wrote partials even though nsplit == 1
    int m_log2;             // partial maxima are in base-2 units
    int balance;            // MFMA scan: may cut the batch by tiles instead of by sequence (ragged lengths)
    int max_slots;          // partials the workspace holds per (sequence, head): >= nsplit
    unsigned* tickets;      // fp16 step: G * num_kv_heads words, zero before and after a launch, or NULL
    int slots_from_ws;      // merge: the spare word of partial 0 holds the number of partials (0: even chunks)
    int even_chunks;        // the chunks are the fp16 whole-row scan's (even_chunk_range), not chunk_range's
    // optional output gate (gated attention, kernels.cu:2987-2995): out = half(float(half(out)) * sigmoid(gate))
    const half_t* gate;     // row g at gate + g * gate_stride, laid out like a row of out; NULL = none
    long long gate_stride;
    // fp16 cache, batch decode: the K and V rows of the new token (position positions[g]).  The scan takes them
    // from here instead of the cache and one workgroup per (sequence, KV head) stores them there, which makes
    // the append part of the attention launch (kv_cache_write_batch_kernel, kernels.cu:964-977).  NULL = none.
    const half_t* k_new;    // (G, kv_new_stride)
    const half_t* v_new;
    long long kv_new_stride;
};

constexpr int kPartialFloats = kHeadDim + 4;  // acc[128], running max, running sum, 2 pad (16-byte rows)

void launch_attention_valu(const AttnArgs& a, hipStream_t s);
bool attention_valu_merges(const AttnArgs& a);     // its chunks merge themselves (AttnArgs::tickets): no launch_attention_merge
// fp16 cache: will launch_attention_valu run the kernel whose waves read whole rows (eight KV heads)?  Its workgroups
// have eight waves that share one chunk, so the split planner gives it more and smaller chunks.
bool attention_rows_usable(const AttnArgs& a);
int attention_rows_groups(const AttnArgs& a);      // workgroups per (sequence, chunk)
void launch_attention_rows_layers(const AttnArgs& a, const LayerStrides& layers, hipStream_t s);   // nsplit even chunks of every sequence
bool attention_rows_balances(const AttnArgs& a);   // may cut a ragged batch by tokens instead (needs max_slots set)
void launch_attention_merge(const AttnArgs& a, hipStream_t s, const LayerStrides& layers = LayerStrides{});
bool launch_merge_rotate(const AttnArgs& a, hipStream_t s);   // MFMA merge + rotate-back; false = not applicable
// MFMA path, two steps so that the scan kernel can be timed alone:
// prepare = shape check + query rotation (false = shape not covered), then the scan.
bool prepare_attention_mfma(AttnArgs& a, hipStream_t s, bool rotate_query);
float attention_mfma_q_scale(int bits);
bool launch_attention_mfma_scan(const AttnArgs& a, hipStream_t s);   // true: the output is finished, no merge
// One decode step of a layer in one launch (kv_decode_fused.hip): append the new K and V rows, rotate the
// query, scan, merge and rotate back.  AttnArgs as for the batch decode over the contiguous compressed
// cache (positions array; no workspace needed), plus the rows to append and the cache as writable pointers.
struct FusedArgs {
    const half_t* k_src;    // (G, kv_stride) fp16 rows of the new token
    const half_t* v_src;
    long long kv_stride;
    uint8_t* k_codes;       // the arrays AttnArgs::k, v, k_norms, v_norms point at
    uint8_t* v_codes;
    half_t* k_norms;
    half_t* v_norms;
    int hkw, nhg;           // KV heads per workgroup, workgroups for all of them (launch_decode_fused fills these in)
    int by_xcd;             // sequence g's workgroups on XCD g % 8 (likewise)
    float q_scale;          // likewise
    float row_norm;         // an upper bound on the norms of R's rows; 0: the kernel finds one
    // A unit's context shared by several workgroups, for batches whose units alone leave compute units idle:
    int shares;             // a power of two up to 64 (launch_decode_fused fills this in; > 1 only with the two below)
    float* share_ws;        // G * num_heads * shares * (kHeadDim + 4) floats for the shares' unnormalised sums
    unsigned* tickets;      // one word per (sequence, KV head): zero before the first launch, left zero by every launch
    // optional producers of q and k applied on the way in, as RotArgs has them (V rows stay as they are)
    const half_t* q_weight; // per-head RMSNorm weights (128); both or neither
    const half_t* k_weight;
    float eps;
    int biased;
    const half_t* cos_table; // (positions, rope_dim / 2); both or neither
    const half_t* sin_table;
    int rope_dim;            // 128, or a multiple of 16 up to 64
};
// Everything the choice between the forms of a decode step rests on, in one place: rates and fixed costs measured on
// the device named, looked up once per process by the current device's name (plan_constants()).  A device that is
// not in the table gets the first entry's figures scaled by its own number of compute units only where the estimates
// use that number; tests/test_gpu_plan.py checks on the GPU at hand that the automatic choice is the faster form.
struct PlanConstants {
    const char* device;         // substring of hipDeviceProp_t::gcnArchName
    // one launch; first index of the pairs: waves that scan two KV heads, one head
    double one_fixed_us[2];     // prologue, first tile, epilogue, launch and drain
    double one_vector_us[2];    // more for each vector of the new token that a workgroup has
    double one_round_us[2];     // each further round of workgroups
    double tile_us[2][2][3];    // a wave's tile of 32 tokens, the waves of a compute unit side by side: [4 bit, 2 bit][GQA group 1, 2, 4]
    double one_bw[2][2][4];     // bytes per us the whole chip streams: [batch a multiple of 8, any other][4 bit, 2 bit][1, 2, 4, 8 KV heads per workgroup]
    double handover_us[7];      // shares' sums through memory, by log2(shares)
    // three launches (rotation, scan, merge): [4 bit, 2 bit][GQA group 1, 2, 4]
    double three_fixed_us[2][3];   // the launches, the scan's start and end
    double three_bw[2][3];         // bytes per us of the scan
    double three_tile_us[2][3];    // a wave's tile of 32 tokens
    double three_tile_odd_us[2];   // the same for an odd number of KV heads (one head per wave): [4 bit, 2 bit]
    double three_partial_us;       // a piece of a (sequence, head) through memory and the merge
    // the walk of a ragged batch: fixed, per token of its longest sequence, and this share of the estimate for the mean length
    double ragged_us, ragged_token_us, ragged_mean_share;
    // every layer in one launch
    double layers_launch_us;
    double layers_unit_us[2], layers_vector_us;  // a workgroup's start and end: [4 waves, 8 waves], and for each of its vectors
    double layers_tile_us[2][3];   // a wave's tile, two waves a SIMD: [4 bit, 2 bit][GQA group 1, 2, 4]
    double layers_alone;           // this share of it for a workgroup of four waves that has its compute unit for itself
    double layers_bw[2][3];        // bytes per us: [4 bit, 2 bit][2, 4, 8 KV heads per workgroup]
    double layers_both;            // this share of the smaller of (longest unit, all units) on top of the larger
    bool whole_tiles;              // fitted with a whole tile for each wave of a unit that has fewer tiles than waves
};
const PlanConstants& plan_constants(int G = 0);          // of the device; batches past 256 sequences have figures of their own
const PlanConstants& plan_constants_without_room();      // the line between one launch and three where scratch has no room for partials
bool decode_fused_usable(const AttnArgs& a, const FusedArgs& f);
// estimated microseconds of one launch with hkw KV heads per workgroup and `shares` workgroups per sequence and head group,
// the longest sequence at ctx tokens and the mean one at fill * ctx
double decode_fused_estimate_us(int G, int num_heads, int num_kv_heads, int bits, bool allow_pairs, int hkw, int shares, double ctx,
                                double fill, const PlanConstants& pc = plan_constants());
// estimated microseconds of the same step as three launches (rotation, scan, merge), all sequences at ctx tokens
double decode_three_estimate_us(int G, int num_heads, int num_kv_heads, int bits, double ctx, const PlanConstants& pc = plan_constants());
// The launch's shape when a unit's context may be shared by up to max_shares workgroups (1: the caller has no tickets
// or no room for the shares' sums): KV heads per workgroup, shares, and the estimate for sequences of ctx tokens.
struct FusedShape { int hkw, shares; double us; };
FusedShape decode_fused_shape(int G, int num_heads, int num_kv_heads, int bits, bool allow_pairs, int max_shares, double ctx,
                              const PlanConstants& pc = plan_constants());
// test hook (tw_kv_debug_set_fused_shape): force hkw and / or shares (0 = automatic)
void decode_fused_force_shape(int hkw, int shares);
int decode_fused_forced_hkw();
// whether the waves ask for their first tile in the prologue (allow_pairs as below; ctx_bound: no sequence is longer)
bool decode_fused_early(int num_heads, int num_kv_heads, int bits, bool allow_pairs, int hkw, int shares, int ctx_bound);
// How a compressed decode step runs: as three launches, or as one of this shape.  decode_step_plan (kv_capi.hip) is
// what both the launch and the engine go by; a captured step holds the launches of exactly one such plan.
struct StepPlan {
    bool one;
    int hkw, shares;
    bool early;
    // The step of an engine whose layers go together (layers > 1): all of them in one launch of this shape (kv_decode_layers.hip)
    // instead, KV heads and waves per workgroup.  The fields above stay what a layer by itself would take.
    // (fp16 cache: in pieces of each sequence's context)
    int layers, layers_hkw, layers_waves, layers_pieces;
    bool operator==(const StepPlan& o) const {                         // the same launches
        if (layers != o.layers) return false;
        if (layers > 1) return layers_hkw == o.layers_hkw && layers_waves == o.layers_waves && layers_pieces == o.layers_pieces;
        return one == o.one && hkw == o.hkw && shares == o.shares && early == o.early;
    }
};
// layers: how many the caller can hand over at once (1: a layer by itself)
StepPlan decode_step_plan(int G, int num_heads, int num_kv_heads, int bits, int max_seq_len, int ctx_min, int ctx_max, double ctx_mean, bool can_share,
                          int layers = 1);
// tw_layer_attention_step for a caller that knows the mean of positions + 1 as well (0: unknown)
void layer_attention_step(const tw_layer_step_args* p, double ctx_mean, hipStream_t s);
// Every layer of a compressed decode step in one launch (kv_decode_layers.hip).  Pointers are layer 0's; layer l's lie l times
// these distances further on: q and out q_layer halves, k and v kv_layer halves, the four cache arrays cache_layer bytes
// (even), the norm weights kHeadDim halves.
struct LayersArgs {
    const half_t *q, *k, *v;    // (G, q_stride), (G, kv_stride)
    half_t* out;
    uint8_t *k_codes, *v_codes;
    half_t *k_norms, *v_norms;
    const half_t* rotation;     // (128, 128)
    const uint4* rot_ops;       // order_rotation's 64 KB
    int* positions;             // one token on when the launch is done
    unsigned* tickets;          // G words, zero before the launch and left zero
    int layers, G, num_kv_heads;
    int nhg;                    // num_kv_heads / the launch's heads per workgroup
    uint32_t g_magic;           // ceil(2^32 / G) where (layers * G + 8) * G < 2^32: a division by multiplication; 0 elsewhere
    int q_stride, kv_stride;
    long long q_layer, kv_layer, cache_layer;
    long long seq_stride_rows;
    float q_scale;
    const half_t *q_weight, *k_weight;     // as FusedArgs has them
    float eps;
    int biased;
    const half_t *cos_table, *sin_table;
    int rope_dim;
};
void order_rotation(const uint16_t* rot, uint16_t* ops);       // 128 x 128 halves -> 2 x 128 x 128 halves, host
void launch_decode_layers(const LayersArgs& a, int num_heads, int bits, int hkw, int waves, hipStream_t s);
// The shape of that launch with the smallest estimate (hkw 0: none serves these heads), for contexts up to ctx_max, ctx_mean on average.
struct LayersShape { int hkw, waves; double us; };
LayersShape decode_layers_shape(int layers, int G, int num_heads, int num_kv_heads, int bits, double ctx_max, double ctx_mean);
// The distances above for tw_layer_step_args of layer 0 (no gate).
struct StepLayers {
    int n;
    long long q, kv, cache;
    const void* rot_ops;         // compressed
    float* ws;                   // fp16: n * G * num_heads * pieces * kPartialFloats floats (pieces > 1)
};
// fp16 cache: pieces every sequence's context is cut into when all layers go together, with ws_floats of workspace (0: not together)
int rows_layers_most_pieces(int layers, int G, int num_heads, int num_kv_heads);     // the workspace is made for
int rows_layers_pieces(int layers, int G, int num_heads, int num_kv_heads, int max_seq_len, double ctx_max, double ctx_mean, size_t ws_floats);
// Whether the buffers admit it (a plan with layers > 1 is for those that do)
bool layers_attention_usable(const tw_layer_step_args* p, const StepLayers& layers);
// (again: the launches of a fixed step after its first time, which tw_kv_decode_fused_launches counts no more than a graph's replays)
void layers_attention_step(const tw_layer_step_args* p, const StepLayers& layers, const StepPlan& plan, hipStream_t s, bool again);
// allow_pairs: the kernel whose waves scan two KV heads each, where the shape admits it (false: one head per wave)
void launch_decode_fused(const AttnArgs& a, const FusedArgs& f, hipStream_t s, bool allow_pairs, const StepPlan& plan);
// the pair kernel (hkw KV heads a workgroup, no shares, no producers) for attention alone, or for the step over the paged cache
// (a.block_table)
void launch_decode_fused_mode(const AttnArgs& a, const FusedArgs& f, hipStream_t s, int hkw);
// KV heads per workgroup of that launch where it is the faster form for sequences of at most ctx_bound tokens; 0: the three launches are
int decode_fused_mode_shape(int G, int num_heads, int num_kv_heads, int bits, int ctx_bound, bool paged);
// causal prefill with blocks of query tokens per wave (kv_prefill_mfma.hip); same workspace and merge
bool prefill_mfma_usable(const AttnArgs& a);
void launch_prefill_mfma_scan(const AttnArgs& a, hipStream_t s);
// causal prefill over the fp16 cache on the matrix cores (kv_prefill_f16_mfma.hip); writes `out` directly
bool prefill_f16_mfma_usable(const AttnArgs& a);
// form: 0 = chosen from the prompt length, else as tw_kv_debug_set_prefill_form (4: taken as 0 here)
void launch_prefill_f16_mfma(const AttnArgs& a, hipStream_t s, int form);
// causal prefill over the compressed cache with tiles expanded once per workgroup (kv_prefill_tq_mfma.hip);
// one launch, no workspace; forms as for launch_prefill_f16_mfma
bool prefill_tq_mfma_usable(const AttnArgs& a);
void launch_prefill_tq_mfma(const AttnArgs& a, hipStream_t s, int form);
// test hook (tw_kv_debug_set_prefill_form)
int prefill_form();
// 4-bit decode scan whose waves take two KV heads each and read whole cache lines (kv_attention_pair.hip); same
// workspace, partials and merge as attention_mfma_kernel
bool attention_pair_usable(const AttnArgs& a);
// will launch_attention_mfma_scan run it: then the rotated queries are left as operands
bool attention_takes_operands(const AttnArgs& a);
void launch_attention_pair_scan(const AttnArgs& a, hipStream_t s);
// test hook (tw_kv_debug_set_attention_variant): 0 automatic, 1 vector-ALU kernels, 2 MFMA kernels, 3 MFMA kernels
// with one KV head per wave also where the 4-bit scan would give a wave two
int attention_variant();

}  // namespace twkv
