// egg_launch.h -- host-side launchers of the kernels, one per .hip translation unit.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <limits.h>
#include "egg_params.h"

hipError_t egg_launch_mlp(const MlpParams &p, bool first, hipStream_t s);
hipError_t egg_launch_qkv(const QkvParams &p, hipStream_t s);
hipError_t egg_launch_attn(const AttnParams &p, hipStream_t s);
hipError_t egg_launch_blocks(const BlocksParams &p, bool *taken, hipStream_t s);      // taken: false where the stages are to be launched one by one
hipError_t egg_launch_head(const HeadParams &p, hipStream_t s);
hipError_t egg_prepare_forward(int H, int head_dim, int T);

struct PlinParams {
    const int8_t *X;        // [members*T][K] natural order
    const int8_t *Wfrag;    // fragment-major copy of W (natural k order) as egg_launch_plinear_swizzle lays it out for (T, K, N)
    int members, T, K, N;
    uint32_t seed; int off_a, off_b, shift, sigma, mask;
    int32_t *Y32; int8_t *Y8;
    int plain;              // the shared-weight product alone: no rank-1 term (the reference's ns == 0 case)
    int own_noise;          // every member draws its own (A, B) with ns = +1 instead of sharing a pair's draw with ns = +-1
    const int8_t *Wblocked; // the canonical blocked matrix: set (with a shape egg_plinear_ws_shape accepts) to run the
                            // W-stationary kernel, which needs no fragment-major copy
};
bool egg_plinear_ws_shape(int K, int N);
bool egg_plinear_small(int members, int T, int K, int N);                 // one launch on the canonical W (egg_linear.hip)
hipError_t egg_launch_plinear_ws(const PlinParams &p, hipStream_t s);      // egg_linear_ws.hip
hipError_t egg_launch_plinear(const PlinParams &p, hipStream_t s);
int egg_plinear_block(int K, int N);
// canonical blocked W -> the layout the kernel chosen for (T, K, N) reads
hipError_t egg_launch_plinear_swizzle(const int8_t *W_blocked, int8_t *W_frag, int T, int K, int N, hipStream_t s);
// canonical blocked [K/4][N][4] -> fragment-major (see egg_device.h); nat = natural k order inside a k-step
hipError_t egg_launch_swizzle(const int8_t *W_blocked, int8_t *W_frag, int K, int N, int B, int nat, hipStream_t s);

// small utility kernels (egg_update.hip)
hipError_t egg_launch_noise_fill(uint32_t seed, uint32_t first, int n, int mask, int8_t *out, hipStream_t s);
hipError_t egg_launch_zero_u64(unsigned long long *p, int64_t n, hipStream_t s);
hipError_t egg_launch_loss_finalize(unsigned long long *acc, int32_t *loss, int first, int count, hipStream_t s);
hipError_t egg_launch_fitness(const int32_t *loss, int32_t *fit, int pairs, hipStream_t s);
// ws: vocab ints (plain sampler) or 2 * vocab ints (d-eggs sampler) of device scratch; token_bytes: 1 or 4
hipError_t egg_launch_sample(const int32_t *logits, const int32_t *exp_lut, int vocab, int bt, uint32_t seed, int t,
                             int *ws, void *out, int token_bytes, hipStream_t s);
hipError_t egg_launch_sample_deggs(const int32_t *logits, const int32_t *exp_lut, int vocab, int bt, uint32_t seed, int t,
                                   const void *tokens, float temp, int min_p_limit, int penalty_int, int *ws, void *out, int token_bytes, hipStream_t s);

// ---- votes and optimizer step (egg_votes.hip)
// the noise of every tensor as shifted windows of one table, see egg_votes.hip
#define EGG_MODEL_SEEDS 920        // seed offsets of the tensors outside the layers and of layer 0 lie below this
#define EGG_LAYER_SEEDS 416        // those of a layer's tensors, above its 1000 * layer
#define EGG_NOISE_FRONT 16         // a row's entry t lies at byte EGG_NOISE_FRONT + t
struct NoiseTable {
    // Rows [0, layer_rows) of ld bytes (a multiple of 128).  Rows from there on belong to the embedding's columns alone, whose
    // window ends in front of entry emb_t: they need emb_ld bytes (a multiple of 128), and as many of them as fit ld share one
    // place -- emb_rows places (a multiple of 128) hold rows layer_rows + i, + emb_rows, + 2 emb_rows ... of place i side by
    // side, so that the rows of a tile of 64 or 128 lie ld apart like all others.
    int8_t *table; size_t ld, emb_ld; int rows, layer_rows, emb_rows, emb_t;
    // masks by pair (pairs_pad, a multiple of 128, of them): 0xff where the fitness is -1 / is not 0, zeros in front and behind.
    // Copy k of four, mask_ld bytes apart, has pair p at byte EGG_NOISE_FRONT + k + p, so that any shift of the pairs finds
    // its masks on a dword.
    int8_t *neg, *nonzero; size_t mask_ld; int pairs_pad;
    int *general;                              // 1: some fitness lies outside {-1, 0, 1}
};
// what a whole step does between its forward and its update: losses and fitness from the loss sums, which go back to
// zero, into device memory and the host's copies.  acc null: the fitness is given.
struct StepEnd { unsigned long long *acc; int32_t *loss, *fit, *h_loss, *h_fit; };
// rows [0, rows) of the entries [t_lo, t_hi) (rows from layer_rows on only below emb_t), the fitness masks, and *counter = 0
// unless it is null
hipError_t egg_launch_noise_table(const NoiseTable &nt, const uint32_t *d_seed, const int32_t *d_fit, const StepEnd &end, int pairs, int mask, int rows,
                                  int t_lo, int t_hi, int n_layers, unsigned long long *counter, hipStream_t s);
struct MatDesc {
    int8_t *W, *frag; float *state;    // canonical weights, their fragment-major copy, optimizer state ({m,v,acc} or Muon's {m,acc})
    float *muon_x;                     // Muon: the matrix's [rows][cols] slot of the workspace, else null
    int64_t offset;                    // in the model blob (and in the overlay's flags)
    int rows, cols, block;             // rows = input dim (k), cols = output dim (n); block: edge of the fragment-major blocks
    int tile_first;                    // number of 64 x 64 tiles of the matrices in front of it in its list
    int t_a, t_b;                      // first table entry of its output-side and input-side noise
    int limit; float lr_scale;         // weights saturate at +-limit: 127 (mgpu.cu:1056-1062), or the configured limit
    int64_t muon_at;                   // the slot's place in the workspace, in floats (last: in front of what k_update reads it costs that 8 spilled registers)
};
// a vector tensor; `first` is the running element count.  flags (adaptive noise overlay), per element, or null
struct VecDesc { int8_t *W; float *state; int n, first, off_a, off_b, seed_base; float lr_scale; int8_t *flags; };
struct UpdLaunch {
    const MatDesc *mat; int n_mat, tiles;          // device array and its number of 64 x 64 tiles
    bool wide;                                     // all sides are multiples of 128
    const VecDesc *vec; int n_vec, vec_total;      // device array; may be empty
    NoiseTable noise;
    const int32_t *fit; int pairs;
    const float *d_lr; float beta1, beta2, eps, wd, muon_momentum;
    unsigned long long *counter, *h_counter;       // changed weights; the host's copy
    int count_of;                      // workgroups that report changes in the whole update
    int32_t *votes_out;                // optional, one matrix: only its votes (blocked order), no update
    int8_t *flags;                     // optional (adaptive noise overlay), laid out like the model blob: a matrix's rows, then its
                                       // cols, set to 1 where a weight changed (de/include/optimizer/adam.cuh:77-83)
};
int egg_update_blocks(const UpdLaunch &p);             // its workgroups
size_t egg_noise_ld(int entries);                      // bytes of a table row that holds so many entries
size_t egg_noise_mask_ld(int pairs_pad);
hipError_t egg_launch_update(const UpdLaunch &p, hipStream_t s);
hipError_t egg_launch_muon_apply(const UpdLaunch &p, float wd, const float *x, hipStream_t s);      // x: the orthogonalised matrices, each at its MatDesc::muon_at
hipError_t egg_launch_frag(const MatDesc *d_mat, int n_mat, int tiles, hipStream_t s);

// adaptive noise overlay (de/src/kernels.cu:61-77): for every entry of every segment, +inc where the flag is set, -dec
// elsewhere, clamped to [-127, 127]; also writes q = clamp(overlay, 0, 64) and clears the flag
struct OvSeg { int offset, count; };
hipError_t egg_launch_overlay_update(int8_t *overlay, int8_t *q, int8_t *flags, const OvSeg *d_segs, int n_segs, int max_count,
                                     int inc, int dec, hipStream_t s);
hipError_t egg_launch_overlay_q(const int8_t *overlay, int8_t *q, int64_t n, hipStream_t s);

// ---- continuation of one sequence (egg_decode.hip)
struct DecodeParams {
    const int8_t *model, *frag;        // the model blob and the fragment-major copies of its matrices; offsets in both:
    uint32_t embedding, emb_bias, ln_init, ln_init_bias, w_up_init, b_up_init, w_dn_init, b_dn_init, ln_1, ln_1_bias, w_q, w_k, w_v, w_o,
        ln_2, ln_2_bias, w_up, b_up, w_dn, b_dn, ln_f, ln_f_bias;
    const int32_t *exp_lut; const int8_t *act_lut; const int32_t *rope_lut;
    int n_layers, head_dim, T, vocab, shift_attn, shift_out, shift_logit, shift_up, shift_dn, rope_bit;
    const uint8_t *tokens;             // the prompt: tokens 0..t_first of token_bytes each
    void *out; int token_bytes;        // token t + 1 goes to out[t + 1]
    int t_first, count;                // positions t_first .. t_first + count - 1 are evaluated and sampled from
    int8_t *kv;                        // [layer][K, V][T][H] slot order: the rows of the positions in front of t_first
    int8_t *kcache, *vcache;           // [H / 16][layer][T][head_dim], [H / 16][layer][T][16]
    int32_t *logits;                   // vocab of them, scratch
    // zero before the first launch: egg_decode_slots messages, the number of the last exchange, and the flag that a wait ran
    // into its bound of wait_limit polls
    unsigned long long *slots; uint32_t *epoch; int *fail; int wait_limit;
    uint32_t seed; int deggs; float temp; int min_p_limit, penalty_int;
};
// a layer's two matrices behind a strip exchange their products' partial sums (egg_decode.hip) instead of their inputs
constexpr bool egg_decode_sums(int H) { return H <= 256; }
constexpr int64_t egg_decode_slots(int H) { return (int64_t)(H / 16) * 67 + (egg_decode_sums(H) ? H / 16 * H : 4 * H) + 8; }
hipError_t egg_prepare_decode(int H, int vocab);      // before the first launch
hipError_t egg_launch_decode(const DecodeParams &p, int H, hipStream_t s);

// ternary-packed matrix weights <-> canonical int8 (n_elems a multiple of 4); *d_bad is set when a weight is not in {-1,0,1}
hipError_t egg_launch_ternary_unpack(const uint8_t *packed, int8_t *dst, int n_elems, hipStream_t s);
hipError_t egg_launch_ternary_pack(const int8_t *src, uint8_t *packed, int n_elems, int *d_bad, hipStream_t s);

// Muon chain (muon_internal.cuh:15-342): momentum + gather (epilogue of the votes), Frobenius normalisation,
// 5 Newton-Schulz iterations with products at float32 accuracy, quantised apply (egg_launch_muon_apply).
struct MuonWork { float *x, *swap, *gram, *bterm, *partials, *norm; };   // x/swap: rows*cols, gram/bterm: K*K, partials: 1024
hipError_t egg_launch_newton_schulz(const MuonWork &w, int rows, int cols, int iters, hipStream_t s);
hipError_t egg_launch_newton_schulz_batched(const MuonWork &w, int rows, int cols, int iters, int batch, hipStream_t s, const float **result);
// ---- device memory to the caller's memory (egg_hostout.hip)
struct HostOut { int8_t *mem = nullptr; size_t slot = 0; hipEvent_t done[8] = {}; };
hipError_t egg_host_out_create(HostOut *o, size_t largest);       // largest: the longest piece that is usually asked for
void egg_host_out_destroy(HostOut *o);
// in stream order; returns when the bytes are in `dst`.  src 16-byte aligned.
hipError_t egg_host_out(HostOut &o, void *dst, const void *src, size_t bytes, hipStream_t s);
// message returned by egg_last_error(NULL) on this thread, for entry points that take no context
void egg_set_thread_error(const char *what);
#define EGG_MAX_DEVICES 64
