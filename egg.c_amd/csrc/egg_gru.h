// egg_gru.h -- what the two ways of evaluating full_trained_egg.c ("egg.c") share: egg_gru.hip (one persistent workgroup per
// 32 members; noise, update, C ABI) and egg_gru_pipe.hip (the pipeline over layers and chunks of tokens).
#pragma once
#include "egg_device.h"
#include "egg_launch.h"

struct GruMat {            // one weight matrix, W[rows = out][cols = in] row-major (egg.c:42-50)
    long long w_off;       // byte offset in the model blob (and in the fragment copies)
    int rows, cols;
    long long a_off, b_off;   // offsets of the per-pair noise vectors (both orders), [pair][rows] / [pair][cols]
    long long pa_off, pb_off; // offsets of the update panels [rows][pairs_pad] / [cols][pairs_pad]
    int seed_off;          // 100*l + k, or 999 for the head (egg.c:242-290)
    int shift;
};

// rank-1 term, shift and clamp of one strip (egg.c:167-175); returns the 16 int8 results packed in slot order
__device__ __forceinline__ v4i gru_finish(const v16i &acc, int xb, const v4i &a4, int ns, int sigma, int shift) {
    v4i out;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            int noise = (xb * sx8(a4[q], e)) * ns;
            o[e] = clip127((acc[4 * q + e] + (noise >> sigma)) >> shift);
        }
        out[q] = pack4(o[0], o[1], o[2], o[3]);
    }
    return out;
}
__device__ __forceinline__ int cadd(int a, int b) { return clip127(a + b); }   // clipped_add, egg.c:62-67

// ---- the pipeline (egg_gru_pipe.hip)
// "Pipe order" of a row: within each 64 consecutive indices, index 32 v + 16 c + 4 g + e (v, c < 2; g, e < 4) lies at byte
// 16 g + 8 c + 4 v + e.  Dword d of a 64-group in pipe order is natural dword pipe_dword(d).
__host__ __device__ constexpr int pipe_dword(int d) { return 8 * (d & 1) + 4 * ((d >> 1) & 1) + (d >> 2); }
__host__ __device__ constexpr int pipe_pos(int n) { return (n & ~63) + 16 * ((n >> 2) & 3) + 8 * ((n >> 4) & 1) + 4 * ((n >> 5) & 1) + (n & 3); }

#define GRU_CHUNK 32               // tokens per chunk
#define GRU_PIPE_MEMBERS 512       // members evaluated at a time
#define GRU_MAX_LAYERS 8
struct PipeMat { uint32_t w_off; long long a_off, b_off; };
struct PipeParams {
    const int8_t *frag;            // fragment-major copies of the matrices at their offsets in the model blob
    const int8_t *rows;            // embedding [V][H] | biases [L][2][H] | gains [L][2][H] | output gains [H], each row in pipe order
    const int8_t *noise_slot;      // A vectors, slot order
    const int8_t *noise_pipe;      // A and B vectors, pipe order
    const uint8_t *data; long long data_len, start_idx;
    int8_t *states;                // [population][L][H], natural order
    int8_t *h;                     // [L][members][H], pipe order
    int8_t *act;                   // gru_pipe_act_bytes
    int32_t *loss;                 // [population]
    const int32_t *exp2;           // [256]
    int L, T, V, population, first, members, sigma;       // members first .. first + members - 1 of the population
    PipeMat m[6 * GRU_MAX_LAYERS + 1];
};
size_t gru_pipe_act_bytes(int members, int H, int L);
size_t gru_pipe_rows_bytes(int H, int L, int V);
hipError_t gru_pipe_prepare(int H);
// one step's forward of the members of `p` (in stream order: state in, ticks, state out)
hipError_t gru_pipe_forward(const PipeParams &p, int H, hipStream_t s);
// frag and rows from the model blob
hipError_t gru_pipe_refresh(const int8_t *model, int8_t *frag, int8_t *rows, const GruMat *d_mats, int n_mats, int H, int L, int V,
                            long long off_emb, long long off_gru_b, long long off_ln_w, long long off_ln_out, hipStream_t s);
