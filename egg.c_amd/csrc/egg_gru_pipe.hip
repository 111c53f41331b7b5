// egg_gru_pipe.hip -- forward_pass of full_trained_egg.c (egg.c:213-296) for a population, as a pipeline over layers and chunks
// of 32 tokens on gfx950.
//
// Of a layer's products only two are recurrent: W1 h and W3 (f h) of a token need the state that the token before left.
// The other 10.5 of 12.5 H^2 weights (W0 x, W2 x, the MLP) see a layer's input or output sequence and may take many tokens at
// once.  So a layer's chunk passes four stages, one per launch (a tick):
//   A  norm, W0 x and W2 x of 32 tokens of a member            matrix products with the tokens as columns
//   R  the recurrence over the chunk's tokens                  one workgroup per 8 members, W1 and W3 resident on its CU
//   E  norm, MLP expand                                        as A
//   D  MLP project, residual                                   as A
// and layer l's chunk c is at stage k in tick c + 4 l + k; a launch carries every stage of every layer (and the head, as layer
// L).  Before, a tick was one stage of single tokens: 2 T + 6 L + 1 launches of 9.6 us, each streaming the weights again.
// Here there are T / 32 + 4 L, and R's chain of T steps that never leaves a CU is what a sequence takes.
//
// R: a workgroup of eight waves keeps W1 and W3 (512 KB at hidden 512) in its CU: all of W1 and a part of W3 in registers, the
// larger part of W3 in LDS.  Wave w owns 64 rows of both; a token is two products of 4 strips of 16 rows by 8 members on
// v_mfma_i32_16x16x64_i8 with a barrier behind each.  The 16 columns hold the 8 members twice: lanes of the first copy finish
// strips 0 and 2, lanes of the second strips 1 and 3, so the elementwise arithmetic -- more than the products -- uses every
// lane.  What bounds a token (2.35 us at hidden 512) is one wave per SIMD issuing, one behind the other, the reads of operand and
// LDS fragments, 64 MFMAs and about 300 vector instructions; the order between them changed nothing.
// "Pipe order" (egg_gru.h) of a row is the order in which those lanes hold 64 rows' results, so what a wave stores is operand
// for the next product as it stands.
//
// A, E, D, head: a workgroup of eight waves takes 8 members; a wave has 32 tokens of one member as the columns of
// v_mfma_i32_32x32x32_i8 (one member: its noise vectors are wave-uniform), the weights go by in blocks of 64 output columns
// through four LDS buffers that all eight waves read.
//
// A tick at hidden 512, 4 layers, 128 members (272 workgroups): R 90 us (the weights 15, 32 tokens of 2.3), E 71, D 61, A 45, the head 22 behind an A.
// D was 106 and the tick's length: its input row came from memory once for every 64 output columns, and every stage's wait for a
// small load of a block took the copy that had just been requested along.
#include "egg_gru.h"

#pragma clang fp contract(off)

namespace {

constexpr int THREADS = 512, WAVES = 8, C = GRU_CHUNK;

// ---- buffers: units of members * 32 * H bytes.  What a stage writes is read in the next tick (G, M) or the next two
// (the residual streams X in front of a layer and X1 behind its recurrence), hence two and four copies by chunk number.
__host__ __device__ inline size_t unit(int members, int H) { return (size_t)members * C * H; }
__device__ __forceinline__ int8_t *buf_x(const PipeParams &p, int H, int l, int c) { return p.act + unit(p.members, H) * (4 * l + (c & 3)); }
__device__ __forceinline__ int8_t *buf_x1(const PipeParams &p, int H, int l, int c) { return p.act + unit(p.members, H) * (4 * (p.L + 1) + 4 * l + (c & 3)); }
__device__ __forceinline__ int8_t *buf_g(const PipeParams &p, int H, int l, int which, int c) {
    return p.act + unit(p.members, H) * (4 * (p.L + 1) + 4 * p.L + 4 * l + 2 * which + (c & 1));
}
__device__ __forceinline__ int8_t *buf_m(const PipeParams &p, int H, int l, int c) { return p.act + unit(p.members, H) * (4 * (p.L + 1) + 8 * p.L + 8 * l + 4 * (c & 1)); }

__device__ __forceinline__ int *buf_xb(const PipeParams &p, int H, int l, int c) {      // [member][token] of a layer's E, for its D
    return reinterpret_cast<int *>(p.act + unit(p.members, H) * (20 * p.L + 4)) + (size_t)(2 * l + (c & 1)) * p.members * C;
}

__device__ __forceinline__ const int8_t *row_bias(const PipeParams &p, int H, int l, int which) { return p.rows + (size_t)(p.V + 2 * l + which) * H; }
__device__ __forceinline__ const int8_t *row_gain(const PipeParams &p, int H, int l, int which) { return p.rows + (size_t)(p.V + 2 * p.L + 2 * l + which) * H; }
__device__ __forceinline__ const int8_t *row_gain_out(const PipeParams &p, int H) { return p.rows + (size_t)(p.V + 4 * p.L) * H; }

// ---------------------------------------------------------------- stage R
template <int H>
struct Rec {
    static constexpr int KS = H / 64;              // k-steps of 64, and waves with rows
    // fragments (strip s, k-step ks) of W3 that do not fit the registers beside W1: the k-steps from 4 on, and two more
    static constexpr bool in_lds(int s, int ks) { return KS == 8 && (ks >= 4 || (ks == 3 && s < 2)); }
    static constexpr int lds_slot(int s, int ks) { return ks >= 4 ? 4 * (ks - 4) + s : 16 + s; }
    static constexpr int LDS_W = KS == 8 ? WAVES * 18 * 1024 : 0, OPERAND = KS * 512;
    static constexpr int LDS = LDS_W + 2 * OPERAND + 2 * 256;
};
// Fragments of W1 / W3: [strip of 16 rows][k-step][lane (row, k quarter)][16 bytes], 1 KB per (strip, k-step)
__device__ __forceinline__ v4i rec_frag(const int8_t *f, uint32_t strip, int ks, int KS, int lane) {
    return *reinterpret_cast<const v4i *>(f + (strip * (uint32_t)KS + ks) * 1024u + lane * 16u);
}
template <int N>
__device__ __forceinline__ int swap_row8(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x120 | N, 0xf, 0xf, false); }
// over the lanes that hold pieces of one member's row (same lane number mod 8)
__device__ __forceinline__ int member_sum(int v) {
    v += swap_row8<8>(v);
    const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    return sum_halves((int)(r[0] + r[1]));
}
__device__ __forceinline__ int2 ld8(const int8_t *p) { return *reinterpret_cast<const int2 *>(p); }

template <int H>
__device__ __forceinline__ void stage_rec(const PipeParams &p, int l, int tile, int chunk, int8_t *lds) {
    typedef Rec<H> R;
    constexpr int KS = R::KS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m = lane & 7, g = lane >> 4, local = tile * 8 + m;
    const bool second = lane & 8;                  // this lane finishes strips 1 and 3
    const int tokens = min(C, p.T - chunk * C);
    int8_t *const w3l = lds + wave * 18 * 1024 + lane * 16, *const op_h = lds + R::LDS_W, *const op_g = op_h + R::OPERAND;
    int *const xb_h = reinterpret_cast<int *>(op_g + R::OPERAND), *const xb_g = xb_h + 64;      // [member][wave]
    if (wave >= KS) {                              // hidden below 512: the waves without rows only keep the barriers
        for (int t = 0; t < 2 * tokens + 1; t++) __syncthreads();
        return;
    }
    const PipeMat m1 = p.m[6 * l + 1], m3 = p.m[6 * l + 3];
    v4i w1[4][KS], w3[4][KS];
    // (straight to LDS what stays there: through registers the loads behind it waited for those stores.  Inline assembly for the reason given at
    // dma_unit, egg_device.h; waited for in front of the token loop)
    const uint32_t w3_lds = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(size_t)(const __attribute__((address_space(3))) int8_t *)lds) + wave * 18 * 1024;
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            if (R::in_lds(s, ks))
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                             : : "s"(w3_lds + R::lds_slot(s, ks) * 1024), "v"((uint32_t)lane * 16), "s"(p.frag + m3.w_off + ((4 * wave + s) * (uint32_t)KS + ks) * 1024u) : "memory", "m0");
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            w1[s][ks] = rec_frag(p.frag + m1.w_off, 4 * wave + s, ks, KS, lane);
            if (!R::in_lds(s, ks)) w3[s][ks] = rec_frag(p.frag + m3.w_off, 4 * wave + s, ks, KS, lane);
        }
    const uint32_t at = 64 * wave + 16 * g + (second ? 8 : 0);          // this lane's 8 bytes of a row: strips 0 and 2, or 1 and 3
    const long long pair = (p.first + local) >> 1;
    const int ns = (local & 1) ? -1 : 1;
    const int2 a1 = ld8(p.noise_pipe + m1.a_off + pair * H + at), b1 = ld8(p.noise_pipe + m1.b_off + pair * H + at),
               a3 = ld8(p.noise_pipe + m3.a_off + pair * H + at), b3 = ld8(p.noise_pipe + m3.b_off + pair * H + at),
               bf = ld8(row_bias(p, H, l, 0) + at), bh = ld8(row_bias(p, H, l, 1) + at);
    int8_t *const hs = p.h + ((size_t)l * p.members + local) * H + at;
    // uniform bases, one offset
    const int8_t *const g0p = buf_g(p, H, l, 0, chunk), *const g2p = buf_g(p, H, l, 1, chunk), *const xp = buf_x(p, H, l, chunk);
    int8_t *const op = buf_x1(p, H, l, chunk);
    uint32_t off = (uint32_t)local * C * H + at;
    const uint32_t put = ((wave * 4 + g) * 8 + m) * 16 + (second ? 8 : 0);
    uint32_t get = g * 128 + m * 16;
    int2 h = ld8(hs);
    auto publish = [&](int2 v, int8_t *operand, int2 b, int *xb) {
        *reinterpret_cast<int2 *>(operand + put) = v;
        const int part = member_sum(dot4(v.x, b.x, dot4(v.y, b.y, 0)));
        if (lane < 8) xb[m * 8 + wave] = part;
    };
    auto total = [&](const int *xb) {
        int s = 0;
#pragma unroll
        for (int w = 0; w < KS; w++) s += xb[m * 8 + w];
        return s * ns;
    };
    auto value = [&](int acc, int xb, int a) { return clip127((acc + (mul24(xb, a) >> p.sigma)) >> 8); };     // egg.c:167-175, shift 8
    publish(h, op_h, b1, xb_h);
    __syncthreads();
    // Two passes of two strips that each read the operand again: with the four accumulators of one pass, or the operand kept,
    // fragments go to scratch (2.8 us a token at hidden 512; 2.35 as it is, of which the matrix unit has 0.9).
    auto product = [&](const v4i (&w)[4][KS], bool third, const int8_t *operand, auto one) {
        v4i mine = {0, 0, 0, 0};
#pragma unroll
        for (int v = 0; v < 2; v++) {
            v4i c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const v4i b = *reinterpret_cast<const v4i *>(operand + ks * 512 + get);
                const v4i f0 = third && R::in_lds(2 * v, ks) ? *reinterpret_cast<const v4i *>(w3l + R::lds_slot(2 * v, ks) * 1024) : w[2 * v][ks],
                          f1 = third && R::in_lds(2 * v + 1, ks) ? *reinterpret_cast<const v4i *>(w3l + R::lds_slot(2 * v + 1, ks) * 1024) : w[2 * v + 1][ks];
                c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(f0, b, c0, 0, 0, 0);
                c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(f1, b, c1, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (v == 1) one(0, e, mine[e]);
                mine[e] = second ? c1[e] : c0[e];
            }
            asm volatile("" : "+v"(get));          // the operand is read again for the other two strips, not kept
        }
#pragma unroll
        for (int e = 0; e < 4; e++) one(1, e, mine[e]);
    };
    int2 g0 = ld8(g0p + off);
    __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0) here, so that no wait inside the loop has to allow for it
    for (int t = 0; t < tokens; t++, off += H) {
        int2 ft, xo;
        {   // W1 h, ft = cadd(cadd(W0 x, W1 h), b_f), gated = ((ft + 127) h) >> 8 (egg.c:246-258)
            const int xb1 = total(xb_h);
            int f[4], gt[4];
            int2 gated;
            product(w1, false, op_h, [&](int v, int e, int a) {
                const int r = value(a, xb1, sx8(v ? a1.y : a1.x, e));
                f[e] = cadd(cadd(sx8(v ? g0.y : g0.x, e), r), sx8(v ? bf.y : bf.x, e));
                gt[e] = mul24(f[e] + 127, sx8(v ? h.y : h.x, e)) >> 8;
                if (e == 3) { (v ? ft.y : ft.x) = pack4(f[0], f[1], f[2], f[3]); (v ? gated.y : gated.x) = pack4(gt[0], gt[1], gt[2], gt[3]); }
            });
            publish(gated, op_g, b3, xb_g);
        }
        __syncthreads();
        {   // W3 gated, ht = cadd(cadd(W2 x, W3 gated), b_h), h += ((ft + 127) (ht - h)) >> 8, x = cadd(h, x) (egg.c:260-271)
            // the next token's loads go in front of this token's store: a wait for a load waits for the stores before it
            const int2 g2 = ld8(g2p + off), x = ld8(xp + off);
            g0 = ld8(g0p + off + (t + 1 < tokens ? H : 0));
            const int xb3 = total(xb_g);
            int hv[4], xv[4];
            product(w3, true, op_g, [&](int v, int e, int a) {
                const int r = value(a, xb3, sx8(v ? a3.y : a3.x, e));
                const int ht = cadd(cadd(sx8(v ? g2.y : g2.x, e), r), sx8(v ? bh.y : bh.x, e)), h0 = sx8(v ? h.y : h.x, e);
                hv[e] = cadd(h0, mul24(sx8(v ? ft.y : ft.x, e) + 127, ht - h0) >> 8);
                xv[e] = cadd(hv[e], sx8(v ? x.y : x.x, e));
                if (e == 3) { (v ? h.y : h.x) = pack4(hv[0], hv[1], hv[2], hv[3]); (v ? xo.y : xo.x) = pack4(xv[0], xv[1], xv[2], xv[3]); }
            });
            publish(h, op_h, b1, xb_h);
        }
        *reinterpret_cast<int2 *>(op + off) = xo;
        __syncthreads();
    }
    *reinterpret_cast<int2 *>(hs) = h;
}

// ---------------------------------------------------------------- stages A, E, D and the head
// Weights of these products: [64 output columns][k-step of 32][half][64 columns][16 bytes], k in pipe order.  A block is 64
// columns by H inputs, contiguous; the workgroup copies it straight to LDS.
template <int H>
__device__ __forceinline__ void fetch_block(int8_t *dst, const int8_t *src) {
    constexpr int PER = H >= 128 ? H / 128 : 1;    // KB per wave
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (H < 128 && wave >= 4) return;
    const uint32_t m0v = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(size_t)(const __attribute__((address_space(3))) int8_t *)dst) + wave * PER * 1024;
    const uint64_t b = (uint64_t)(src + wave * PER * 1024);
    const uint32_t blo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b), bhi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    const uint64_t sb = ((uint64_t)bhi << 32) | blo;
    const uint32_t v = (threadIdx.x & 63) * 16;
    // inline assembly for the reason given at dma_unit (egg_device.h); waited for in next_block
    if (PER == 1) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(m0v), "v"(v), "s"(sb) : "memory", "m0");
    else if (PER == 2) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024"
                                    : : "s"(m0v), "v"(v), "s"(sb) : "memory", "m0");
    else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\tglobal_load_lds_dwordx4 %1, %2 offset:1024\n\t"
                      "global_load_lds_dwordx4 %1, %2 offset:2048\n\tglobal_load_lds_dwordx4 %1, %2 offset:3072" : : "s"(m0v), "v"(v), "s"(sb) : "memory", "m0");
}
// The blocks of one or two matrices in turn, through a ring of four buffers: a block is requested three blocks ahead of its use.  A wave
// waits for its own part of the oldest by counting the younger copies, so a request follows every take (past the end the last
// block again, which no one reads), and other loads and stores in flight make the wait longer, never shorter.  The caller puts a
// block's small loads in front of `request`: loads return in order, and the compiler, which does not see the copies, waits for
// everything behind the last load that it knows of.
template <int H>
struct Blocks {
    static constexpr int BUFS = 4, SIZE = 64 * H, PER = H >= 128 ? H / 128 : 1;
    int8_t *base;
    const int8_t *a, *b; int na, n, next, used;    // blocks 0 .. na - 1 at a, na .. n - 1 at b
    __device__ __forceinline__ void begin(int8_t *lds, const int8_t *first, int n_first, const int8_t *second, int n_second) {
        base = lds; a = first; b = second; na = n_first; n = n_first + n_second; next = used = 0;
    }
    __device__ __forceinline__ void request(int i) {        // i: the block's place in its matrix
        fetch_block<H>(base + (next & (BUFS - 1)) * SIZE, i < na ? a + (size_t)i * SIZE : b + (size_t)(i - na) * SIZE);
        next++;
    }
    __device__ __forceinline__ void request() { request(min(next, n - 1)); }
    __device__ __forceinline__ const int8_t *take() {
        static_assert((BUFS - 2) * PER < 16, "the wait's low field");
        __builtin_amdgcn_s_waitcnt(0x0F70 | ((BUFS - 2) * PER));
        __syncthreads();
        return base + (used++ & (BUFS - 1)) * SIZE;
    }
    // the copies that no one reads: a workgroup's LDS must not be written behind its end
    __device__ __forceinline__ void drain() { __builtin_amdgcn_s_waitcnt(0x0F70); }
};
template <int NK>
__device__ __forceinline__ void multiply(v16i (&acc)[2], const v4i (&x)[NK], const int8_t *block, int lane) {
#pragma unroll
    for (int ks = 0; ks < NK; ks++) {
        const int8_t *f = block + ((2 * ks + (lane >> 5)) * 64 + (lane & 31)) * 16;
        const v4i f0 = *reinterpret_cast<const v4i *>(f), f1 = *reinterpret_cast<const v4i *>(f + 512);
        acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f0, x[ks], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f1, x[ks], acc[1], 0, 0, 0);
    }
}
// the same, and each k-step's operand gives way to the one at `ops` (load_ops) when it has been multiplied
template <int NK>
__device__ __forceinline__ void multiply_reload(v16i (&acc)[2], v4i (&x)[NK], const int8_t *block, const int8_t *ops, int lane) {
#pragma unroll
    for (int ks = 0; ks < NK; ks++) {
        const int8_t *f = block + ((2 * ks + (lane >> 5)) * 64 + (lane & 31)) * 16;
        const v4i f0 = *reinterpret_cast<const v4i *>(f), f1 = *reinterpret_cast<const v4i *>(f + 512);
        acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f0, x[ks], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f1, x[ks], acc[1], 0, 0, 0);
        x[ks] = *reinterpret_cast<const v4i *>(ops + 1024 * ks + (uint32_t)lane * 16);
    }
}
template <int NK>
__device__ __forceinline__ void load_row(v4i (&x)[NK], const int8_t *row, int g) {
#pragma unroll
    for (int ks = 0; ks < NK; ks++) x[ks] = *reinterpret_cast<const v4i *>(row + 32 * ks + 16 * g);
}
// the same from the MLP's intermediate, which is kept in the order of these loads: [member][k-step][half][token][16 bytes]
template <int NK>
__device__ __forceinline__ void load_ops(v4i (&x)[NK], const int8_t *ops, uint32_t lane16) {      // ops: uniform
#pragma unroll
    for (int ks = 0; ks < NK; ks++) x[ks] = *reinterpret_cast<const v4i *>(ops + 1024 * ks + lane16);
}
template <int NK>
__device__ __forceinline__ int noise_dot(const v4i (&x)[NK], const int8_t *b, int g) {
    int s = 0;
#pragma unroll
    for (int ks = 0; ks < NK; ks++) {
        const v4i n = *reinterpret_cast<const v4i *>(b + 32 * ks + 16 * g);
#pragma unroll
        for (int q = 0; q < 4; q++) s = dot4(x[ks][q], n[q], s);
    }
    return s;
}
// egg_ln (egg.c:180-210) of the lane's token
template <int NK>
__device__ __forceinline__ void norm(v4i (&x)[NK], const int8_t *gains, int g) {
    int sum = sum_halves(sumabs_groups<NK>(x));
    if (sum == 0) sum = 1;
    int mean = sum / (32 * NK);
    if (mean == 0) mean = 1;
    const float rcp = 1.0f / (float)mean;
#pragma unroll
    for (int ks = 0; ks < NK; ks++) {
        const v4i w = *reinterpret_cast<const v4i *>(gains + 32 * ks + 16 * g);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            int o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = clip127(div_trunc(sx8(x[ks][q], e) * sx8(w[q], e), rcp));
            x[ks][q] = pack4(o[0], o[1], o[2], o[3]);
        }
    }
}
// the accumulators of a block start from the rank-1 term, (x.B A ns) >> sigma (egg.c:167-175); xbn: x.B times the member's sign
__device__ __forceinline__ void begin_block(v16i (&acc)[2], int xbn, const v4i &a0, const v4i &a1, int sigma) {
#pragma unroll
    for (int r = 0; r < 16; r++) { acc[0][r] = mul24(xbn, sx8(a0[r >> 2], r & 3)) >> sigma; acc[1][r] = mul24(xbn, sx8(a1[r >> 2], r & 3)) >> sigma; }
}
__device__ __forceinline__ v4i clamped(const v16i &acc, int shift) {
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; q++)
        o[q] = pack4(clip127(acc[4 * q] >> shift), clip127(acc[4 * q + 1] >> shift), clip127(acc[4 * q + 2] >> shift), clip127(acc[4 * q + 3] >> shift));
    return o;
}
// a block's 64 results of the lane's token, its half: the 16-byte pieces g and g + 2 of the row's 64-group in pipe order
struct Pieces { v4i lo, hi; };
__device__ __forceinline__ Pieces finish_block(const v16i (&acc)[2], int shift) {
    const v4i r0 = clamped(acc[0], shift), r1 = clamped(acc[1], shift);
    Pieces o;
    o.lo = v4i{r0[0], r1[0], r0[2], r1[2]};
    o.hi = v4i{r0[1], r1[1], r0[3], r1[3]};
    return o;
}
__device__ __forceinline__ void store_pieces(int8_t *group, const Pieces &o, int g) {
    *reinterpret_cast<v4i *>(group + 16 * g) = o.lo;
    *reinterpret_cast<v4i *>(group + 32 + 16 * g) = o.hi;
}
__device__ __forceinline__ v4i cadd16(v4i a, v4i b) {
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = cadd(sx8(a[q], e), sx8(b[q], e));
        o[q] = pack4(v[0], v[1], v[2], v[3]);
    }
    return o;
}
__device__ __forceinline__ long long stream_pos(const PipeParams &p, int member) {
    const long long stride = p.data_len / (p.population / 2);                    // egg.c:553-554
    return (p.start_idx + (long long)(member >> 1) * stride) % (p.data_len - p.T);
}
__device__ __forceinline__ v4i ld16(const int8_t *p) { return *reinterpret_cast<const v4i *>(p); }

struct Tile { int local, member, ns, g, lane, token; long long pair; };
__device__ __forceinline__ Tile tile_of(const PipeParams &p, int unit8, int chunk) {
    Tile t;
    t.lane = threadIdx.x & 63; t.g = t.lane >> 5;
    t.local = unit8 * 8 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    t.member = p.first + t.local; t.ns = (t.member & 1) ? -1 : 1; t.pair = t.member >> 1;
    t.token = min(chunk * C + (t.lane & 31), p.T - 1);          // tokens past the end repeat the last one; nothing reads their results
    return t;
}

template <int H>
__device__ __forceinline__ void stage_a(const PipeParams &p, int l, int unit8, int chunk, int8_t *lds) {
    constexpr int NK = H / 32, NB = H / 64;
    const Tile t = tile_of(p, unit8, chunk);
    const PipeMat m0 = p.m[6 * l], m2 = p.m[6 * l + 2];
    Blocks<H> blocks;
    blocks.begin(lds, p.frag + m0.w_off, NB, p.frag + m2.w_off, NB);
    const size_t row = ((size_t)t.local * C + (t.lane & 31)) * H;
    v4i x[NK];
    if (l == 0) {                                  // egg.c:238
        const int tok = p.data[stream_pos(p, t.member) + t.token];
        load_row<NK>(x, p.rows + (size_t)tok * H, t.g);
#pragma unroll
        for (int ks = 0; ks < NK; ks++) *reinterpret_cast<v4i *>(buf_x(p, H, 0, chunk) + row + 32 * ks + 16 * t.g) = x[ks];
    } else
        load_row<NK>(x, buf_x(p, H, l, chunk) + row, t.g);
    norm<NK>(x, row_gain(p, H, l, 0), t.g);
    const int xb0 = t.ns * sum_halves(noise_dot<NK>(x, p.noise_pipe + m0.b_off + t.pair * H, t.g)),
              xb2 = t.ns * sum_halves(noise_dot<NK>(x, p.noise_pipe + m2.b_off + t.pair * H, t.g));
    auto noise_of = [&](int b) { return p.noise_slot + (b >= NB ? m2.a_off : m0.a_off) + t.pair * H + 64 * (b >= NB ? b - NB : b) + 16 * t.g; };
    v4i a0 = ld16(noise_of(0)), a1 = ld16(noise_of(0) + 32);
    for (int i = 0; i < 3; i++) blocks.request();
    for (int b = 0; b < 2 * NB; b++) {
        const int which = b >= NB, nb = which ? b - NB : b;
        const int8_t *w = blocks.take();
        v16i acc[2];
        begin_block(acc, which ? xb2 : xb0, a0, a1, p.sigma);
        const int8_t *a = noise_of(min(b + 1, 2 * NB - 1));
        a0 = ld16(a); a1 = ld16(a + 32);
        blocks.request();
        multiply<NK>(acc, x, w, t.lane);
        store_pieces(buf_g(p, H, l, which, chunk) + row + 64 * nb, finish_block(acc, 8), t.g);
    }
    blocks.drain();
}
template <int H>
__device__ __forceinline__ void stage_e(const PipeParams &p, int l, int unit8, int chunk, int8_t *lds) {
    constexpr int NK = H / 32, NB = 4 * H / 64;
    const Tile t = tile_of(p, unit8, chunk);
    const PipeMat m = p.m[6 * l + 4];
    Blocks<H> blocks;
    blocks.begin(lds, p.frag + m.w_off, NB, nullptr, 0);
    const size_t row = (size_t)t.local * C + (t.lane & 31);
    v4i x[NK];
    load_row<NK>(x, buf_x1(p, H, l, chunk) + row * H, t.g);
    norm<NK>(x, row_gain(p, H, l, 1), t.g);
    const int xb = t.ns * sum_halves(noise_dot<NK>(x, p.noise_pipe + m.b_off + t.pair * H, t.g));
    const int8_t *a = p.noise_slot + m.a_off + t.pair * 4 * H + 16 * t.g, *bd = p.noise_pipe + p.m[6 * l + 5].b_off + t.pair * 4 * H + 16 * t.g;
    int8_t *out = buf_m(p, H, l, chunk) + (size_t)t.local * C * 4 * H + t.lane * 16;
    int xbd = 0;                                   // the projection's x . B, of the results as they leave
    v4i a0 = ld16(a), a1 = ld16(a + 32), nn0 = ld16(bd), nn1 = ld16(bd + 32);
    for (int i = 0; i < 3; i++) blocks.request();
    for (int b = 0; b < NB; b++) {
        const int8_t *w = blocks.take();
        v16i acc[2];
        begin_block(acc, xb, a0, a1, p.sigma);
        const v4i n0 = nn0, n1 = nn1;
        const int ahead = 64 * min(b + 1, NB - 1);
        a0 = ld16(a + ahead); a1 = ld16(a + ahead + 32); nn0 = ld16(bd + ahead); nn1 = ld16(bd + ahead + 32);
        blocks.request();
        multiply<NK>(acc, x, w, t.lane);
        const Pieces o = finish_block(acc, 8);
#pragma unroll
        for (int q = 0; q < 4; q++) xbd = dot4(o.lo[q], n0[q], dot4(o.hi[q], n1[q], xbd));
        *reinterpret_cast<v4i *>(out + 2048 * b) = o.lo;
        *reinterpret_cast<v4i *>(out + 2048 * b + 1024) = o.hi;
    }
    xbd = t.ns * sum_halves(xbd);
    if (t.g == 0) buf_xb(p, H, l, chunk)[row] = xbd;
    blocks.drain();
}
template <int H>
__device__ __forceinline__ void stage_d(const PipeParams &p, int l, int unit8, int chunk, int8_t *lds) {
    constexpr int NK = H / 32, NB = H / 64;
    const Tile t = tile_of(p, unit8, chunk);
    const PipeMat m = p.m[6 * l + 5];
    Blocks<H> blocks;
    blocks.begin(lds, p.frag + m.w_off, 4 * NB, nullptr, 0);
    const size_t row = (size_t)t.local * C + (t.lane & 31);
    const uint32_t lane16 = t.lane * 16;
    const int8_t *in = buf_m(p, H, l, chunk) + (size_t)t.local * C * 4 * H, *res = buf_x1(p, H, l, chunk) + row * H + 16 * t.g,
                 *a = p.noise_slot + m.a_off + t.pair * H + 16 * t.g;
    int8_t *out = buf_x(p, H, l + 1, chunk) + row * H;
    const int xb = buf_xb(p, H, l, chunk)[row];
    // NBP blocks of 64 columns at a time, for which the input row goes by in quarters (with one block at a time it came from memory eight
    // times, four times the weights' bytes); the next quarter replaces this one as the last block's products leave it.
    constexpr int NBP = NB < 4 ? NB : 4;
    auto place = [&](int n) { n = min(n, 4 * NB - 1); const int part = n / (4 * NBP), kc = n / NBP % 4, j = n % NBP; return (part * NBP + j) * 4 + kc; };
    v4i x[NK];
    load_ops<NK>(x, in, lane16);
    for (int i = 0; i < 3; i++) blocks.request(place(i));
#pragma unroll 1
    for (int part = 0; part < NB / NBP; part++) {
        v16i acc[NBP][2];
#pragma unroll
        for (int j = 0; j < NBP; j++) begin_block(acc[j], xb, ld16(a + 64 * (part * NBP + j)), ld16(a + 64 * (part * NBP + j) + 32), p.sigma);
#pragma unroll 1
        for (int kc = 0; kc < 4; kc++)
#pragma unroll
            for (int j = 0; j < NBP; j++) {
                const int8_t *w = blocks.take();
                blocks.request(place(blocks.next));
                if (j + 1 < NBP) multiply<NK>(acc[j], x, w, t.lane);
                else multiply_reload<NK>(acc[j], x, w, in + ((kc + 1) & 3) * NK * 1024, t.lane);
            }
#pragma unroll
        for (int j = 0; j < NBP; j++) {
            const int at = 64 * (part * NBP + j);
            Pieces o = finish_block(acc[j], 9);
            o.lo = cadd16(o.lo, ld16(res + at));
            o.hi = cadd16(o.hi, ld16(res + at + 32));
            store_pieces(out + at, o, t.g);
        }
    }
    blocks.drain();
}
// output norm, logits (egg.c:288-294), loss (egg.c:321-330)
template <int H>
__device__ __forceinline__ void stage_head(const PipeParams &p, int unit8, int chunk, int8_t *lds) {
    constexpr int NK = H / 32;
    const Tile t = tile_of(p, unit8, chunk);
    const PipeMat m = p.m[6 * p.L];
    Blocks<H> blocks;
    blocks.begin(lds, p.frag + m.w_off, p.V / 64, nullptr, 0);
    int *exp2 = reinterpret_cast<int *>(lds + Blocks<H>::BUFS * 64 * H);
    if (threadIdx.x < 256) exp2[threadIdx.x] = p.exp2[threadIdx.x];            // the first take() synchronises
    v4i x[NK];
    load_row<NK>(x, buf_x(p, H, p.L, chunk) + ((size_t)t.local * C + (t.lane & 31)) * H, t.g);
    norm<NK>(x, row_gain_out(p, H), t.g);
    const int xb = t.ns * sum_halves(noise_dot<NK>(x, p.noise_pipe + m.b_off + t.pair * H, t.g));
    const int8_t *a = p.noise_slot + m.a_off + t.pair * p.V + 16 * t.g;
    const int target = p.data[stream_pos(p, t.member) + t.token + 1];
    int sum_exp = 0, tl = 0;
    v4i a0 = ld16(a), a1 = ld16(a + 32);
    for (int i = 0; i < 3; i++) blocks.request();
    for (int b = 0; b < p.V / 64; b++) {
        const int8_t *w = blocks.take();
        v16i acc[2];
        begin_block(acc, xb, a0, a1, p.sigma);
        const int ahead = 64 * min(b + 1, p.V / 64 - 1);
        a0 = ld16(a + ahead); a1 = ld16(a + ahead + 32);
        blocks.request();
        multiply<NK>(acc, x, w, t.lane);
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const v4i r = clamped(acc[half], 8);
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int v = sx8(r[q], e);
                    sum_exp += exp2[v + 128];
                    if (64 * b + 32 * half + 8 * q + 4 * t.g + e == target) tl = v;
                }
        }
    }
    blocks.drain();
    sum_exp = sum_halves(sum_exp); tl = sum_halves(tl);
    int lg2 = 0;                                   // log2_fixed (egg.c:309-319)
    if (sum_exp > 0) {
        const int k = 31 - __clz(sum_exp);
        const int frac = (k >= 4) ? ((sum_exp - (1 << k)) >> (k - 4)) : ((sum_exp - (1 << k)) << (4 - k));
        lg2 = (k << 4) + frac - 64;
    }
    int loss = t.lane < 32 && chunk * C + t.lane < p.T ? lg2 - (tl + 128) : 0;
    for (int o = 16; o > 0; o >>= 1) loss += __shfl_xor(loss, o, 64);
    if (t.lane == 0) atomicAdd(p.loss + t.member, loss);
}

// one tick: the longest units first
template <int H>
__global__ void __launch_bounds__(THREADS, 2) k_gru_tick(PipeParams p, int tick, int chunks) {
    extern __shared__ __align__(16) int8_t lds[];
    // Workgroups go to the eight XCDs in turn; those of one XCD take consecutive units of a role, so that the tiles of a layer meet in one
    // or two L2s and its weights (3 MB at hidden 512) stay there.
    const int n = p.members / 8, units = p.L * n, role = (int)blockIdx.x / units, at = (int)blockIdx.x % units;
    const int i = units & 7 ? at : (at & 7) * (units >> 3) + (at >> 3), l = i / n, u = i % n;
    auto chunk_at = [&](int layer, int stage) { const int c = tick - 4 * layer - stage; return c >= 0 && c < chunks ? c : -1; };
    int c;
    if (role == 0) { if ((c = chunk_at(l, 1)) >= 0) stage_rec<H>(p, l, u, c, lds); }
    else if (role == 1) { if ((c = chunk_at(l, 2)) >= 0) stage_e<H>(p, l, u, c, lds); }
    else if (role == 2) { if ((c = chunk_at(l, 3)) >= 0) stage_d<H>(p, l, u, c, lds); }
    else if (role == 3) { if ((c = chunk_at(l, 0)) >= 0) stage_a<H>(p, l, u, c, lds); }
    else if ((c = chunk_at(p.L, 0)) >= 0) stage_head<H>(p, at, c, lds);
}

// the state between its natural order, [member][L][H], and the pipe order of the ticks, [L][member][H]; zero losses
__global__ void k_gru_state(PipeParams p, int H, int out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, groups = H / 64, d = i & 15, grp = (i >> 4) % groups, r = (i >> 4) / groups;
    if (!out && i < p.members) p.loss[p.first + i] = 0;
    if (r >= p.L * p.members) return;
    const int l = r / p.members, m = r % p.members;
    int *nat = reinterpret_cast<int *>(p.states + ((size_t)(p.first + m) * p.L + l) * H + 64 * grp) + pipe_dword(d);
    int *pipe = reinterpret_cast<int *>(p.h + ((size_t)l * p.members + m) * H + 64 * grp) + d;
    if (out) *nat = *pipe; else *pipe = *nat;
}

// fragment copies: of the recurrent matrices (role 1 or 3 of a layer) by strips of 16 rows and k-steps of 64, of the others by
// blocks of 64 rows and k-steps of 32; in both the k index runs in pipe order
__global__ void k_gru_frag(const int8_t *model, int8_t *frag, const GruMat *mats, int n_mats, int L) {
    const GruMat m = mats[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;         // a 16-byte piece of a row: pipe-order bytes 16 pc .. of row n
    const int pieces = m.cols / 16;
    if (i >= m.rows * pieces) return;
    const bool rec = (int)blockIdx.y < 6 * L && ((blockIdx.y % 6) == 1 || (blockIdx.y % 6) == 3);
    int n, pc;
    if (rec) { n = ((i >> 6) / (m.cols / 64)) * 16 + (i & 15); pc = ((i >> 6) % (m.cols / 64)) * 4 + ((i >> 4) & 3); }
    else { n = (i >> 6) / pieces * 64 + (i & 63); pc = (i >> 6) % pieces; }
    const int *src = reinterpret_cast<const int *>(model + m.w_off + (size_t)n * m.cols + 64 * (pc >> 2));
    v4i v;
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = src[pipe_dword(4 * (pc & 3) + q)];
    reinterpret_cast<v4i *>(frag + m.w_off)[i] = v;
}
__global__ void k_gru_rows(const int8_t *model, int8_t *rows, int H, int L, int V, long long off_emb, long long off_gru_b, long long off_ln_w, long long off_ln_out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, per = H / 4, r = i / per, d = i % per;
    if (r >= V + 4 * L + 1) return;
    const long long src = r < V ? off_emb + (long long)r * H : r < V + 2 * L ? off_gru_b + (long long)(r - V) * H
                        : r < V + 4 * L ? off_ln_w + (long long)(r - V - 2 * L) * H : off_ln_out;
    reinterpret_cast<int *>(rows + (size_t)r * H)[d] = reinterpret_cast<const int *>(model + src)[(d & ~15) + pipe_dword(d & 15)];
}

template <int H>
constexpr int tick_lds() { return Rec<H>::LDS > Blocks<H>::BUFS * 64 * H + 1024 ? Rec<H>::LDS : Blocks<H>::BUFS * 64 * H + 1024; }
template <int H>
hipError_t forward(const PipeParams &p, hipStream_t s) {
    const int chunks = (p.T + C - 1) / C, n = p.members / 8, items = std::max(p.members, p.L * p.members * (H / 4));
    hipLaunchKernelGGL(k_gru_state, dim3((items + 255) / 256), dim3(256), 0, s, p, H, 0);
    // the last chunk is at the head in tick chunks - 1 + 4 L
    for (int tick = 0; tick < chunks + 4 * p.L; tick++)
        hipLaunchKernelGGL(k_gru_tick<H>, dim3((4 * p.L + 1) * n), dim3(THREADS), tick_lds<H>(), s, p, tick, chunks);
    hipLaunchKernelGGL(k_gru_state, dim3((items + 255) / 256), dim3(256), 0, s, p, H, 1);
    return hipGetLastError();
}

}  // namespace

size_t gru_pipe_act_bytes(int members, int H, int L) { return unit(members, H) * (20 * L + 4) + (size_t)2 * L * members * C * sizeof(int); }
size_t gru_pipe_rows_bytes(int H, int L, int V) { return (size_t)(V + 4 * L + 1) * H; }
hipError_t gru_pipe_prepare(int H) {
#define EGG_PREP(HH) hipFuncSetAttribute(reinterpret_cast<const void *>(&k_gru_tick<HH>), hipFuncAttributeMaxDynamicSharedMemorySize, tick_lds<HH>())
    switch (H) { case 64: return EGG_PREP(64); case 128: return EGG_PREP(128); case 256: return EGG_PREP(256); case 512: return EGG_PREP(512); }
#undef EGG_PREP
    return hipErrorInvalidValue;
}
hipError_t gru_pipe_forward(const PipeParams &p, int H, hipStream_t s) {
    if (p.members < 8 || p.members % 8 || p.L < 1 || p.L > GRU_MAX_LAYERS || p.T < 1 || p.V != 256 || p.data_len <= p.T + 1) return hipErrorInvalidValue;
    switch (H) { case 64: return forward<64>(p, s); case 128: return forward<128>(p, s); case 256: return forward<256>(p, s); case 512: return forward<512>(p, s); }
    return hipErrorInvalidValue;
}
hipError_t gru_pipe_refresh(const int8_t *model, int8_t *frag, int8_t *rows, const GruMat *d_mats, int n_mats, int H, int L, int V,
                            long long off_emb, long long off_gru_b, long long off_ln_w, long long off_ln_out, hipStream_t s) {
    const int most = std::max(4 * H * H, V * H) / 16;
    hipLaunchKernelGGL(k_gru_frag, dim3((most + 255) / 256, n_mats), dim3(256), 0, s, model, frag, d_mats, n_mats, L);
    hipLaunchKernelGGL(k_gru_rows, dim3(((V + 4 * L + 1) * (H / 4) + 255) / 256), dim3(256), 0, s, model, rows, H, L, V, off_emb, off_gru_b, off_ln_w, off_ln_out);
    return hipGetLastError();
}
