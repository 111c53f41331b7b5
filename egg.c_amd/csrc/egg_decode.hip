// egg_decode.hip -- token-by-token continuation of one sequence (generate_sequence_kernel, mgpu.cu:1154-1283, and d-eggs'
// form of its sampler, d-eggs/src/kernels.cu:307-490) as one persistent launch on gfx950.
//
// A token of the unperturbed model is a chain of small matrix-vector products: what bounds it is not the weights (29 MB at
// hidden 512, 8 layers: 6 us at the memory's rate) but how fast one stage's result reaches the next stage's workgroups.
// As launches over one 32-token tile (one workgroup each, 2 L + 2 of them streaming whole matrices through one CU) a
// token took 1.76 ms at that size (vocabulary 8192) and 0.25 ms at hidden 256, 4 layers, vocabulary 256.  Here H / 16 workgroups stay for the whole
// continuation; workgroup w owns 16 columns of every H-wide product (48 of Q | K | V, 64 of the MLP's up projection, V / 16
// tiles of the head dealt round) and they exchange results through tagged messages: 8 bytes, the value and the number
// of the exchange, written and polled with device-scope accesses, so the data is its own arrival flag and an exchange costs
// one store-to-load trip (0.6 us on one XCD, 1.0 us across them) instead of a launch.  Everything every workgroup needs
// whole -- the residual row, the norms -- each computes for itself.  The weights of a stage are requested in front of the
// wait for its input.
//
// An exchange takes 1.2 to 2.2 us with the waits for the slowest workgroup, the short dependent computations between
// two of them 0.3 to 1.5 us, so their number counts.  Gathered, the attention's output and the MLP's intermediate are two exchanges a
// layer, and what the product of each gives are two more.  Up to hidden 256 a workgroup multiplies its own strip of them with the rows
// of the next matrix instead and the partial sums are exchanged (`Rows`): three exchanges a layer in place of five.
// Measured, 64 tokens behind a prompt of 32, alone and with three contexts that generate at the same time (one each
// finishes), five exchanges -> three: hidden 64, 2 layers 1.57 / 0.57 -> 1.22 / 0.43 ms; hidden 128, 4 layers 3.04 / 1.03 -> 2.29 / 0.78;
// hidden 256, 4 layers 2.95 / 1.06 -> 2.66 / 0.96; hidden 256, 8 layers, vocabulary 8192 5.65 / 2.10 -> 5.09 / 1.89.  Each workgroup reads H * H / 4
// bytes of messages for it, 16 KB at hidden 256 and 64 KB at 512, where such an exchange takes 2.5 to 3.2 us and the
// two-column messages 350 registers: 7.02 -> 7.24 ms alone, so hidden 512 gathers (97 us a token).
// All workgroups on one XCD were 5 % faster at hidden 256 and 8 % slower at 512 (the weights do not fit its L2), and several such
// launches would share that XCD.
//
// A message slot is written again one exchange of the same kind later.  Every workgroup sends in every exchange of a layer
// and takes in all it needs of an exchange before it sends in the next, so a slot is only written again when its last
// reader is past it.  Workgroups hold few resources (256 threads, two to a CU by their registers) and need not start together, only be
// resident together in the end.  A wait that is not answered within its bound raises `fail` and ends the launch; the launch
// behind it (k_decode_alone) then does the whole continuation with one workgroup, which waits for nobody, and clears the
// messages.  So a continuation always arrives, in stream order, and what is queued behind it finds everything in its initial state.
#include "egg_device.h"
#include "egg_launch.h"

#pragma clang fp contract(off)

namespace {

constexpr int THREADS = 256;
typedef unsigned long long u64;

// ---- messages
// slots: a uniform base and a lane's index
__device__ __forceinline__ void send(u64 *slots, uint32_t i, uint32_t tag, int value) {
    __hip_atomic_store(slots + i, ((u64)tag << 32) | (uint32_t)value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// N slots `stride` apart, all wanted with the same tag; slots from `count` on are not waited for.  false: not within `limit` polls
template <int N>
__device__ __forceinline__ bool receive(int (&out)[N], const u64 *slots, uint32_t first, uint32_t stride, int count, uint32_t tag, int limit) {
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = 0;
    for (int polls = 0; polls < limit; polls++) {
        u64 m[N];
#pragma unroll
        for (int i = 0; i < N; i++) m[i] = __hip_atomic_load(slots + (i < count ? first + i * stride : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool all = true;
#pragma unroll
        for (int i = 0; i < N; i++) { all &= i >= count || (uint32_t)(m[i] >> 32) == tag; out[i] = (int)(uint32_t)m[i]; }
        if (all) return true;
    }
    return count <= 0;
}

// ---- reductions
template <int N> __device__ __forceinline__ int row_ror(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x120 | N, 0xf, 0xf, false); }
template <bool MAX> __device__ __forceinline__ int join(int a, int b) { return MAX ? max(a, b) : a + b; }
// over the 16 lanes of a row; every lane gets the result
template <bool MAX> __device__ __forceinline__ int row_reduce(int v) {
    v = join<MAX>(v, row_ror<8>(v)); v = join<MAX>(v, row_ror<4>(v)); v = join<MAX>(v, row_ror<2>(v));
    return join<MAX>(v, row_ror<1>(v));
}
template <bool MAX> __device__ __forceinline__ int row_pair_reduce(int v) {          // rows 0, 1 and rows 2, 3
    const auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    return join<MAX>((int)r[0], (int)r[1]);
}
template <bool MAX> __device__ __forceinline__ int half_reduce(int v) {              // the two halves of the wave
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return join<MAX>((int)r[0], (int)r[1]);
}
template <bool MAX> __device__ __forceinline__ int wave_reduce(int v) { return half_reduce<MAX>(row_pair_reduce<MAX>(row_reduce<MAX>(v))); }
// over the workgroup; two calls in a row must use different `red`
template <bool MAX> __device__ __forceinline__ int wg_reduce(int v, int *red) {
    v = wave_reduce<MAX>(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return join<MAX>(join<MAX>(red[0], red[1]), join<MAX>(red[2], red[3]));
}
// inclusive sums over the wave: within the rows, then row 0 -> 1 and 2 -> 3, then the lower half -> the upper
__device__ __forceinline__ long long scan64(long long v) {
#define EGG_SCAN(CTRL, ROWS) v += ((long long)__builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xf, false) << 32) | \
                                  (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
    EGG_SCAN(0x111, 0xf) EGG_SCAN(0x112, 0xf) EGG_SCAN(0x114, 0xf) EGG_SCAN(0x118, 0xf) EGG_SCAN(0x142, 0xa) EGG_SCAN(0x143, 0xc)
#undef EGG_SCAN
    return v;
}
__device__ __forceinline__ long long lane64(long long v, int lane) {      // lane: uniform
    return ((long long)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32) | (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}

// byte position of hidden index k in slot order (egg_device.h), k a multiple of 4
__device__ __forceinline__ int slot_of(int k) { return (k & ~31) + 16 * ((k >> 2) & 1) + 4 * ((k >> 3) & 3); }

struct Lds {
    __align__(16) int8_t op[4 * 512];          // operand of the next product, slot order
    int part[4 * 64];                          // partial sums of a product, by wave
    int redm[4], reds[4], smax[4];
    int8_t x[512];                             // residual row
    int w[512];                                // attention weights
    int pv[64 * 17];                           // by group of positions: the strip's 16 weighted sums and the sum of the weights
    __align__(16) int8_t qs[64], ks[64], vs[16];      // the head's new query and key, the strip's new value
    __align__(16) int8_t own[64];                     // the strip's attention output, its columns of the MLP's intermediate
    int lut[256]; int8_t act[256];
    long long tsum[64];
    int tok[512];                              // the sequence
    int dead;
};

// One column strip's part of a product: T tiles of 16 columns, K inputs.  Lane (pl, n) of wave q takes the 16-byte units
// p = 16 i + 4 q + pl of column n (fragment-major copy), so a load instruction reads four runs of 256 bytes.
template <int T, int K>
struct Strip {
    static constexpr int P = K / 16, IT = P < 16 ? 1 : P / 16;
    v4i w[T * IT];
    // tile t <- columns [col, col + 16) of a matrix of `cols` columns whose fragment-major blocks are B wide
    template <int B>
    __device__ __forceinline__ void load(int t, const int8_t *frag, int cols, int col) {
        const uint32_t wave = threadIdx.x >> 6, pl = (threadIdx.x >> 4) & 3, n = (uint32_t)col + (threadIdx.x & 15);
        // a uniform base and 32-bit offsets: no 64-bit address arithmetic, no address registers
        uint32_t at = n / B * (B * B) + n % B * 16;
        // computed here and not ahead of the loop over the layers, where the offsets of all loads take registers that the sums need
        if constexpr (egg_decode_sums(K)) asm volatile("" : "+v"(at));
#pragma unroll
        for (int i = 0; i < IT; i++) {
            const uint32_t p = 16 * i + 4 * wave + pl;
            if (P >= 16 || p < P) w[t * IT + i] = *reinterpret_cast<const v4i *>(frag + (at + p / (B / 16) * ((uint32_t)cols * B) + p % (B / 16) * (B * 16)));
        }
    }
    // the T * 16 sums, one per thread (threads below T * 16); synchronises twice: in front (operand written) and inside
    __device__ __forceinline__ int finish(Lds &s) {
        const int wave = threadIdx.x >> 6, pl = (threadIdx.x >> 4) & 3, n = threadIdx.x & 15;
        __syncthreads();
        int acc[T];
#pragma unroll
        for (int t = 0; t < T; t++) acc[t] = 0;
#pragma unroll
        for (int i = 0; i < IT; i++) {
            const int p = 16 * i + 4 * wave + pl;
            if (P >= 16 || p < P) {
                const v4i x = *reinterpret_cast<const v4i *>(s.op + p * 16);
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[t] = dot4(w[t * IT + i][q], x[q], acc[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int v = half_reduce<false>(row_pair_reduce<false>(acc[t]));
            if (pl == 0) s.part[wave * (T * 16) + t * 16 + n] = v;
        }
        __syncthreads();
        const int i = threadIdx.x;
        return i < T * 16 ? s.part[i] + s.part[T * 16 + i] + s.part[2 * T * 16 + i] + s.part[3 * T * 16 + i] : 0;
    }
};

template <int H>
struct Norm {                                   // gains and biases of a standard norm, a thread's elements k = tid + 256 i
    static constexpr int NE = (H + 255) / 256;
    int w[NE], b[NE];
    __device__ __forceinline__ void load(const int8_t *ln_w, const int8_t *ln_b) {
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int k = threadIdx.x + 256 * i;
            w[i] = k < H ? ln_w[(uint32_t)k] : 0; b[i] = k < H ? ln_b[(uint32_t)k] : 0;
        }
    }
    // apply_standard_norm (mgpu.cu:646-678) of x -> s.op; |x w| <= 127 * 127, so the quotient may go through floats
    __device__ __forceinline__ void apply(Lds &s, const int (&x)[NE]) {
        int tot = 0;
#pragma unroll
        for (int i = 0; i < NE; i++) tot += abs(x[i]);
        int mn = wg_reduce<false>(tot, s.reds) / H;
        if (!mn) mn = 1;
        const float rcp = 1.0f / (float)mn;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int k = threadIdx.x + 256 * i;
            if (k < H) s.op[slot_of(k & ~3) + (k & 3)] = (int8_t)clip127(div_trunc(x[i] * w[i], rcp) + b[i]);
        }
    }
};

// the residual values of an exchange: adaptive norm (egg_adaptive_normalize.h:10-103) -> new residual row, in x and in s.x
template <int H>
__device__ __forceinline__ bool take_residual(Lds &s, const u64 *slots, uint32_t tag, int (&x)[Norm<H>::NE], int limit) {
    constexpr int NE = Norm<H>::NE;
    const int tid = threadIdx.x;
    int v[NE];
    if (!receive<NE>(v, slots, tid, 256, tid < H ? NE : 0, tag, limit)) s.dead = 1;
    int mx = 0;
#pragma unroll
    for (int i = 0; i < NE; i++) { if (tid >= H) v[i] = 0; mx = max(mx, abs(v[i])); }
    mx = wg_reduce<true>(mx, s.redm);
    const float scale = 127.0f / ((float)mx + 1e-9f);
#pragma unroll
    for (int i = 0; i < NE; i++) {
        x[i] = round_half_away((float)v[i] * scale);
        if (tid < H) s.x[tid + 256 * i] = (int8_t)x[i];
    }
    return !s.dead;
}

// ---- products of a strip of rows, up to hidden 256: workgroup w multiplies its own R values (of the attention's output, of the MLP's
// intermediate) with the R rows of the next matrix that belong to them, which lie together in the canonical blocked weights, and sends
// the partial sums of every column; a receiver adds up the H / 16 of them.  They are exact integers, so the sums are
// what a product of the gathered row gives, and the row itself is never exchanged.
// A message holds two columns' sums of 21 bits (64 * 127 * 128 < 2^20) and 22 bits of the exchange's number: what a slot held before
// is the exchange in front, so far fewer would tell them apart.
constexpr uint32_t TAG22 = (1u << 22) - 1u;
template <int H, int R>
struct Rows {
    static constexpr int D = R / 8;             // a thread's column pair and its half of the rows: the other half is 32 lanes away
    int2 w[D];
    static __device__ __forceinline__ int pair() { return (int)((threadIdx.x >> 6) * 32 + (threadIdx.x & 31)); }
    static __device__ __forceinline__ int half() { return (int)((threadIdx.x >> 5) & 1); }
    __device__ __forceinline__ void load(const int8_t *W, int row0) {           // W: uniform
        if (pair() >= H / 2) return;
        uint32_t at = half() * (D * H * 4) + 8 * pair();
        asm volatile("" : "+v"(at));
        W += (uint32_t)(row0 >> 2) * H * 4u;
#pragma unroll
        for (int i = 0; i < D; i++) w[i] = *reinterpret_cast<const int2 *>(W + (at + i * H * 4u));
    }
    __device__ __forceinline__ void send_sums(const int8_t *values, u64 *slots, int wg, uint32_t tag) const {
        int a = 0, b = 0;
        if (pair() < H / 2) {
#pragma unroll
            for (int i = 0; i < D; i++) {
                const int v = *reinterpret_cast<const int *>(values + 4 * (half() * D + i));
                a = dot4(w[i].x, v, a); b = dot4(w[i].y, v, b);
            }
        }
        a = half_reduce<false>(a); b = half_reduce<false>(b);
        if (pair() < H / 2 && half() == 0)
            __hip_atomic_store(slots + (uint32_t)(wg * (H / 2) + pair()), ((u64)(tag & TAG22) << 42) | ((u64)((uint32_t)b & 0x1fffffu) << 21) | ((uint32_t)a & 0x1fffffu),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
// x + (sum >> shift) + bias of an exchange of partial sums, then the adaptive norm (egg_adaptive_normalize.h:10-103) -> new residual row
// Thread k has column k; it takes half of the messages of its pair of columns, its neighbour the other half.
template <int H>
__device__ __forceinline__ bool take_sums(Lds &s, const u64 *slots, uint32_t tag, int shift, int bias, int &x, int limit) {
    constexpr int M = H / 32;
    const int tid = threadIdx.x;
    int v = 0;
    if (tid < H) {
        bool all = false;
        int lo = 0, hi = 0;
        const u64 *from = slots + ((tid >> 1) + (tid & 1) * (M * (H / 2)));
        asm volatile("" : "+v"(from));           // one address and offsets: M addresses for each exchange would be kept over the layers
        for (int polls = 0; polls < limit && !all; polls++) {
            u64 m[M];
#pragma unroll
            for (int g = 0; g < M; g++) m[g] = __hip_atomic_load(from + g * (H / 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            all = true;
            lo = hi = 0;
#pragma unroll
            for (int g = 0; g < M; g++) {
                all &= (uint32_t)(m[g] >> 42) == (tag & TAG22);
                lo += (int)((uint32_t)m[g] << 11) >> 11;
                hi += (int)((uint32_t)(m[g] >> 21) << 11) >> 11;
            }
        }
        if (!all) s.dead = 1;
        v = (tid & 1 ? hi : lo) + __builtin_amdgcn_update_dpp(0, tid & 1 ? lo : hi, 0xB1, 0xf, 0xf, false);
        v = x + (v >> shift) + bias;
    }
    const int mx = wg_reduce<true>(abs(v), s.redm);
    x = round_half_away((float)v * (127.0f / ((float)mx + 1e-9f)));
    return !s.dead;
}
template <int H>
__device__ __forceinline__ bool take(Lds &s, const u64 *slots, uint32_t tag, int shift, int bias, int (&x)[Norm<H>::NE], int limit) {
    if constexpr (egg_decode_sums(H)) return take_sums<H>(s, slots, tag, shift, bias, x[0], limit);
    else return take_residual<H>(s, slots, tag, x, limit);
}

__device__ __forceinline__ int exp_of(const Lds &s, const DecodeParams &p, int logit, int mx) {
    if (!p.deggs) {
        const int d = mx - logit;
        return s.lut[d < 0 ? 0 : (d > 255 ? 255 : d)];
    }
    const int shifted = (int)((uint32_t)logit - (uint32_t)mx);
    const float q = (float)shifted / p.temp;
    // float -> int32 as the reference's GPU converts it: truncation, saturation at the ends, NaN -> 0
    const int scaled = q != q ? 0 : (q >= 2147483648.0f ? INT_MAX : (q <= -2147483648.0f ? INT_MIN : (int)q));
    if (scaled < p.min_p_limit) return 0;
    const int idx = (int)(0u - (uint32_t)scaled);
    return s.lut[idx < 0 ? 0 : (idx > 255 ? 255 : idx)];
}

// a wait ran into its bound: say so and leave (the others run into theirs, and who has not started yet does not begin)
__device__ void give_up(const DecodeParams &p) {
    if (threadIdx.x == 0) __hip_atomic_store(p.fail, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The sampler (mgpu.cu:1212-1283, d-eggs/src/kernels.cu:382-478): maximum, table weights, threshold hash_rng(seed + 555 t, 0)
// % sum, first entry whose running sum exceeds it in the order of the reference's threads: thread r of bt = H owns v = r,
// r + H, ...  Workgroup w's head tiles are columns 16 w + H i, i.e. exactly those of threads 16 w .. 16 w + 15, so it
// keeps its logits to itself (`logit`: entry 16 i + n is column 16 w + n + H i); two exchanges, the maxima and the sums,
// make the rest local: the workgroup in whose threads the threshold falls picks the entry and sends it round.
template <int H>
__device__ bool sample(Lds &s, int *logit, int count, const DecodeParams &p, int wg, u64 *m_max, u64 *m_sum, u64 *m_tok, uint32_t tag, int t) {
    constexpr int G = H / 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = tid & 15;
    if (p.deggs && p.penalty_int) {
        // every earlier occurrence of a token lowers its logit (d-eggs/src/kernels.cu:398-402)
        for (int i = tid; i <= t; i += THREADS) {
            const int v = s.tok[i];
            if ((unsigned)v < (unsigned)p.vocab && v % H / 16 == wg) atomicSub(&logit[v / H * 16 + v % 16], p.penalty_int);
        }
        __syncthreads();
    }
    int mx = INT_MIN;
    for (int i = tid; i < count; i += THREADS) mx = max(mx, logit[i]);
    mx = wg_reduce<true>(mx, s.redm);
    if (tid == 0) send(m_max, wg, tag, mx);
    if (wave == 0) {
        int got[1];
        if (!receive<1>(got, m_max, lane & 31, 0, (lane & 31) < G ? 1 : 0, tag, p.wait_limit)) s.dead = 1;
        mx = row_pair_reduce<true>(row_reduce<true>((lane & 31) < G ? got[0] : INT_MIN));
        if (lane == 0) s.smax[0] = mx;
    }
    __syncthreads();
    if (s.dead) return false;
    mx = s.smax[0];
    long long sum = 0;
    for (int i = tid; i < count; i += THREADS) sum += exp_of(s, p, logit[i], mx);          // all of reference thread 16 wg + n
    sum += __shfl_xor(sum, 16, 64); sum += __shfl_xor(sum, 32, 64);
    if (lane < 16) s.tsum[wave * 16 + n] = sum;
    __syncthreads();
    if (wave == 0) {
        const long long mine = s.tsum[n] + s.tsum[16 + n] + s.tsum[32 + n] + s.tsum[48 + n];
        const long long upto16 = scan64(lane < 16 ? mine : 0), all = lane64(upto16, 63);
        if (lane < 2) send(m_sum, 2 * wg + lane, tag, (int)(lane ? all >> 32 : all));
        int got[2];
        if (!receive<2>(got, m_sum, 2 * (lane & 31), 1, (lane & 31) < G ? 2 : 0, tag, p.wait_limit)) s.dead = 1;
        const long long theirs = lane < G ? ((long long)got[1] << 32) | (uint32_t)got[0] : 0;
        const long long upto = scan64(theirs), total = lane64(upto, 63);
        const uint32_t r = hash_rng(p.seed + (uint32_t)t * 555u, 0);
        const long long thresh = total > 0 ? ((long long)r < total ? (long long)r : (long long)(r % (uint32_t)total)) : 0;
        // of all workgroups the first whose running sum exceeds the threshold; none (every entry left out): token 0
        const u64 over = __ballot(upto > thresh);
        const int owner = over ? __builtin_ctzll(over) : 0;
        int got1[1];
        if (owner == wg && !s.dead) {
            int sel = 0;
            if (over) {
                long long before = lane64(upto - theirs, wg);
                const int at = __builtin_ctzll(__ballot(before + upto16 > thresh));
                before += lane64(upto16 - mine, at);
                for (int k0 = 0; 16 * k0 + at < count; k0 += 64) {
                    const int i = 16 * (k0 + lane) + at;
                    const long long in = scan64(i < count ? exp_of(s, p, logit[i], mx) : 0);
                    const u64 hit = __ballot(before + in > thresh);
                    if (hit) { sel = 16 * wg + at + H * (k0 + __builtin_ctzll(hit)); break; }
                    before += lane64(in, 63);
                }
            }
            if (lane == 0) {
                send(m_tok, 0, tag, sel);
                if (p.token_bytes == 4) reinterpret_cast<uint32_t *>(p.out)[t + 1] = (uint32_t)sel;
                else reinterpret_cast<uint8_t *>(p.out)[t + 1] = (uint8_t)sel;
            }
        }
        if (lane == 0) { if (receive<1>(got1, m_tok, 0, 0, 1, tag, p.wait_limit)) s.tok[t + 1] = got1[0]; else s.dead = 1; }
    }
    __syncthreads();
    return !s.dead;
}

// two workgroups to a CU, 256 registers; asked for at hidden 512, which has them anyway, the bound costs 1 % of its time
template <int H>
__global__ void __launch_bounds__(THREADS, egg_decode_sums(H) ? 2 : 1) k_decode(DecodeParams p) {
    constexpr int G = H / 16, NE = Norm<H>::NE;
    constexpr bool SUMS = egg_decode_sums(H);
    __shared__ Lds s;
    extern __shared__ int logit[];              // this workgroup's V / H logits of its 16 columns
    const int wg = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c0 = 16 * wg;
    const int hd = p.head_dim, strips = hd / 16, head = wg / strips, T = p.T, V = p.vocab;
    constexpr int N_AO = SUMS ? 0 : H, N_UP = SUMS ? 0 : H, N_RES = SUMS ? G * (H / 2) : H;
    u64 *const m_qkv = p.slots, *const m_ao = m_qkv + G * 64, *const m_res = m_ao + N_AO, *const m_up = m_res + N_RES, *const m_dn = m_up + N_UP,
               *const m_max = m_dn + N_RES, *const m_sum = m_max + G, *const m_tok = m_sum + 2 * G;
    int8_t *const kc = p.kcache + (size_t)wg * p.n_layers * T * hd, *const vc = p.vcache + (size_t)wg * p.n_layers * T * 16;
    const int8_t *const M = p.model, *const F = p.frag;
    const uint32_t hh = (uint32_t)H * H, h4 = 4u * H;
    uint32_t tag = *p.epoch + 1u;
    if (tid == 0) s.dead = 0;
    s.lut[tid] = p.exp_lut[tid]; s.act[tid] = p.act_lut[tid];
    for (int i = tid; i <= p.t_first; i += THREADS) s.tok[i] = p.token_bytes == 4 ? (int)reinterpret_cast<const uint32_t *>(p.tokens)[i] : (int)p.tokens[i];
    // the prompt's K / V rows (slot order, [layer][K, V][T][H]) -> this workgroup's own copies: its head's keys, its strip's values
    for (int l = 0; l < p.n_layers; l++) {
        const int8_t *K = p.kv + (size_t)(2 * l) * T * H, *Vv = K + (size_t)T * H;
        const int kd = hd / 4;
        for (int i = tid; i < p.t_first * kd; i += THREADS) {
            const int row = i / kd, d = i % kd;
            *reinterpret_cast<int *>(kc + ((size_t)l * T + row) * hd + 4 * d) = *reinterpret_cast<const int *>(K + (size_t)row * H + slot_of(head * hd + 4 * d));
        }
        for (int i = tid; i < p.t_first * 4; i += THREADS) {
            const int row = i >> 2, d = i & 3;
            *reinterpret_cast<int *>(vc + ((size_t)l * T + row) * 16 + 4 * d) = *reinterpret_cast<const int *>(Vv + (size_t)row * H + slot_of(c0 + 4 * d));
        }
    }
    if (tid == 0 && __hip_atomic_load(p.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) s.dead = 1;
    __syncthreads();
    if (s.dead) return;
    const uint32_t steps = (uint32_t)p.n_layers + 2u;
    for (int t = p.t_first; t < p.t_first + p.count; t++, tag += steps) {
        // ---- embedding (mgpu.cu:901-934, ns = 0)
        int x[NE];
        Norm<H> ln; ln.load(M + p.ln_init, M + p.ln_init_bias);
        const int token = s.tok[t];
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int k = tid + 256 * i;
            x[i] = k < H ? clip127((int)(M + p.embedding)[((uint32_t)(k >> 2) * V + token) * 4 + (k & 3)] + (int)(M + p.emb_bias)[(uint32_t)k]) : 0;
            if (k < H) s.x[k] = (int8_t)x[i];
        }
        int bd = 0;                            // of the down projection in front, where its sums are exchanged
        for (int l = -1; l < p.n_layers; l++) {
            const uint32_t tg = tag + (uint32_t)(l + 1);
            if (l >= 0) {
                // ---- Q | K | V of the strip, RoPE, and the maxima of the adaptive norms
                Strip<3, H> qkv;
                qkv.template load<H>(0, F + (p.w_q + l * hh), H, c0);
                qkv.template load<H>(1, F + (p.w_k + l * hh), H, c0);
                qkv.template load<H>(2, F + (p.w_v + l * hh), H, c0);
                const int row = (tid >> 4) & 3, n = tid & 15;
                const int rope_at = t * hd + ((c0 + n) % hd & ~1);
                const int cs = p.rope_lut[rope_at], sn = p.rope_lut[rope_at + 1];
                if (!take<H>(s, m_dn, tg - 1, p.shift_dn, bd, x, p.wait_limit)) return give_up(p);
                ln.apply(s, x);
                const int acc = qkv.finish(s);
                v4i kr[2][4]; int vr[8];
                int8_t *const kl = kc + (size_t)l * T * hd, *const vl = vc + (size_t)l * T * 16;
                const int pg = tid >> 2, dq = tid & 3;
#pragma unroll
                for (int i = 0; i < 2; i++)
                    if (tid + 256 * i < t) {
                        const uint32_t at = (uint32_t)(tid + 256 * i) * hd;
                        kr[i][0] = *reinterpret_cast<const v4i *>(kl + at); kr[i][1] = *reinterpret_cast<const v4i *>(kl + (at + 16));
                        if (hd == 64) { kr[i][2] = *reinterpret_cast<const v4i *>(kl + (at + 32)); kr[i][3] = *reinterpret_cast<const v4i *>(kl + (at + 48)); }
                    }
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (64 * i < t && pg + 64 * i < t) vr[i] = *reinterpret_cast<const int *>(vl + (uint32_t)(4 * tid + 1024 * i));
                int mine = acc;
                if (tid < 64) {
                    const int nb = __builtin_amdgcn_update_dpp(0, acc, 0xB1, 0xf, 0xf, false);
                    const long long half = 1ll << (p.rope_bit - 1);
                    const long long rot = (n & 1) ? (long long)nb * sn + (long long)acc * cs : (long long)acc * cs - (long long)nb * sn;
                    if (row < 2) mine = (int)((rot + half) >> p.rope_bit);
                    const int mx = row_reduce<true>(abs(mine));
                    if (row < 2) send(m_qkv, wg * 64 + tid, tg, mine);
                    if (row < 3 && n == 0) send(m_qkv, wg * 64 + 48 + row, tg, mx);
                }
                // threads 0..95: the maxima of all strips; threads 128..255: query and key of the head
                const bool head_thread = tid >= 128 && lane < hd, max_thread = tid < 96 && (tid & 31) < G;
                int got[1];
                if (!receive<1>(got, m_qkv, head_thread ? (head * strips + lane / 16) * 64 + (tid < 192 ? 0 : 16) + (lane & 15) : (tid & 31) * 64 + 48 + (tid >> 5), 0,
                                head_thread || max_thread ? 1 : 0, tg, p.wait_limit)) s.dead = 1;
                const int mx32 = row_pair_reduce<true>(row_reduce<true>(max_thread ? got[0] : 0));
                if (tid < 96 && (tid & 31) == 0) s.smax[tid >> 5] = mx32;
                __syncthreads();
                if (s.dead) return give_up(p);
                if (head_thread) {
                    const float scale = 127.0f / ((float)s.smax[tid < 192 ? 0 : 1] + 1e-9f);
                    (tid < 192 ? s.qs : s.ks)[lane] = (int8_t)round_half_away((float)got[0] * scale);
                }
                if (tid < 64 && row == 2) s.vs[n] = (int8_t)round_half_away((float)mine * (127.0f / ((float)s.smax[2] + 1e-9f)));
                __syncthreads();
                if (tid < hd / 4) *reinterpret_cast<int *>(kl + (uint32_t)(t * hd + 4 * tid)) = reinterpret_cast<const int *>(s.ks)[tid];
                else if (tid >= 64 && tid < 68) *reinterpret_cast<int *>(vl + (uint32_t)(t * 16 + 4 * (tid - 64))) = reinterpret_cast<const int *>(s.vs)[tid - 64];
                Rows<H, 16> wo_rows; Strip<1, H> wo;
                if constexpr (SUMS) wo_rows.load(M + (p.w_o + l * hh), c0); else wo.template load<H>(0, F + (p.w_o + l * hh), H, c0);
                int sc[2], mx = INT_MIN;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int at = tid + 256 * i;
                    sc[i] = INT_MIN;
                    if (at > t) continue;
                    if (at == t) {
#pragma unroll
                        for (int d = 0; d < 4; d++) kr[i][d] = reinterpret_cast<const v4i *>(s.ks)[d];
                    }
                    int a = 0;
#pragma unroll
                    for (int d = 0; d < 4; d++)
                        if (d < 2 || hd == 64) {
                            const v4i q4 = reinterpret_cast<const v4i *>(s.qs)[d];
#pragma unroll
                            for (int e = 0; e < 4; e++) a = dot4(kr[i][d][e], q4[e], a);
                        }
                    sc[i] = a >> p.shift_attn;
                    mx = max(mx, sc[i]);
                }
                mx = wg_reduce<true>(mx, s.redm);
#pragma unroll
                for (int i = 0; i < 2; i++)
                    if (tid + 256 * i <= t) { const int d = mx - sc[i]; s.w[tid + 256 * i] = s.lut[d > 255 ? 255 : d]; }
                __syncthreads();
                int sum[4] = {0, 0, 0, 0}, tot = 0;
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (64 * i > t) break;
                    const int at = pg + 64 * i;
                    const int w = at <= t ? s.w[at] : 0, v4 = at == t ? reinterpret_cast<const int *>(s.vs)[dq] : vr[i];
#pragma unroll
                    for (int e = 0; e < 4; e++) sum[e] += mul24(w, sx8(v4, e));
                    tot += w;
                }
#pragma unroll
                for (int e = 0; e < 4; e++) s.pv[pg * 17 + 4 * dq + e] = sum[e];
                if (dq == 0) s.pv[pg * 17 + 16] = tot;
                __syncthreads();
                {
                    const int col = tid >> 4, part = tid & 15;
                    int lo = 0, hi = 0, den = 0;
#pragma unroll
                    for (int i = 0; i < 4; i++) { const int v = s.pv[(4 * part + i) * 17 + col]; lo += v & 0xffff; hi += v >> 16; den += s.pv[(4 * part + i) * 17 + 16]; }
                    lo = row_reduce<false>(lo); hi = row_reduce<false>(hi); den = row_reduce<false>(den);
                    den = den ? den : 1;
                    const long long num = ((long long)hi << 16) + lo, mag = num < 0 ? -num : num;
                    int quo = (int)((float)mag * __builtin_amdgcn_rcpf((float)den));
                    const long long rest = mag - (long long)quo * den;
                    quo += rest < 0 ? -1 : (rest >= den ? 1 : 0);
                    const int r = num < 0 ? -quo : quo;
                    const int packed = pack4(__builtin_amdgcn_readlane(r, 0), __builtin_amdgcn_readlane(r, 16), __builtin_amdgcn_readlane(r, 32), __builtin_amdgcn_readlane(r, 48));
                    if ((tid & 63) == 0) { if constexpr (SUMS) reinterpret_cast<int *>(s.own)[wave] = packed; else send(m_ao, 4 * wg + wave, tg, packed); }
                }
                // ---- output projection of the strip, residual
                if constexpr (SUMS) {
                    __syncthreads();
                    wo_rows.send_sums(s.own, m_res, wg, tg);
                } else {
                    int a[1];
                    if (!receive<1>(a, m_ao, tid, 0, tid < H / 4 ? 1 : 0, tg, p.wait_limit)) s.dead = 1;
                    if (tid < H / 4) *reinterpret_cast<int *>(s.op + slot_of(4 * tid)) = a[0];
                    const int o = wo.finish(s);
                    if (s.dead) return give_up(p);
                    if (tid < 16) send(m_res, c0 + tid, tg, (int)s.x[c0 + tid] + (o >> p.shift_out));
                }
            }
            // ---- MLP (mgpu.cu:708-759): up projection of 64 columns, table, down projection of the strip, residual
            const int8_t *b_up = M + (l < 0 ? p.b_up_init : p.b_up + l * h4), *b_dn = M + (l < 0 ? p.b_dn_init : p.b_dn + l * (uint32_t)H);
            Strip<4, H> up;
#pragma unroll
            for (int i = 0; i < 4; i++) up.template load<H>(i, F + (l < 0 ? p.w_up_init : p.w_up + 4 * l * hh), 4 * H, 64 * wg + 16 * i);
            const int bu = tid < 64 ? b_up[(uint32_t)(64 * wg + tid)] : 0;
            Rows<H, 64> dn_rows;
            if constexpr (SUMS) dn_rows.load(M + (l < 0 ? p.w_dn_init : p.w_dn + 4 * l * hh), 64 * wg);
            if (l >= 0) {
                ln.load(M + (p.ln_2 + l * (uint32_t)H), M + (p.ln_2_bias + l * (uint32_t)H));
                if (!take<H>(s, m_res, tg, p.shift_out, 0, x, p.wait_limit)) return give_up(p);
            }
            ln.apply(s, x);
            const int a = up.finish(s), g = tid < 64 ? (int)s.act[(uint8_t)clip127((a >> p.shift_up) + bu)] : 0;
            if constexpr (SUMS) {
                if (tid < 64) s.own[tid] = (int8_t)g;
                __syncthreads();
                dn_rows.send_sums(s.own, m_dn, wg, tg);
                bd = tid < H ? (int)b_dn[(uint32_t)tid] : 0;
            } else {
                if (tid < 64) {
                    const int g0 = g & 255, g1 = __builtin_amdgcn_update_dpp(0, g0, 0x55, 0xf, 0xf, false), g2 = __builtin_amdgcn_update_dpp(0, g0, 0xAA, 0xf, 0xf, false),
                              g3 = __builtin_amdgcn_update_dpp(0, g0, 0xFF, 0xf, 0xf, false);     // lanes 1, 2, 3 of the quad
                    if ((tid & 3) == 0) send(m_up, 16 * wg + (tid >> 2), tg, g0 | (g1 << 8) | (g2 << 16) | (g3 << 24));
                }
                Strip<1, 4 * H> dn; dn.template load<H>(0, F + (l < 0 ? p.w_dn_init : p.w_dn + 4 * l * hh), H, c0);
                const int b = tid < 16 ? b_dn[(uint32_t)(c0 + tid)] : 0;
                int up4[NE];
                if (!receive<NE>(up4, m_up, tid, 256, tid < H ? NE : 0, tg, p.wait_limit)) s.dead = 1;
#pragma unroll
                for (int i = 0; i < NE; i++)
                    if (tid < H) *reinterpret_cast<int *>(s.op + slot_of(4 * (tid + 256 * i))) = up4[i];
                const int d = dn.finish(s);
                if (s.dead) return give_up(p);
                if (tid < 16) send(m_dn, c0 + tid, tg, (int)s.x[c0 + tid] + (d >> p.shift_dn) + b);
            }
            // the next norm's gains: the next layer's first, or the last
            const bool last = l + 1 == p.n_layers;
            ln.load(M + (last ? p.ln_f : p.ln_1 + (l + 1) * (uint32_t)H), M + (last ? p.ln_f_bias : p.ln_1_bias + (l + 1) * (uint32_t)H));
        }
        // ---- head: tiles of 16 columns dealt round, four at a time
        const uint32_t tg = tag + (uint32_t)p.n_layers + 1u;
        constexpr int BLOCK = H > 256 ? 256 : H;
        if (!take<H>(s, m_dn, tg - 1, p.shift_dn, bd, x, p.wait_limit)) return give_up(p);
        ln.apply(s, x);
        int count = 0;                          // logits of this workgroup
        for (int t0 = wg; t0 < V / 16; t0 += 4 * G) {
            if (t0 + 3 * G < V / 16) {
                Strip<4, H> lg;
#pragma unroll
                for (int i = 0; i < 4; i++) lg.template load<BLOCK>(i, F + p.embedding, V, 16 * (t0 + i * G));
                const int a = lg.finish(s);
                if (tid < 64) logit[count + tid] = a >> p.shift_logit;
                count += 64;
            } else
                for (int tt = t0; tt < V / 16; tt += G, count += 16) {
                    Strip<1, H> lg; lg.template load<BLOCK>(0, F + p.embedding, V, 16 * tt);
                    const int a = lg.finish(s);
                    if (tid < 16) logit[count + tid] = a >> p.shift_logit;
                }
        }
        __syncthreads();
        if (!sample<H>(s, logit, count, p, wg, m_max, m_sum, m_tok, tg, t)) return give_up(p);
    }
    // every workgroup has read the epoch before it sent anything, and workgroup 0 has heard from all of them
    if (wg == 0 && tid == 0) *p.epoch = tag;
}

// The same continuation by one workgroup, if the launch in front gave up: no exchange, nothing to wait for.  It reads the canonical
// weights (a thread a column), keeps the K / V rows behind the prompt's and the logits in memory, and then puts messages, epoch
// and flag back to what a first launch finds.  Written to be right, not fast (0.2 ms a token at hidden 256, 4 layers,
// 2.1 ms at hidden 512, 8 layers, vocabulary 8192); with nothing to do its launch does not show in a continuation's time.
struct Alone {
    int8_t q[512], ao[512];                     // slot order
    int wide[3 * 512];                          // results of a product, by column
    long long tsum[512];
    int tok;
};
__device__ __forceinline__ int column(const Lds &s, const int8_t *W, int K, int N, int n) {
    const int *w = reinterpret_cast<const int *>(W) + n;
    int acc = 0;
    for (int k = 0; k < K / 4; k++) acc = dot4(w[(size_t)k * N], *reinterpret_cast<const int *>(s.op + slot_of(4 * k)), acc);
    return acc;
}
template <int H>
__global__ void __launch_bounds__(THREADS) k_decode_alone(DecodeParams p) {
    constexpr int NE = Norm<H>::NE;
    __shared__ Lds s;
    __shared__ Alone a;
    if (!*p.fail) return;
    const int tid = threadIdx.x, T = p.T, V = p.vocab, hd = p.head_dim;
    const int8_t *const M = p.model;
    const size_t hh = (size_t)H * H;
    s.lut[tid] = p.exp_lut[tid]; s.act[tid] = p.act_lut[tid];
    for (int i = tid; i <= p.t_first; i += THREADS) s.tok[i] = p.token_bytes == 4 ? (int)reinterpret_cast<const uint32_t *>(p.tokens)[i] : (int)p.tokens[i];
    __syncthreads();
    int x[NE];
    Norm<H> ln;
    auto byte_of = [](int k) { return slot_of(k & ~3) + (k & 3); };
    // adaptive norm of H values of a.wide (egg_adaptive_normalize.h:10-103) -> out(k, value)
    auto adapt = [&](const int *v, auto out) {
        __syncthreads();
        int mx = 0;
        for (int k = tid; k < H; k += THREADS) mx = max(mx, abs(v[k]));
        mx = wg_reduce<true>(mx, s.redm);
        const float scale = 127.0f / ((float)mx + 1e-9f);
        for (int k = tid; k < H; k += THREADS) out(k, round_half_away((float)v[k] * scale));
        __syncthreads();
    };
    auto residual = [&] {                       // a.wide -> the residual row
        adapt(a.wide, [&](int k, int v) { s.x[k] = (int8_t)v; });
#pragma unroll
        for (int i = 0; i < NE; i++) { const int k = tid + 256 * i; x[i] = k < H ? (int)s.x[k] : 0; }
    };
    auto norm = [&](uint32_t w, uint32_t b) { ln.load(M + w, M + b); ln.apply(s, x); __syncthreads(); };
    for (int t = p.t_first; t < p.t_first + p.count; t++) {
        const int token = s.tok[t];
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int k = tid + 256 * i;
            x[i] = k < H ? clip127((int)(M + p.embedding)[((size_t)(k >> 2) * V + token) * 4 + (k & 3)] + (int)(M + p.emb_bias)[k]) : 0;
            if (k < H) s.x[k] = (int8_t)x[i];
        }
        for (int l = -1; l < p.n_layers; l++) {
            if (l >= 0) {
                norm(p.ln_1 + l * (uint32_t)H, p.ln_1_bias + l * (uint32_t)H);
                for (int n = tid; n < H; n += THREADS) {
                    a.wide[n] = column(s, M + p.w_q + l * hh, H, H, n);
                    a.wide[H + n] = column(s, M + p.w_k + l * hh, H, H, n);
                    a.wide[2 * H + n] = column(s, M + p.w_v + l * hh, H, H, n);
                }
                __syncthreads();
                for (int i = tid; i < H; i += THREADS) {          // RoPE of the pairs of Q, then of K
                    int *v = a.wide + 2 * i;
                    const int at = t * hd + 2 * i % H % hd;
                    const long long c = p.rope_lut[at], sn = p.rope_lut[at + 1], half = 1ll << (p.rope_bit - 1), v0 = v[0], v1 = v[1];
                    v[0] = (int)((v0 * c - v1 * sn + half) >> p.rope_bit);
                    v[1] = (int)((v0 * sn + v1 * c + half) >> p.rope_bit);
                }
                int8_t *const K = p.kv + (size_t)(2 * l) * T * H, *const Vv = K + (size_t)T * H;
                adapt(a.wide, [&](int k, int v) { a.q[byte_of(k)] = (int8_t)v; });
                adapt(a.wide + H, [&](int k, int v) { K[(size_t)t * H + byte_of(k)] = (int8_t)v; });
                adapt(a.wide + 2 * H, [&](int k, int v) { Vv[(size_t)t * H + byte_of(k)] = (int8_t)v; });
                for (int c0 = 0; c0 < H; c0 += hd) {              // a head
                    int mx = INT_MIN;
                    for (int at = tid; at <= t; at += THREADS) {
                        int d = 0;
                        for (int i = 0; i < hd / 4; i++)
                            d = dot4(*reinterpret_cast<const int *>(K + (size_t)at * H + c0 + 4 * i), *reinterpret_cast<const int *>(a.q + c0 + 4 * i), d);
                        s.w[at] = d >> p.shift_attn;
                        mx = max(mx, s.w[at]);
                    }
                    mx = wg_reduce<true>(mx, s.smax);
                    for (int at = tid; at <= t; at += THREADS) s.w[at] = s.lut[min(mx - s.w[at], 255)];
                    __syncthreads();
                    if (tid < hd) {
                        const int at0 = byte_of(c0 + tid);
                        long long num = 0, den = 0;
                        for (int at = 0; at <= t; at++) { num += (long long)s.w[at] * Vv[(size_t)at * H + at0]; den += s.w[at]; }
                        a.ao[at0] = (int8_t)(num / (den ? den : 1));
                    }
                    __syncthreads();
                }
                for (int k = tid; k < H / 4; k += THREADS) reinterpret_cast<int *>(s.op)[k] = reinterpret_cast<const int *>(a.ao)[k];
                __syncthreads();
                for (int n = tid; n < H; n += THREADS) a.wide[n] = (int)s.x[n] + (column(s, M + p.w_o + l * hh, H, H, n) >> p.shift_out);
                residual();
                norm(p.ln_2 + l * (uint32_t)H, p.ln_2_bias + l * (uint32_t)H);
            } else
                norm(p.ln_init, p.ln_init_bias);
            const int8_t *up = M + (l < 0 ? p.w_up_init : p.w_up + 4 * l * hh), *b_up = M + (l < 0 ? p.b_up_init : p.b_up + l * (size_t)(4 * H));
            const int8_t *dn = M + (l < 0 ? p.w_dn_init : p.w_dn + 4 * l * hh), *b_dn = M + (l < 0 ? p.b_dn_init : p.b_dn + l * (size_t)H);
            int g[4 * NE];
#pragma unroll
            for (int i = 0; i < 4 * NE; i++) {
                const int n = tid + 256 * i;
                g[i] = n < 4 * H ? s.act[(uint8_t)clip127((column(s, up, H, 4 * H, n) >> p.shift_up) + b_up[n])] : 0;
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 4 * NE; i++) { const int n = tid + 256 * i; if (n < 4 * H) s.op[byte_of(n)] = (int8_t)g[i]; }
            __syncthreads();
            for (int n = tid; n < H; n += THREADS) a.wide[n] = (int)s.x[n] + (column(s, dn, 4 * H, H, n) >> p.shift_dn) + b_dn[n];
            residual();
        }
        norm(p.ln_f, p.ln_f_bias);
        int mx = INT_MIN;
        for (int v = tid; v < V; v += THREADS) {
            int lg = column(s, M + p.embedding, H, V, v) >> p.shift_logit;
            if (p.deggs && p.penalty_int) {
                uint32_t count = 0;
                for (int i = 0; i <= t; i++) count += s.tok[i] == v;
                lg = (int)((uint32_t)lg - count * (uint32_t)p.penalty_int);
            }
            p.logits[v] = lg;
            mx = max(mx, lg);
        }
        mx = wg_reduce<true>(mx, s.redm);
        // the order of the reference's H threads: thread r owns v = r, r + H, ... (see sample)
        for (int r = tid; r < H; r += THREADS) {
            long long sum = 0;
            for (int v = r; v < V; v += H) sum += exp_of(s, p, p.logits[v], mx);
            a.tsum[r] = sum;
        }
        __syncthreads();
        if (tid == 0) {
            long long total = 0, running = 0;
            for (int r = 0; r < H; r++) total += a.tsum[r];
            const long long thresh = total > 0 ? (long long)hash_rng(p.seed + (uint32_t)t * 555u, 0) % total : 0;
            int r = 0, sel = 0;
            while (r < H && running + a.tsum[r] <= thresh) running += a.tsum[r++];
            for (int v = r; r < H && v < V; v += H) {
                running += exp_of(s, p, p.logits[v], mx);
                if (running > thresh) { sel = v; break; }
            }
            s.tok[t + 1] = sel;
            if (p.token_bytes == 4) reinterpret_cast<uint32_t *>(p.out)[t + 1] = (uint32_t)sel;
            else reinterpret_cast<uint8_t *>(p.out)[t + 1] = (uint8_t)sel;
        }
        __syncthreads();
    }
    for (int64_t i = tid; i < egg_decode_slots(H); i += THREADS) p.slots[i] = 0;
    if (tid == 0) { *p.epoch = 0; *p.fail = 0; }
}

// the logits that the workgroup with the most head tiles keeps
int logit_bytes(int H, int vocab) { return (vocab / 16 + H / 16 - 1) / (H / 16) * 16 * (int)sizeof(int); }
template <int H>
hipError_t launch(const DecodeParams &p, hipStream_t s) {
    hipLaunchKernelGGL(k_decode<H>, dim3(H / 16), dim3(THREADS), logit_bytes(H, p.vocab), s, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_decode_alone<H>, dim3(1), dim3(THREADS), 0, s, p);
    return hipGetLastError();
}

}  // namespace

hipError_t egg_prepare_decode(int H, int vocab) {
    const int bytes = logit_bytes(H, vocab);
    if (bytes + (int)sizeof(Lds) <= 64 * 1024) return hipSuccess;
    const void *f = H == 64 ? (const void *)k_decode<64> : H == 128 ? (const void *)k_decode<128> : H == 256 ? (const void *)k_decode<256> : (const void *)k_decode<512>;
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}
hipError_t egg_launch_decode(const DecodeParams &p, int H, hipStream_t s) {
    if (p.count < 1 || p.t_first < 0 || p.t_first + p.count > p.T - 1 || p.T > 512 || p.vocab % 256 || !(p.head_dim == 32 || p.head_dim == 64)) return hipErrorInvalidValue;
    switch (H) {
    case 64: return launch<64>(p, s);
    case 128: return launch<128>(p, s);
    case 256: return launch<256>(p, s);
    case 512: return launch<512>(p, s);
    }
    return hipErrorInvalidValue;
}
