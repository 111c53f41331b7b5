// egg_votes.hip -- vote reconstruction and the optimizer step of every tensor of the model on gfx950.
//
// Reference: apply_adam_update, update_matrix_adam_kernel, update_vector_adam_kernel (mgpu.cu:1040-1152), the Muon
// momentum, gather and apply kernels (muon_internal.cuh:15-74, :112-170).
//
// The reference draws two noise values per (weight, pair).  Which value a tensor draws for pair p and row or column i is
// hash_rng(seed + p + seed_base + off, i): tensors differ in a shift of the pair index only.  So ONE table
//     N[i][t] = noise_from_hash(seed + t, i)
// holds every tensor's noise, a tensor's row i being N[i][seed_base + off ...].  It has 4 hidden rows of pairs + 1000 layers
// entries and, for the columns of the embedding, vocab - 4 hidden more rows of pairs entries -- 25 million hashes at hidden 256, 4 layers, 20,480 pairs, where panels of one tensor
// after the other were 440 million -- and the vote matrices  sum_p fit_p A_p[n] B_p[k]  of all tensors are int8 matrix
// products over shifted windows of it.
#include "egg_device.h"
#include "egg_launch.h"
#include <type_traits>

#pragma clang fp contract(off)

// ---------------------------------------------------------------- noise table
// Thread: 16 consecutive entries of one row, one 16-byte store.  Bound by the hash (about 15 vector instructions an entry);
// entries no tensor reads are left out: rows past `layer_rows` belong to the embedding alone (and share the space of one:
// 28 MB instead of 0.5 GB at vocabulary 65,536, hidden 64, 8 layers), and between the layers' windows there are gaps
// while there are fewer pairs than a layer's 1000 seeds.
// The first workgroups turn the fitness into byte masks and clear the update counter (when it is to be cleared).  In a whole
// step (end.acc) they do what stands between the forward and the update as well, four pairs a thread: losses and
// fitness, in device memory and in the host's copy, and the loss sums set back to zero: three launches less, and no copies
// when the host asks (a step of hidden 64, 2 layers, 64 members with its results read: 207 -> 146 us).
typedef int int_any __attribute__((aligned(1)));
__device__ __forceinline__ int8_t *noise_row(const NoiseTable &nt, int r) {
    if (r < nt.layer_rows) return nt.table + (size_t)r * nt.ld;
    const unsigned at = (unsigned)(r - nt.layer_rows), slot = at / (unsigned)nt.emb_rows;
    return nt.table + (size_t)(r - (int)slot * nt.emb_rows) * nt.ld + slot * nt.emb_ld;
}
__device__ __forceinline__ void store_masks(const NoiseTable &nt, int pair, int neg, int nz) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const size_t at = k * nt.mask_ld + EGG_NOISE_FRONT + k + pair;
        *reinterpret_cast<int_any *>(nt.neg + at) = neg;
        *reinterpret_cast<int_any *>(nt.nonzero + at) = nz;
    }
}
__device__ __forceinline__ void masks_of_fitness(const NoiseTable &nt, const int32_t *fit, int pairs) {
    __shared__ int other;
    if (threadIdx.x == 0) other = 0;
    __syncthreads();
    for (int c = threadIdx.x; c < nt.pairs_pad / 16; c += 256) {
        int odd = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            int n4 = 0, z4 = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int pr = 16 * c + 4 * q + e, f = pr < pairs ? fit[pr] : 0;
                n4 |= (f == -1 ? 0xff : 0) << (8 * e);
                z4 |= (f != 0 ? 0xff : 0) << (8 * e);
                odd |= f < -1 || f > 1;
            }
            store_masks(nt, 16 * c + 4 * q, n4, z4);
        }
        if (odd) other = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) *nt.general = other;
}
__device__ __forceinline__ void end_of_step(const NoiseTable &nt, const StepEnd &end, int pairs) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c == 0) *nt.general = 0;
    if (c >= nt.pairs_pad / 4) return;
    int n4 = 0, z4 = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int pr = 4 * c + e;
        if (pr >= pairs) continue;
        unsigned long long *acc = end.acc + 2 * pr;
        const int2 l = {(int)(long long)acc[0], (int)(long long)acc[1]};           // mgpu.cu:1028
        const int f = l.x < l.y ? 1 : l.y < l.x ? -1 : 0;                         // mgpu.cu:1031-1036
        acc[0] = acc[1] = 0ull;
        reinterpret_cast<int2 *>(end.loss)[pr] = l; reinterpret_cast<int2 *>(end.h_loss)[pr] = l;
        end.fit[pr] = f; end.h_fit[pr] = f;
        n4 |= (f == -1 ? 0xff : 0) << (8 * e);
        z4 |= (f != 0 ? 0xff : 0) << (8 * e);
    }
    store_masks(nt, 4 * c, n4, z4);
}
__global__ void __launch_bounds__(256) k_noise_table(NoiseTable nt, const uint32_t *d_seed, const int32_t *fit, StepEnd end, int first, int pairs,
                                                     int mask, int rows, int t_lo, int t_hi, int n_layers, unsigned long long *counter) {
    if ((int)blockIdx.x < first) {
        if (blockIdx.x == 0 && threadIdx.x == 0 && counter) *counter = 0ull;
        if (end.acc) end_of_step(nt, end, pairs); else masks_of_fitness(nt, fit, pairs);
        return;
    }
    const int per_row = (t_hi - t_lo + 15) / 16;
    const int64_t i = (int64_t)((int)blockIdx.x - first) * 256 + threadIdx.x;
    const int r = (int)(i / per_row), t0 = t_lo + 16 * (int)(i % per_row);
    if (r >= rows || (r >= nt.layer_rows && t0 >= nt.emb_t)) return;
    if (pairs < 512) {
        const int l = min(t0 / 1000, n_layers - 1), rel = t0 - 1000 * l;
        if (rel >= (l ? EGG_LAYER_SEEDS : EGG_MODEL_SEEDS) + nt.pairs_pad + 16) return;
    }
    const uint32_t s = *d_seed + (uint32_t)t0;
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = noise_from_hash(s + (uint32_t)(4 * q + e), (uint32_t)r, mask);
        o[q] = pack4(v[0], v[1], v[2], v[3]);
    }
    *reinterpret_cast<v4i *>(noise_row(nt, r) + EGG_NOISE_FRONT + t0) = o;
}
// the last window ends with the entries; it is read in whole chunks of 128 from 15 bytes in front of it on
size_t egg_noise_ld(int entries) { return ((size_t)EGG_NOISE_FRONT + entries + 128 + 32 + 127) / 128 * 128; }
size_t egg_noise_mask_ld(int pairs_pad) { return (size_t)EGG_NOISE_FRONT + pairs_pad + 128 + 16; }
hipError_t egg_launch_noise_table(const NoiseTable &nt, const uint32_t *d_seed, const int32_t *d_fit, const StepEnd &end, int pairs, int mask, int rows,
                                  int t_lo, int t_hi, int n_layers, unsigned long long *counter, hipStream_t s) {
    t_lo &= ~15;
    t_hi = (t_hi + 15) & ~15;
    if (rows < 1 || rows > nt.rows || t_lo < 0 || (size_t)t_hi + EGG_NOISE_FRONT > nt.ld || (size_t)nt.emb_t + 16 + EGG_NOISE_FRONT > nt.emb_ld)
        return hipErrorInvalidValue;
    const int64_t items = (int64_t)rows * ((t_hi - t_lo) / 16);
    const int first = end.acc ? (nt.pairs_pad / 4 + 255) / 256 : 1;
    hipLaunchKernelGGL(k_noise_table, dim3((unsigned)((items + 255) / 256 + first)), dim3(256), 0, s, nt, d_seed, d_fit, end, first, pairs, mask, rows,
                       t_lo, t_hi, n_layers, counter);
    return hipGetLastError();
}

// ---------------------------------------------------------------- optimizer rules
// apply_adam_update (mgpu.cu:1040-1064); every float operation is a single IEEE-754 operation
struct AdamHyper { float b1, b2, eps, wd; int limit; };     // limit: the weight saturates at +-limit (127 in the reference)
// the accumulator's thresholds: returns whether the weight moved
__device__ __forceinline__ int threshold_apply(float &acc, int &w, int limit) {
    int change = 0;
    if (acc >= 1.0f) {
        if (w < limit) { w++; change = 1; acc -= 1.0f; } else acc = 1.0f;
    } else if (acc <= -1.0f) {
        if (w > -limit) { w--; change = 1; acc += 1.0f; } else acc = -1.0f;
    }
    return change;
}
__device__ __forceinline__ int adam_apply(float &m, float &v, float &acc, int &w, float gr, float lr, const AdamHyper &h) {
    float t1 = h.b1 * m; float t2 = (1.0f - h.b1) * gr; m = t1 + t2;
    float t3 = h.b2 * v; float gg = gr * gr; float t4 = (1.0f - h.b2) * gg; v = t3 + t4;
    float den = sqrtf(v) + h.eps;
    float q = m / den;
    float wdw = h.wd * (float)w;
    float step = (-lr) * (q + wdw);
    acc += step;
    return threshold_apply(acc, w, h.limit);
}

// Number of changed weights of a workgroup (`mine`: of this wave, in its lane 0), added to the counter.  While an update runs,
// the counter's upper 24 bits count the workgroups that have reported; the last of p.count_of leaves the number alone in it
// and writes it to the host's copy, so that a caller who asks for it needs no copy of its own.
__device__ __forceinline__ void count_changes(const UpdLaunch &p, int mine, int *sums) {
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x) return;
    unsigned long long n = 1ull << 40;
    for (int w = 0; w < EGG_WAVES; w++) n += (unsigned long long)sums[w];
    n += atomicAdd(p.counter, n);
    if (n >> 40 != (unsigned long long)p.count_of) return;
    n &= (1ull << 40) - 1;
    *p.counter = n;
    *p.h_counter = n;
}

// index of the last of n ascending entries first(i) that is <= at (first(0) <= at), found by all lanes of a wave together
template <typename F>
__device__ __forceinline__ int find_last(int n, int at, F first) {
    const int lane = threadIdx.x & 63;
    int d = 0;
    for (int base = 0; base < n; base += 64) {
        const unsigned long long m = __ballot(base + lane < n && first(base + lane) <= at);
        if (!m) break;
        d = base + 63 - __builtin_clzll(m);
    }
    return __builtin_amdgcn_readfirstlane(d);
}
// Where the 16 bytes (k = 32 ks + 8q + 4g + e, q and e ascending; column n) of a matrix lie in its fragment-major copy
// (egg_device.h): what a lane of the MFMA result layout holds is exactly one such unit.
__device__ __forceinline__ v4i *frag_unit(const MatDesc &t, int ks, int g, int n) {
    const int bk = t.block / 32, kb = ks / bk, nb = n / t.block;
    return reinterpret_cast<v4i *>(t.frag + ((size_t)kb * (t.cols / t.block) + nb) * t.block * t.block +
                                   ((size_t)(2 * (ks % bk) + g) * t.block + n % t.block) * 16);
}

// Two windows of the table side by side, positions counted from the last 16-byte boundary in front of the first: the first
// is read in aligned pieces (the pair of position i is i - shift), the other one dword-aligned and moved by the rest of
// its offset in registers, the masks from the copy that has them on a dword.  A 16-byte load at any byte takes the memory
// pipe four times as long as an aligned one, and six of them a chunk were what the kernel below spent its time on.
struct Windows {
    size_t a, b; int shift, rest; const int8_t *neg, *nz;
    __device__ __forceinline__ Windows(const NoiseTable &nt, int t_a, int t_b) {
        shift = t_a & 15;
        a = EGG_NOISE_FRONT + (t_a & ~15);
        const int at = EGG_NOISE_FRONT + t_b - shift;
        b = at & ~3; rest = at & 3;
        const size_t m = (shift & 3) * nt.mask_ld + EGG_NOISE_FRONT - (shift & ~3);
        neg = nt.neg + m; nz = nt.nonzero + m;
    }
    __device__ __forceinline__ int length(int pairs) const { return shift + pairs; }
};
typedef int v4i_dword __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ v4i load_dwords(const int8_t *p) { return *reinterpret_cast<const v4i_dword *>(p); }
__device__ __forceinline__ v4i moved(v4i x, int next, int rest) {
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; q++) o[q] = (int)__builtin_amdgcn_alignbyte((unsigned)(q < 3 ? x[q + 1] : next), (unsigned)x[q], (unsigned)rest);
    return o;
}
// The noise of 16 pairs times their fitness.  Fitness in {-1, 0, 1}: (x ^ neg) & nonzero is x, 0, or -x - 1; the caller adds
// the missing sum of the other factor over the negative pairs.
__device__ __forceinline__ v4i signed_noise(v4i x, v4i neg, v4i nz) {
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; q++) o[q] = (x[q] ^ neg[q]) & nz[q];
    return o;
}
__device__ __forceinline__ int sum_negative(v4i x, v4i neg, int c) {
#pragma unroll
    for (int q = 0; q < 4; q++) c = dot4(x[q], neg[q] & 0x01010101, c);
    return c;
}
// any other fitness: byte products, wrapped to 8 bits
__device__ __forceinline__ v4i scaled_noise(v4i x, const int32_t *fit, int first, int pairs) {
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) { const int pr = first + 4 * q + e; v[e] = pr >= 0 && pr < pairs ? fit[pr] * sx8(x[q], e) : 0; }
        o[q] = pack4(v[0], v[1], v[2], v[3]);
    }
    return o;
}

// update_vector_adam_kernel (mgpu.cu:1114-1152): VEC consecutive elements a wave (tensors have multiples of 64), 16 pairs a
// lane, all elements' rows in flight together; lane i applies the rule to element i.  One element a wave was 98 us of the
// update of hidden 512, 8 layers at 256 pairs, 10 thousand workgroups of descriptor look-ups and load latency; four take
// a quarter of it.
// Returns the number of changed weights, in lane 0.
constexpr int VEC = 4;
__device__ __forceinline__ int vector_elements(const UpdLaunch &p, int gi) {
    const int lane = threadIdx.x & 63;
    const int d = find_last(p.n_vec, gi, [&](int i) { return p.vec[i].first; });
    const VecDesc t = p.vec[d];
    const int idx = gi - t.first;
    const int8_t *row = p.noise.table + (size_t)idx * p.noise.ld;          // vector tensors have at most layer_rows elements
    float *const st = t.state + (size_t)(idx + lane) * 3;
    float m = 0.f, v = 0.f, acc = 0.f;
    int w = 0;
    if (lane < VEC) { m = st[0]; v = st[1]; acc = st[2]; w = t.W[idx + lane]; }
    int vote[VEC];
#pragma unroll
    for (int i = 0; i < VEC; i++) vote[i] = 0;
    if (!*p.noise.general) {
        const Windows at(p.noise, t.seed_base + t.off_a, t.seed_base + t.off_b);
        const int n = at.length(p.pairs);
        for (int s = 16 * lane; s < n; s += 1024) {
            const v4i neg = load_dwords(at.neg + s), nz = load_dwords(at.nz + s);
            v4i a[VEC], b[VEC];
            int more[VEC];
#pragma unroll
            for (int i = 0; i < VEC; i++) {
                a[i] = *reinterpret_cast<const v4i *>(row + i * p.noise.ld + at.a + s);
                b[i] = load_dwords(row + i * p.noise.ld + at.b + s);
                more[i] = *reinterpret_cast<const int *>(row + i * p.noise.ld + at.b + s + 16);
            }
#pragma unroll
            for (int i = 0; i < VEC; i++) {
                const v4i x = signed_noise(a[i], neg, nz), y = moved(b[i], more[i], at.rest);
#pragma unroll
                for (int q = 0; q < 4; q++) vote[i] = dot4(x[q], y[q], vote[i]);
                vote[i] = sum_negative(y, neg, vote[i]);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < VEC; i++) {
            const int8_t *ra = row + i * p.noise.ld + EGG_NOISE_FRONT + t.seed_base + t.off_a, *rb = row + i * p.noise.ld + EGG_NOISE_FRONT + t.seed_base + t.off_b;
            for (int pr = lane; pr < p.pairs; pr += 64) vote[i] += p.fit[pr] * ra[pr] * rb[pr];
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int i = 0; i < VEC; i++) vote[i] += __shfl_xor(vote[i], off, 64);
    int mine = vote[0];
#pragma unroll
    for (int i = 1; i < VEC; i++) mine = lane == i ? vote[i] : mine;
    int ch = 0;
    if (lane < VEC) {
        const AdamHyper hy = {p.beta1, p.beta2, p.eps, p.wd, 127};     // vector tensors keep the reference's +-127
        ch = adam_apply(m, v, acc, w, -(float)mine, (*p.d_lr) * t.lr_scale, hy);
        t.W[idx + lane] = (int8_t)w; st[0] = m; st[1] = v; st[2] = acc;
        if (ch && t.flags) t.flags[idx + lane] = 1;
    }
    return __popcll(__ballot(ch != 0));
}

// A 32 (k) x 32 (n) piece of a matrix's weights and optimizer state in the MFMA result layout: accumulator register 4q + e of
// lane (n, g) -> k = kt + 8q + 4g + e; blocked index of (k, n) (mgpu.cu:1085-1089).  Read as a whole ahead of its use: left to
// themselves the reads of each q wait for the stores of the one in front.
struct Piece {
    int w[4]; float4 s[4][3];
    __device__ __forceinline__ void read(const UpdLaunch &p, const MatDesc &t, int kt, int n, int g) {
        if (p.votes_out) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const size_t idx = ((size_t)((kt >> 2) + 2 * q + g) * t.cols + n) * 4;
            const float4 *sp = reinterpret_cast<const float4 *>(t.state + idx * (t.muon_x ? 2 : 3));
            s[q][0] = sp[0]; s[q][1] = sp[1];
            if (!t.muon_x) { s[q][2] = sp[2]; w[q] = *reinterpret_cast<const int *>(t.W + idx); }
        }
    }
    // returns the number of changed weights
    __device__ __forceinline__ int apply(const UpdLaunch &p, const MatDesc &t, int kt, int n, int g, const v16i &vote, float lr, const AdamHyper &hy) const {
        int changes = 0;
        v4i unit;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const size_t idx = ((size_t)((kt >> 2) + 2 * q + g) * t.cols + n) * 4;
            if (p.votes_out) {
                v4i o4;
#pragma unroll
                for (int e = 0; e < 4; e++) o4[e] = vote[4 * q + e];
                *reinterpret_cast<v4i *>(p.votes_out + idx) = o4;
                continue;
            }
            const float4 s0 = s[q][0], s1 = s[q][1], s2 = s[q][2];
            if (t.muon_x) {
                // muon_momentum_update_kernel + muon_gather_m_kernel (muon_internal.cuh:15-74): m = mu*m + vote
                float mv[4] = {s0.x, s0.z, s1.x, s1.z};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float m = p.muon_momentum * mv[e];
                    mv[e] = m + (float)vote[4 * q + e];
                    t.muon_x[(size_t)(kt + 8 * q + 4 * g + e) * t.cols + n] = mv[e];
                }
                float4 *sp = reinterpret_cast<float4 *>(t.state + idx * 2);
                sp[0] = make_float4(mv[0], s0.y, mv[1], s0.w);
                sp[1] = make_float4(mv[2], s1.y, mv[3], s1.w);
                continue;
            }
            float st[12] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w, s2.x, s2.y, s2.z, s2.w};
            int wv[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                wv[e] = sx8(w[q], e);
                const int ch = adam_apply(st[3 * e], st[3 * e + 1], st[3 * e + 2], wv[e], -(float)vote[4 * q + e], lr, hy);
                changes += ch;
                // overlay flags (de/include/optimizer/adam.cuh:77-83): every writer stores the same value, so plain stores do
                if (ch && p.flags) { p.flags[t.offset + kt + 8 * q + 4 * g + e] = 1; p.flags[t.offset + t.rows + n] = 1; }
            }
            unit[q] = pack4(wv[0], wv[1], wv[2], wv[3]);
            *reinterpret_cast<int *>(t.W + idx) = unit[q];
            float4 *sp = reinterpret_cast<float4 *>(t.state + idx * 3);
            sp[0] = make_float4(st[0], st[1], st[2], st[3]);
            sp[1] = make_float4(st[4], st[5], st[6], st[7]);
            sp[2] = make_float4(st[8], st[9], st[10], st[11]);
        }
        if (!p.votes_out && !t.muon_x) *frag_unit(t, kt >> 5, g, n) = unit;
        return changes;
    }
};

// Votes and optimizer step of every matrix of a list (and of every vector tensor, in the workgroups behind the matrix
// tiles).  One workgroup per 64 WT (k) x 64 WT (n) tile of a vote matrix, whatever the matrix: all tiles of the model in one
// launch.  The pairs go by in chunks of 128: every thread fetches 16 pairs of 2 WT k rows and 2 WT n rows (a row's 128 bytes
// by eight neighbouring lanes, see Windows), applies the fitness to the n rows and stores them into LDS in MFMA operand order.
// The next chunk's loads are in flight meanwhile; two LDS buffers, one barrier a chunk.  A chunk column (16 pairs of all
// rows) is 32 bytes longer than its rows, so that the eight lanes of a row store to different banks.
// WT = 1: wave w multiplies the chunk's 32-pair step w, two by two fragments of 32 rows; the four partial tiles are added up
// in two exchanges (half a tile each, then a quarter), after which wave w owns the 32 x 32 quarter (w >> 1, w & 1).
// WT = 2: wave w multiplies the whole chunk for its 64 x 64 quarter: a quarter of the loads per weight, and nothing to add
// up, but 66 KB of LDS and a quarter of the workgroups.
// The owner of a piece applies the optimizer rule and writes the weights' fragment-major copy.
// Bound by the state's 24 bytes a weight at few pairs, and by the latency of a chunk's chain (loads, LDS, MFMAs) at many.
// Hidden 512, 8 layers (AdamW), 256 pairs: 0.33 -> 0.22 ms with the table's 0.01, 8,192 pairs: 1.0 -> 0.66 ms; hidden 256, 4
// layers, 20,480 pairs: 0.38 -> 0.26 ms; hidden 128, 8 layers, 512 pairs: 50 -> 30 us.
template <int WT>
__global__ void __launch_bounds__(EGG_THREADS, WT == 1 ? 3 : 2) k_update(UpdLaunch p) {
    constexpr int ROWS = 64 * WT, COL = ROWS * 16 + 32, OPERAND = 8 * COL, PARTS = 2 * WT;
    __shared__ __align__(16) int8_t lds[4 * OPERAND];
    __shared__ int corr[ROWS];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 5, j = lane & 31;
    const int tiles = p.tiles / (WT * WT);
    if ((int)blockIdx.x >= tiles) {
        const int gi = (((int)blockIdx.x - tiles) * EGG_WAVES + wave) * VEC;
        count_changes(p, gi < p.vec_total ? vector_elements(p, gi) : 0, corr);
        return;
    }
    const MatDesc t = p.mat[find_last(p.n_mat, blockIdx.x, [&](int i) { return p.mat[i].tile_first / (WT * WT); })];
    const int tiles_n = t.cols / ROWS, tile = blockIdx.x - t.tile_first / (WT * WT);
    const int k0 = (tile / tiles_n) * ROWS, n0 = (tile % tiles_n) * ROWS;
    const int c = threadIdx.x & 7, r = threadIdx.x >> 3;
    const Windows w(p.noise, t.t_a, t.t_b);
    const size_t down = 32 * p.noise.ld;                     // a tile's rows lie ld apart wherever they start (see NoiseTable)
    const int8_t *pa = noise_row(p.noise, n0) + (size_t)r * p.noise.ld + w.a + 16 * c;
    const int8_t *pb = p.noise.table + (size_t)(k0 + r) * p.noise.ld + w.b + 16 * c;
    const int general = *p.noise.general, length = w.length(p.pairs);
    v4i a[PARTS], b[PARTS], neg, nz;
    int more[PARTS];
    auto fetch = [&](int s) {
#pragma unroll
        for (int i = 0; i < PARTS; i++) {
            a[i] = *reinterpret_cast<const v4i *>(pa + i * down + s);
            b[i] = load_dwords(pb + i * down + s);
            more[i] = *reinterpret_cast<const int *>(pb + i * down + s + 16);
        }
        neg = load_dwords(w.neg + s + 16 * c);
        nz = load_dwords(w.nz + s + 16 * c);
    };
    v16i acc[2][2];
    zero_acc<2>(acc[0]); zero_acc<2>(acc[1]);
    int negative[PARTS], buf = 0;
#pragma unroll
    for (int i = 0; i < PARTS; i++) negative[i] = 0;
    fetch(0);
    // (two loops: with the general form beside it, the ternary one's few instructions lie scattered over kilobytes of code and
    // carry the other's addresses along)
    auto chunks = [&](auto any) {
        for (int s = 0; s < length; s += 128) {
            int8_t *A = lds + buf * 2 * OPERAND + c * COL + r * 16, *B = A + OPERAND;
#pragma unroll
            for (int i = 0; i < PARTS; i++) {
                const v4i bm = moved(b[i], more[i], w.rest);
                v4i am;
                if constexpr (any) am = scaled_noise(a[i], p.fit, s + 16 * c - w.shift, p.pairs);
                else { am = signed_noise(a[i], neg, nz); negative[i] = sum_negative(bm, neg, negative[i]); }
                *reinterpret_cast<v4i *>(A + i * 512) = am;
                *reinterpret_cast<v4i *>(B + i * 512) = bm;
            }
            if (s + 128 < length) fetch(s + 128);
            __syncthreads();
            const int ra = WT == 1 ? 0 : (wave & 1) * 64, rb = WT == 1 ? 0 : (wave >> 1) * 64, first = (WT == 1 ? 2 * wave + g : g) * COL;
            const int8_t *fA = lds + buf * 2 * OPERAND + first + (ra + j) * 16, *fB = lds + (buf * 2 + 1) * OPERAND + first + (rb + j) * 16;
            constexpr int STEPS = WT == 1 ? 1 : 4;
            v4i fa[2][2], fb[2][2];                        // the next step's fragments are read ahead of this one's products
            auto frags = [&](int step) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    fa[step & 1][h] = *reinterpret_cast<const v4i *>(fA + 2 * step * COL + 32 * h * 16);
                    fb[step & 1][h] = *reinterpret_cast<const v4i *>(fB + 2 * step * COL + 32 * h * 16);
                }
            };
            frags(0);
#pragma unroll
            for (int step = 0; step < STEPS; step++) {
                if (step + 1 < STEPS) frags(step + 1);
#pragma unroll
                for (int hk = 0; hk < 2; hk++)
#pragma unroll
                    for (int hn = 0; hn < 2; hn++)
                        acc[hk][hn] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[step & 1][hk], fa[step & 1][hn], acc[hk][hn], 0, 0, 0);
            }
            buf ^= 1;
        }
    };
    if (general) chunks(std::true_type()); else chunks(std::false_type());
    // sums over the negative pairs of the k rows, over the eight chunk columns
#pragma unroll
    for (int i = 0; i < PARTS; i++) {
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) negative[i] += __shfl_xor(negative[i], o, 64);
        if (c == 0) corr[r + 32 * i] = negative[i];
    }
    __syncthreads();
    const float lr = p.d_lr ? (*p.d_lr) * t.lr_scale : 0.f;
    const AdamHyper hy = {p.beta1, p.beta2, p.eps, p.wd, t.limit};
    int changes = 0;
    if constexpr (WT == 1) {
        Piece own;
        own.read(p, t, k0 + 32 * (wave >> 1), n0 + 32 * (wave & 1) + j, g);
        int *red = reinterpret_cast<int *>(lds);             // [wave][2 tiles][16][64], then [wave][16][64]
        const bool hi = wave >= 2, odd = wave & 1;
        v16i mine[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                red[((wave * 2 + h) * 16 + e) * 64 + lane] = hi ? acc[0][h][e] : acc[1][h][e];
                mine[h][e] = hi ? acc[1][h][e] : acc[0][h][e];
            }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 16; e++) mine[h][e] += red[(((wave ^ 2) * 2 + h) * 16 + e) * 64 + lane];
        __syncthreads();
        v16i vote;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            red[(wave * 16 + e) * 64 + lane] = odd ? mine[0][e] : mine[1][e];
            vote[e] = odd ? mine[1][e] : mine[0][e];
        }
        __syncthreads();
        const int kt = 32 * (wave >> 1);
#pragma unroll
        for (int e = 0; e < 16; e++) vote[e] += red[((wave ^ 1) * 16 + e) * 64 + lane] + corr[kt + 8 * (e >> 2) + 4 * g + (e & 3)];
        changes = own.apply(p, t, k0 + kt, n0 + 32 * (wave & 1) + j, g, vote, lr, hy);
    } else {
        const int kw = k0 + 64 * (wave >> 1), nw = n0 + 64 * (wave & 1) + j;
        Piece at[2];
        at[0].read(p, t, kw, nw, g);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (i < 3) at[(i + 1) & 1].read(p, t, kw + 32 * ((i + 1) >> 1), nw + 32 * ((i + 1) & 1), g);
            v16i vote = acc[i >> 1][i & 1];
#pragma unroll
            for (int e = 0; e < 16; e++) vote[e] += corr[64 * (wave >> 1) + 32 * (i >> 1) + 8 * (e >> 2) + 4 * g + (e & 3)];
            changes += at[i & 1].apply(p, t, kw + 32 * (i >> 1), nw + 32 * (i & 1), g, vote, lr, hy);
        }
    }
    if (p.votes_out || t.muon_x) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) changes += __shfl_xor(changes, off, 64);
    __syncthreads();                                         // the corrections have been read
    count_changes(p, changes, corr);
}
// 128 x 128 tiles where they occupy five eighths of the 256 CUs: at 200 tiles they take 0.26 ms for 20,480 pairs (64 x 64:
// 0.34), at 110 or fewer the chip is too empty (45 us against 30 for 512 pairs, 74 against 42 for 4,096)
static bool wide_tiles(const UpdLaunch &p) { return p.wide && p.tiles / 4 >= 160; }
int egg_update_blocks(const UpdLaunch &p) { return (wide_tiles(p) ? p.tiles / 4 : p.tiles) + (p.vec_total + EGG_WAVES * VEC - 1) / (EGG_WAVES * VEC); }
hipError_t egg_launch_update(const UpdLaunch &p, hipStream_t s) {
    const int blocks = egg_update_blocks(p);
    if (blocks < 1) return hipSuccess;
    if (p.noise.pairs_pad % 128 || p.noise.layer_rows % 128 || p.noise.emb_rows % 128 || p.vec_total % VEC || (p.tiles && p.n_mat < 1) || (p.vec_total && p.n_vec < 1)) return hipErrorInvalidValue;
    if (wide_tiles(p)) hipLaunchKernelGGL(k_update<2>, dim3(blocks), dim3(EGG_THREADS), 0, s, p);
    else hipLaunchKernelGGL(k_update<1>, dim3(blocks), dim3(EGG_THREADS), 0, s, p);
    return hipGetLastError();
}

// muon_apply_update_kernel (muon_internal.cuh:112-170) for every matrix of a list: a thread takes one 16-byte unit of the
// fragment-major copy (16 rows of one column), so neighbouring lanes read and write neighbouring columns throughout.
// Bound by memory (22 bytes an element).
__global__ void __launch_bounds__(256) k_muon_apply(UpdLaunch p, float wd, const float *ortho) {
    __shared__ int sums[EGG_WAVES];
    const MatDesc t = p.mat[find_last(p.n_mat, blockIdx.x, [&](int i) { return p.mat[i].tile_first; })];
    const int u = ((int)blockIdx.x - t.tile_first) * 256 + (int)threadIdx.x;       // 256 units to a 64 x 64 tile
    const int n = u % t.cols, kk = u / t.cols, ks = kk >> 1, g = kk & 1;
    const float lr = (*p.d_lr) * t.lr_scale;
    int changes = 0;
    v4i unit;
    // (all reads first: each would otherwise wait for the stores in front of it)
    int w4[4];
    float4 s0[4], s1[4];
    float x[4][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int kr = 32 * ks + 8 * q + 4 * g;
        const size_t idx = ((size_t)(kr >> 2) * t.cols + n) * 4;
        const float4 *sp = reinterpret_cast<const float4 *>(t.state + idx * 2);
        w4[q] = *reinterpret_cast<const int *>(t.W + idx);
        s0[q] = sp[0]; s1[q] = sp[1];
#pragma unroll
        for (int e = 0; e < 4; e++) x[q][e] = ortho[t.muon_at + (size_t)(kr + e) * t.cols + n];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const size_t idx = ((size_t)((32 * ks + 8 * q + 4 * g) >> 2) * t.cols + n) * 4;
        float acc[4] = {s0[q].y, s0[q].w, s1[q].y, s1[q].w};
        int wv[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            wv[e] = sx8(w4[q], e);
            const float wdw = wd * (float)wv[e];
            const float step = (-lr) * (x[q][e] + wdw);
            acc[e] += step;
            changes += threshold_apply(acc[e], wv[e], t.limit);
        }
        unit[q] = pack4(wv[0], wv[1], wv[2], wv[3]);
        *reinterpret_cast<int *>(t.W + idx) = unit[q];
        float4 *sp = reinterpret_cast<float4 *>(t.state + idx * 2);
        sp[0] = make_float4(s0[q].x, acc[0], s0[q].z, acc[1]);
        sp[1] = make_float4(s1[q].x, acc[2], s1[q].z, acc[3]);
    }
    *frag_unit(t, ks, g, n) = unit;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) changes += __shfl_xor(changes, off, 64);
    count_changes(p, changes, sums);
}
hipError_t egg_launch_muon_apply(const UpdLaunch &p, float wd, const float *x, hipStream_t s) {
    if (p.tiles < 1 || !x) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_muon_apply, dim3(p.tiles), dim3(256), 0, s, p, wd, x);
    return hipGetLastError();
}

// the fragment-major copies of every matrix of a list from its canonical blocked weights
__global__ void __launch_bounds__(256) k_frag(const MatDesc *mat, int n_mat) {
    const MatDesc t = mat[find_last(n_mat, blockIdx.x, [&](int i) { return mat[i].tile_first; })];
    const int u = ((int)blockIdx.x - t.tile_first) * 256 + (int)threadIdx.x;
    const int n = u % t.cols, kk = u / t.cols, ks = kk >> 1, g = kk & 1;
    v4i unit;
#pragma unroll
    for (int q = 0; q < 4; q++) unit[q] = *reinterpret_cast<const int *>(t.W + ((size_t)(8 * ks + 2 * q + g) * t.cols + n) * 4);
    *frag_unit(t, ks, g, n) = unit;
}
hipError_t egg_launch_frag(const MatDesc *d_mat, int n_mat, int tiles, hipStream_t s) {
    if (n_mat < 1 || tiles < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_frag, dim3(tiles), dim3(256), 0, s, d_mat, n_mat);
    return hipGetLastError();
}
