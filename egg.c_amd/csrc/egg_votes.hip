// egg_votes.hip -- vote reconstruction and the optimizer step of every tensor of the model on gfx950.
//
// Reference: apply_adam_update, update_matrix_adam_kernel, update_vector_adam_kernel (mgpu.cu:1040-1152), the Muon
// momentum, gather and apply kernels (muon_internal.cuh:15-74, :112-170).
//
// The reference draws two noise values per (weight, pair).  Which value a tensor draws for pair p and row or column i is
// hash_rng(seed + p + seed_base + off, i): tensors differ in a shift of the pair index only.  So ONE table
//     N[i][t] = noise_from_hash(seed + t, i)
// holds every tensor's noise, a tensor's row i being N[i][seed_base + off ...].  It has max(4 hidden, vocab) rows of
// pairs + 1000 layers entries -- 25 million hashes at hidden 256, 4 layers, 20,480 pairs, where panels of one tensor
// after the other were 440 million -- and the vote matrices  sum_p fit_p A_p[n] B_p[k]  of all tensors are int8 matrix
// products over shifted windows of it.
#include "egg_device.h"
#include "egg_launch.h"

#pragma clang fp contract(off)

// ---------------------------------------------------------------- noise table
// Thread: 16 consecutive entries of one row, one 16-byte store.  Bound by the hash (about 15 vector instructions an entry);
// entries no tensor reads are left out: rows past `layer_rows` belong to the embedding alone (layer 0 offsets below
// emb_t), and between the layers' windows there are gaps while there are fewer pairs than a layer's 1000 seeds.
// The first workgroups turn the fitness into byte masks and clear the update counter (when it is to be cleared).  In a whole
// step (end.acc) they do what stands between the forward and the update as well, four pairs a thread: losses and
// fitness, in device memory and in the host's copy, and the loss sums set back to zero: three launches less, and no copies
// when the host asks (a step of hidden 64, 2 layers, 64 members with its results read: 207 -> 146 us).
__device__ __forceinline__ void masks_of_fitness(const NoiseTable &nt, const int32_t *fit, int pairs) {
    __shared__ int other;
    if (threadIdx.x == 0) other = 0;
    __syncthreads();
    for (int c = threadIdx.x; c < nt.pairs_pad / 16; c += 256) {
        v4i neg, nz;
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
            neg[q] = n4; nz[q] = z4;
        }
        reinterpret_cast<v4i *>(nt.neg)[c] = neg;
        reinterpret_cast<v4i *>(nt.nonzero)[c] = nz;
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
    reinterpret_cast<int *>(nt.neg)[c] = n4;
    reinterpret_cast<int *>(nt.nonzero)[c] = z4;
}
__global__ void __launch_bounds__(256) k_noise_table(NoiseTable nt, const uint32_t *d_seed, const int32_t *fit, StepEnd end, int first, int pairs,
                                                     int mask, int rows, int layer_rows, int t_lo, int t_hi, int emb_t,
                                                     int n_layers, unsigned long long *counter) {
    if ((int)blockIdx.x < first) {
        if (blockIdx.x == 0 && threadIdx.x == 0 && counter) *counter = 0ull;
        if (end.acc) end_of_step(nt, end, pairs); else masks_of_fitness(nt, fit, pairs);
        return;
    }
    const int per_row = (t_hi - t_lo + 15) / 16;
    const int64_t i = (int64_t)((int)blockIdx.x - first) * 256 + threadIdx.x;
    const int r = (int)(i / per_row), t0 = t_lo + 16 * (int)(i % per_row);
    if (r >= rows || (r >= layer_rows && t0 >= emb_t)) return;
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
    *reinterpret_cast<v4i *>(nt.table + (size_t)r * nt.ld + t0) = o;
}
hipError_t egg_launch_noise_table(const NoiseTable &nt, const uint32_t *d_seed, const int32_t *d_fit, const StepEnd &end, int pairs, int mask, int rows,
                                  int layer_rows, int t_lo, int t_hi, int emb_t, int n_layers, unsigned long long *counter, hipStream_t s) {
    t_lo &= ~15;
    t_hi = (t_hi + 15) & ~15;
    if (rows < 1 || rows > nt.rows || t_lo < 0 || (size_t)t_hi > nt.ld) return hipErrorInvalidValue;
    const int64_t items = (int64_t)rows * ((t_hi - t_lo) / 16);
    const int first = end.acc ? (nt.pairs_pad / 4 + 255) / 256 : 1;
    hipLaunchKernelGGL(k_noise_table, dim3((unsigned)((items + 255) / 256 + first)), dim3(256), 0, s, nt, d_seed, d_fit, end, first, pairs, mask, rows,
                       layer_rows, t_lo, t_hi, emb_t, n_layers, counter);
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

typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));     // a tensor's window of the table starts at any byte
__device__ __forceinline__ v4i load16(const int8_t *p) { return *reinterpret_cast<const v4i_any *>(p); }
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
        for (int e = 0; e < 4; e++) { const int pr = first + 4 * q + e; v[e] = pr < pairs ? fit[pr] * sx8(x[q], e) : 0; }
        o[q] = pack4(v[0], v[1], v[2], v[3]);
    }
    return o;
}

// update_vector_adam_kernel (mgpu.cu:1114-1152): one wave per element, 16 pairs a lane
__device__ __forceinline__ int vector_element(const UpdLaunch &p, int gi) {
    const int lane = threadIdx.x & 63;
    const int d = find_last(p.n_vec, gi, [&](int i) { return p.vec[i].first; });
    const VecDesc t = p.vec[d];
    const int idx = gi - t.first;
    const int8_t *ra = p.noise.table + (size_t)idx * p.noise.ld + t.seed_base + t.off_a;
    const int8_t *rb = p.noise.table + (size_t)idx * p.noise.ld + t.seed_base + t.off_b;
    int vote = 0;
    if (!*p.noise.general) {
#pragma unroll 4
        for (int s = 16 * lane; s < p.noise.pairs_pad; s += 1024) {
            const v4i neg = *reinterpret_cast<const v4i *>(p.noise.neg + s), nz = *reinterpret_cast<const v4i *>(p.noise.nonzero + s);
            const v4i b = load16(rb + s), a = signed_noise(load16(ra + s), neg, nz);
#pragma unroll
            for (int q = 0; q < 4; q++) vote = dot4(a[q], b[q], vote);
            vote = sum_negative(b, neg, vote);
        }
    } else
        for (int pr = lane; pr < p.pairs; pr += 64) vote += p.fit[pr] * ra[pr] * rb[pr];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) vote += __shfl_xor(vote, off, 64);
    int ch = 0;
    if (lane == 0) {
        const AdamHyper hy = {p.beta1, p.beta2, p.eps, p.wd, 127};     // vector tensors keep the reference's +-127
        const float lr = (*p.d_lr) * t.lr_scale;
        float *st = t.state + (size_t)idx * 3;
        float m = st[0], v = st[1], acc = st[2];
        int w = t.W[idx];
        ch = adam_apply(m, v, acc, w, -(float)vote, lr, hy);
        t.W[idx] = (int8_t)w; st[0] = m; st[1] = v; st[2] = acc;
        if (ch && t.flags) t.flags[idx] = 1;
    }
    return ch;
}

// Votes and optimizer step of every matrix of a list (and of every vector tensor, in the workgroups behind the matrix
// tiles).  One workgroup per 64 (k) x 64 (n) tile of a vote matrix, whatever the matrix: all tiles of the model in one
// launch.  The pairs go by in chunks of 128: every thread fetches 16 pairs of two k rows and two n rows (a row's 128 bytes
// by eight neighbouring lanes; a window starts at any byte, so these are unaligned 16-byte loads), applies the fitness to
// the n rows and stores them into LDS in MFMA operand order; wave w multiplies the chunk's 32-pair step w, two by two
// fragments of 32 rows, so each fragment read feeds two MFMAs.  The next chunk's loads are in flight meanwhile; two LDS
// buffers, one barrier a chunk.  A chunk column (16 pairs of 64 rows) is 1,056 bytes, not 1,024, so that the eight lanes
// of a row store to different banks.  The four partial tiles are added up in two exchanges (half a tile each, then a
// quarter), after which wave w owns the 32 x 32 quarter (w >> 1, w & 1), applies the optimizer rule to it and writes the
// weights' fragment-major copy.  Bound by the loads of the table's windows (L2 and the memory-side cache): a tile reads
// 128 rows of pairs for 4,096 weights.  27 matrices and 54 vectors of hidden 256, 4 layers at 20,480 pairs: 2.9 ms for 109
// launches (panels, 32 x 32 tiles, copy, per matrix) -> 0.38 ms for this one and 0.02 ms for the table; 81 matrices
// and vectors of hidden 128 at 4,096 pairs: 0.70 -> 0.05 ms.
constexpr int CHUNK_COL = 1056, OPERAND = 8 * CHUNK_COL;
__global__ void __launch_bounds__(EGG_THREADS, 3) k_update(UpdLaunch p) {
    __shared__ __align__(16) int8_t lds[4 * OPERAND];
    __shared__ int corr[64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 5, j = lane & 31;
    if ((int)blockIdx.x >= p.tiles) {
        const int gi = ((int)blockIdx.x - p.tiles) * EGG_WAVES + wave;
        count_changes(p, gi < p.vec_total ? vector_element(p, gi) : 0, corr);
        return;
    }
    const MatDesc t = p.mat[find_last(p.n_mat, blockIdx.x, [&](int i) { return p.mat[i].tile_first; })];
    const int tiles_n = t.cols / 64, tile = blockIdx.x - t.tile_first;
    const int k0 = (tile / tiles_n) * 64, n0 = (tile % tiles_n) * 64;
    const int c = threadIdx.x & 7, r = threadIdx.x >> 3;
    const size_t down = 32 * p.noise.ld;
    const int8_t *pa = p.noise.table + (size_t)(n0 + r) * p.noise.ld + t.t_a + 16 * c;
    const int8_t *pb = p.noise.table + (size_t)(k0 + r) * p.noise.ld + t.t_b + 16 * c;
    const int general = *p.noise.general;
    v4i a0, a1, b0, b1, neg, nz;
    auto fetch = [&](int s) {
        a0 = load16(pa + s); a1 = load16(pa + down + s); b0 = load16(pb + s); b1 = load16(pb + down + s);
        neg = *reinterpret_cast<const v4i *>(p.noise.neg + s + 16 * c);
        nz = *reinterpret_cast<const v4i *>(p.noise.nonzero + s + 16 * c);
    };
    v16i acc[2][2];
    zero_acc<2>(acc[0]); zero_acc<2>(acc[1]);
    int c0 = 0, c1 = 0, buf = 0;
    fetch(0);
    for (int s = 0; s < p.noise.pairs_pad; s += 128) {
        if (!general) {
            a0 = signed_noise(a0, neg, nz); a1 = signed_noise(a1, neg, nz);
            c0 = sum_negative(b0, neg, c0); c1 = sum_negative(b1, neg, c1);
        } else {
            a0 = scaled_noise(a0, p.fit, s + 16 * c, p.pairs); a1 = scaled_noise(a1, p.fit, s + 16 * c, p.pairs);
        }
        int8_t *A = lds + buf * 2 * OPERAND, *B = A + OPERAND;
        *reinterpret_cast<v4i *>(A + c * CHUNK_COL + r * 16) = a0;
        *reinterpret_cast<v4i *>(A + c * CHUNK_COL + (r + 32) * 16) = a1;
        *reinterpret_cast<v4i *>(B + c * CHUNK_COL + r * 16) = b0;
        *reinterpret_cast<v4i *>(B + c * CHUNK_COL + (r + 32) * 16) = b1;
        if (s + 128 < p.noise.pairs_pad) fetch(s + 128);
        __syncthreads();
        v4i fa[2], fb[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            fa[h] = *reinterpret_cast<const v4i *>(A + (2 * wave + g) * CHUNK_COL + (32 * h + j) * 16);
            fb[h] = *reinterpret_cast<const v4i *>(B + (2 * wave + g) * CHUNK_COL + (32 * h + j) * 16);
        }
#pragma unroll
        for (int hk = 0; hk < 2; hk++)
#pragma unroll
            for (int hn = 0; hn < 2; hn++) acc[hk][hn] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[hk], fa[hn], acc[hk][hn], 0, 0, 0);
        buf ^= 1;
    }
    // sums over the negative pairs of the k rows, over the eight chunk columns
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) { c0 += __shfl_xor(c0, o, 64); c1 += __shfl_xor(c1, o, 64); }
    __syncthreads();
    int *red = reinterpret_cast<int *>(lds);                 // [wave][2 tiles][16][64], then [wave][16][64]
    const bool hi = wave >= 2, odd = wave & 1;
    v16i mine[2];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            red[((wave * 2 + h) * 16 + e) * 64 + lane] = hi ? acc[0][h][e] : acc[1][h][e];
            mine[h][e] = hi ? acc[1][h][e] : acc[0][h][e];
        }
    if (c == 0) { corr[r] = c0; corr[r + 32] = c1; }
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
    const int kt = k0 + 32 * (wave >> 1), n = n0 + 32 * (wave & 1) + j;
#pragma unroll
    for (int e = 0; e < 16; e++) vote[e] += red[((wave ^ 1) * 16 + e) * 64 + lane] + corr[kt - k0 + 8 * (e >> 2) + 4 * g + (e & 3)];
    // accumulator register 4q + e of lane (n, g) -> k = kt + 8q + 4g + e; blocked index of (k, n) (mgpu.cu:1085-1089)
    const float lr = p.d_lr ? (*p.d_lr) * t.lr_scale : 0.f;
    const AdamHyper hy = {p.beta1, p.beta2, p.eps, p.wd, t.limit};
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
        if (t.muon_x) {
            // muon_momentum_update_kernel + muon_gather_m_kernel (muon_internal.cuh:15-74): m = mu*m + vote
            float4 *sp = reinterpret_cast<float4 *>(t.state + idx * 2);
            const float4 s0 = sp[0], s1 = sp[1];
            float mv[4] = {s0.x, s0.z, s1.x, s1.z};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float m = p.muon_momentum * mv[e];
                mv[e] = m + (float)vote[4 * q + e];
                t.muon_x[(size_t)(kt + 8 * q + 4 * g + e) * t.cols + n] = mv[e];
            }
            sp[0] = make_float4(mv[0], s0.y, mv[1], s0.w);
            sp[1] = make_float4(mv[2], s1.y, mv[3], s1.w);
            continue;
        }
        const int w4 = *reinterpret_cast<const int *>(t.W + idx);
        float4 *sp = reinterpret_cast<float4 *>(t.state + idx * 3);
        const float4 s0 = sp[0], s1 = sp[1], s2 = sp[2];
        float st[12] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w, s2.x, s2.y, s2.z, s2.w};
        int wv[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            wv[e] = sx8(w4, e);
            const int ch = adam_apply(st[3 * e], st[3 * e + 1], st[3 * e + 2], wv[e], -(float)vote[4 * q + e], lr, hy);
            changes += ch;
            // overlay flags (de/include/optimizer/adam.cuh:77-83): every writer stores the same value, so plain stores do
            if (ch && p.flags) { p.flags[t.offset + kt + 8 * q + 4 * g + e] = 1; p.flags[t.offset + t.rows + n] = 1; }
        }
        unit[q] = pack4(wv[0], wv[1], wv[2], wv[3]);
        *reinterpret_cast<int *>(t.W + idx) = unit[q];
        sp[0] = make_float4(st[0], st[1], st[2], st[3]);
        sp[1] = make_float4(st[4], st[5], st[6], st[7]);
        sp[2] = make_float4(st[8], st[9], st[10], st[11]);
    }
    if (p.votes_out || t.muon_x) return;
    *frag_unit(t, kt >> 5, g, n) = unit;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) changes += __shfl_xor(changes, off, 64);
    __syncthreads();                                         // the corrections have been read
    count_changes(p, changes, corr);
}
int egg_update_blocks(const UpdLaunch &p) { return p.tiles + (p.vec_total + EGG_WAVES - 1) / EGG_WAVES; }
hipError_t egg_launch_update(const UpdLaunch &p, hipStream_t s) {
    const int blocks = egg_update_blocks(p);
    if (blocks < 1) return hipSuccess;
    if (p.noise.pairs_pad % 128 || (p.tiles && p.n_mat < 1) || (p.vec_total && p.n_vec < 1)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_update, dim3(blocks), dim3(EGG_THREADS), 0, s, p);
    return hipGetLastError();
}

// muon_apply_update_kernel (muon_internal.cuh:112-170) for every matrix of a list: a thread takes one 16-byte unit of the
// fragment-major copy (16 rows of one column), so neighbouring lanes read and write neighbouring columns throughout.
// Bound by memory (22 bytes an element).
__global__ void __launch_bounds__(256) k_muon_apply(UpdLaunch p, float wd) {
    __shared__ int sums[EGG_WAVES];
    const MatDesc t = p.mat[find_last(p.n_mat, blockIdx.x, [&](int i) { return p.mat[i].tile_first; })];
    const int u = ((int)blockIdx.x - t.tile_first) * 256 + (int)threadIdx.x;       // 256 units to a 64 x 64 tile
    const int n = u % t.cols, kk = u / t.cols, ks = kk >> 1, g = kk & 1;
    const float lr = (*p.d_lr) * t.lr_scale;
    int changes = 0;
    v4i unit;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int kr = 32 * ks + 8 * q + 4 * g;
        const size_t idx = ((size_t)(kr >> 2) * t.cols + n) * 4;
        const int w4 = *reinterpret_cast<const int *>(t.W + idx);
        float4 *sp = reinterpret_cast<float4 *>(t.state + idx * 2);
        const float4 s0 = sp[0], s1 = sp[1];
        float acc[4] = {s0.y, s0.w, s1.y, s1.w};
        int wv[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            wv[e] = sx8(w4, e);
            const float x = t.muon_x[(size_t)(kr + e) * t.cols + n];
            const float wdw = wd * (float)wv[e];
            const float step = (-lr) * (x + wdw);
            acc[e] += step;
            changes += threshold_apply(acc[e], wv[e], t.limit);
        }
        unit[q] = pack4(wv[0], wv[1], wv[2], wv[3]);
        *reinterpret_cast<int *>(t.W + idx) = unit[q];
        sp[0] = make_float4(s0.x, acc[0], s0.z, acc[1]);
        sp[1] = make_float4(s1.x, acc[2], s1.z, acc[3]);
    }
    *frag_unit(t, ks, g, n) = unit;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) changes += __shfl_xor(changes, off, 64);
    count_changes(p, changes, sums);
}
hipError_t egg_launch_muon_apply(const UpdLaunch &p, float wd, hipStream_t s) {
    if (p.tiles < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_muon_apply, dim3(p.tiles), dim3(256), 0, s, p, wd);
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
