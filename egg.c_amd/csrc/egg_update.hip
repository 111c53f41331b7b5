// egg_update.hip -- fitness, the adaptive overlay's rule, ternary packing, sampling and the Newton-Schulz chain on gfx950
// (votes and the optimizer step: egg_votes.hip).
//
// Reference: compute_fitness_kernel, mgpu.cu:1031-1036 ("mgpu.cu" = full_cuda_train_transformer_adam_mgpu.cu);
// update_overlay_kernel, de/src/kernels.cu:61-77; generate_sequence_kernel's sampling; perform_newton_schulz.
#include "../../include/egg_hip.h"
#include "egg_device.h"
#include "egg_launch.h"
#include <mutex>
#include <string>
#include <type_traits>

#pragma clang fp contract(off)

__global__ void k_noise_fill(uint32_t seed, uint32_t first, int n, int mask, int8_t *out) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (int8_t)noise_from_hash(seed, first + (uint32_t)i, mask);
}
hipError_t egg_launch_noise_fill(uint32_t seed, uint32_t first, int n, int mask, int8_t *out, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_noise_fill, dim3((n + 255) / 256), dim3(256), 0, s, seed, first, n, mask, out);
    return hipGetLastError();
}

__global__ void k_zero_u64(unsigned long long *p, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}
hipError_t egg_launch_zero_u64(unsigned long long *p, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero_u64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

// accum_loss[p] = (int32_t) my_loss   (mgpu.cu:1028); the sums go back to zero for the next forward
__global__ void k_loss_finalize(unsigned long long *acc, int32_t *loss, int first, int count) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) { loss[first + i] = (int32_t)(long long)acc[first + i]; acc[first + i] = 0ull; }
}
hipError_t egg_launch_loss_finalize(unsigned long long *acc, int32_t *loss, int first, int count, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_loss_finalize, dim3((count + 255) / 256), dim3(256), 0, s, acc, loss, first, count);
    return hipGetLastError();
}

// mgpu.cu:1031-1036
__global__ void k_fitness(const int32_t *loss, int32_t *fit, int pairs) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= pairs) return;
    int32_t p = loss[2 * i], n = loss[2 * i + 1];
    fit[i] = (p < n) ? 1 : ((n < p) ? -1 : 0);
}
hipError_t egg_launch_fitness(const int32_t *loss, int32_t *fit, int pairs, hipStream_t s) {
    if (pairs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fitness, dim3((pairs + 255) / 256), dim3(256), 0, s, loss, fit, pairs);
    return hipGetLastError();
}

// Ternary-packed matrix weights (no counterpart in the reference, whose weights are plain int8): four consecutive
// elements of the blocked matrix -- the four input rows that share one dword -- per byte, element e in bits 2e+1..2e
// as a 2-bit two's complement number (00 = 0, 01 = +1, 11 = -1).  Unpacking writes the canonical int8 blob, from which
// the fragment-major copy the MFMAs read is rebuilt.
__global__ void k_ternary_unpack(const uint8_t *packed, int *words, int n_words) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_words) return;
    const int b = packed[i];
    int w = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int v = ((b >> (2 * e)) & 3) << 30 >> 30;       // sign-extend the 2-bit field
        w |= (v & 0xff) << (8 * e);
    }
    words[i] = w;
}
__global__ void k_ternary_pack(const int *words, uint8_t *packed, int n_words, int *bad) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_words) return;
    const int w = words[i];
    int b = 0, out_of_range = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int v = sx8(w, e);
        out_of_range |= (v < -1) | (v > 1);
        b |= (v & 3) << (2 * e);
    }
    packed[i] = (uint8_t)b;
    if (out_of_range) *bad = 1;      // every writer stores the same value
}
hipError_t egg_launch_ternary_unpack(const uint8_t *packed, int8_t *dst, int n_elems, hipStream_t s) {
    const int n = n_elems / 4;
    hipLaunchKernelGGL(k_ternary_unpack, dim3((n + 255) / 256), dim3(256), 0, s, packed, reinterpret_cast<int *>(dst), n);
    return hipGetLastError();
}
hipError_t egg_launch_ternary_pack(const int8_t *src, uint8_t *packed, int n_elems, int *d_bad, hipStream_t s) {
    const int n = n_elems / 4;
    hipLaunchKernelGGL(k_ternary_pack, dim3((n + 255) / 256), dim3(256), 0, s, reinterpret_cast<const int *>(src), packed, n, d_bad);
    return hipGetLastError();
}

// update_overlay_kernel (de/src/kernels.cu:61-77) over a list of segments of the overlay blob
__global__ void k_overlay_update(int8_t *overlay, int8_t *q, int8_t *flags, const OvSeg *segs, int inc, int dec) {
    const OvSeg sg = segs[blockIdx.y];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= sg.count) return;
    const int at = sg.offset + i;
    int ov = overlay[at];
    if (flags[at]) { ov += inc; if (ov > 127) ov = 127; }
    else { ov -= dec; if (ov < -127) ov = -127; }
    flags[at] = 0;
    overlay[at] = (int8_t)ov;
    q[at] = (int8_t)overlay_q(ov);
}
hipError_t egg_launch_overlay_update(int8_t *overlay, int8_t *q, int8_t *flags, const OvSeg *d_segs, int n_segs, int max_count,
                                     int inc, int dec, hipStream_t s) {
    if (n_segs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_overlay_update, dim3((max_count + 255) / 256, n_segs), dim3(256), 0, s, overlay, q, flags, d_segs, inc, dec);
    return hipGetLastError();
}
__global__ void k_overlay_q(const int8_t *overlay, int8_t *q, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) q[i] = (int8_t)overlay_q(overlay[i]);
}
hipError_t egg_launch_overlay_q(const int8_t *overlay, int8_t *q, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_overlay_q, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, overlay, q, n);
    return hipGetLastError();
}

// Three-pass LUT sampling of generate_sequence_kernel (mgpu.cu:1212-1283) for one position: maximum logit,
// sum of EXP_LUT[clamp(max - logit)], threshold hash_rng(seed + t*555, 0) % sum, then the first vocabulary entry
// whose running sum exceeds the threshold.  The reference accumulates in thread order with thread `tid` owning
// v = tid, tid + bt, ... (bt = its block size = hidden rounded up to 32, at most 1024), so for bt < vocab the scan
// order is thread-major, not natural; `bt` reproduces that: every reference thread's sum is formed (in parallel), the
// thread in whose range the threshold falls is found from their prefix sums, and its entries are walked.
// One workgroup; `ws` holds the vocab weights.  TOK: the token type of the buffer (bytes, or uint32 above vocab 256).
__device__ __forceinline__ void sample_select(const int *ex, int vocab, int bt, uint32_t seed, int t, long long *tsum, int *selected) {
    for (int tid = threadIdx.x; tid < bt; tid += 256) {
        long long sum = 0;
        for (int v = tid; v < vocab; v += bt) sum += ex[v];
        tsum[tid] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        long long total = 0;
        for (int tid = 0; tid < bt; tid++) total += tsum[tid];
        const uint32_t r = hash_rng(seed + (uint32_t)t * 555u, 0);
        const long long thresh = total > 0 ? (long long)r % total : 0;
        int sel = 0; long long running = 0; bool done = false;
        for (int tid = 0; tid < bt && !done; tid++) {
            if (running + tsum[tid] <= thresh) { running += tsum[tid]; continue; }
            for (int v = tid; v < vocab; v += bt) {
                running += ex[v];
                if (running > thresh) { sel = v; done = true; break; }
            }
        }
        *selected = sel;
    }
}
template <typename TOK>
__global__ void __launch_bounds__(256) k_sample(const int32_t *logits, const int32_t *exp_lut, int vocab, int bt,
                                                uint32_t seed, int t, int *ws, TOK *out) {
    __shared__ long long tsum[1024];
    __shared__ int red[256];
    __shared__ int sel;
    int mx = INT_MIN;
    for (int v = threadIdx.x; v < vocab; v += 256) mx = max(mx, logits[v]);
    red[threadIdx.x] = mx; __syncthreads();
    for (int o = 128; o > 0; o >>= 1) { if ((int)threadIdx.x < o) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + o]); __syncthreads(); }
    mx = red[0];
    for (int v = threadIdx.x; v < vocab; v += 256) {
        int idx = mx - logits[v];
        idx = idx < 0 ? 0 : (idx > 255 ? 255 : idx);
        ws[v] = exp_lut[idx];
    }
    __syncthreads();
    sample_select(ws, vocab, bt, seed, t, tsum, &sel);
    if (threadIdx.x == 0) *out = (TOK)sel;
}
hipError_t egg_launch_sample(const int32_t *logits, const int32_t *exp_lut, int vocab, int bt, uint32_t seed, int t,
                             int *ws, void *out, int token_bytes, hipStream_t s) {
    if (bt < 1 || bt > 1024 || !ws) return hipErrorInvalidValue;
    if (token_bytes == 4) hipLaunchKernelGGL(k_sample<uint32_t>, dim3(1), dim3(256), 0, s, logits, exp_lut, vocab, bt, seed, t, ws, (uint32_t *)out);
    else hipLaunchKernelGGL(k_sample<uint8_t>, dim3(1), dim3(256), 0, s, logits, exp_lut, vocab, bt, seed, t, ws, (uint8_t *)out);
    return hipGetLastError();
}

// The d-eggs sampler (d-eggs/src/kernels.cu:382-478): every occurrence of v among the tokens up to position t lowers
// v's logit by penalty_int (repeated int32 subtraction: wraps), the differences to the maximum are divided by the
// temperature in float and truncated, entries below min_p_limit are left out, the rest weigh
// EXP_LUT[clamp(-scaled, 0, 255)]; threshold and scan order as above.  `ws` holds 2 * vocab ints.
// float -> int32 as the GPU's conversion does it: truncation toward zero, saturation at the ends, NaN -> 0
__device__ __forceinline__ int sat_f2i(float x) {
    if (x != x) return 0;
    if (x >= 2147483648.0f) return INT_MAX;
    if (x <= -2147483648.0f) return INT_MIN;
    return (int)x;
}
template <typename TOK>
__global__ void __launch_bounds__(256) k_sample_deggs(const int32_t *logits, const int32_t *exp_lut, int vocab, int bt, uint32_t seed, int t,
                                                      const TOK *tokens, float temp, int min_p_limit, int penalty_int, int *ws, TOK *out) {
    __shared__ long long tsum[1024];
    __shared__ int red[256];
    __shared__ int sel;
    int *lg = ws, *ex = ws + vocab;
    int mx = INT_MIN;
    for (int v = threadIdx.x; v < vocab; v += 256) {
        uint32_t count = 0;
        for (int i = 0; i <= t; i++) count += (int)tokens[i] == v;
        const int l = (int)((uint32_t)logits[v] - count * (uint32_t)penalty_int);
        lg[v] = l;
        mx = max(mx, l);
    }
    red[threadIdx.x] = mx; __syncthreads();
    for (int o = 128; o > 0; o >>= 1) { if ((int)threadIdx.x < o) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + o]); __syncthreads(); }
    mx = red[0];
    for (int v = threadIdx.x; v < vocab; v += 256) {
        const int shifted = (int)((uint32_t)lg[v] - (uint32_t)mx);
        const int scaled = sat_f2i((float)shifted / temp);
        int e = 0;
        if (scaled >= min_p_limit) {
            int idx = (int)(0u - (uint32_t)scaled);
            idx = idx < 0 ? 0 : (idx > 255 ? 255 : idx);
            e = exp_lut[idx];
        }
        ex[v] = e;
    }
    __syncthreads();
    sample_select(ex, vocab, bt, seed, t, tsum, &sel);
    if (threadIdx.x == 0) *out = (TOK)sel;
}
hipError_t egg_launch_sample_deggs(const int32_t *logits, const int32_t *exp_lut, int vocab, int bt, uint32_t seed, int t,
                                   const void *tokens, float temp, int min_p_limit, int penalty_int, int *ws, void *out, int token_bytes, hipStream_t s) {
    if (bt < 1 || bt > 1024 || t < 0 || !ws) return hipErrorInvalidValue;
    if (token_bytes == 4)
        hipLaunchKernelGGL(k_sample_deggs<uint32_t>, dim3(1), dim3(256), 0, s, logits, exp_lut, vocab, bt, seed, t, (const uint32_t *)tokens, temp,
                           min_p_limit, penalty_int, ws, (uint32_t *)out);
    else
        hipLaunchKernelGGL(k_sample_deggs<uint8_t>, dim3(1), dim3(256), 0, s, logits, exp_lut, vocab, bt, seed, t, (const uint8_t *)tokens, temp,
                           min_p_limit, penalty_int, ws, (uint8_t *)out);
    return hipGetLastError();
}

// canonical blocked weights -> fragment-major copy consumed by the GEMM kernels (layout in egg_device.h)
__global__ void k_swizzle(const uint32_t *src, v4i *dst, int K, int N, int B, int nat) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= K * N / 16) return;
    const int per_block = B * B / 16;
    int block = c / per_block, idx = c % per_block;
    int p = idx / B, n = idx % B, kb = block / (N / B), nb = block % (N / B), ks = p >> 1, g = p & 1;
    v4i v;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        int kq = (kb * B) / 4 + 8 * ks + (nat ? (4 * g + q) : (2 * q + g));
        v[q] = (int)src[(size_t)kq * N + nb * B + n];
    }
    dst[c] = v;
}
hipError_t egg_launch_swizzle(const int8_t *W, int8_t *Wf, int K, int N, int B, int nat, hipStream_t s) {
    if (K % B || N % B || B % 32) return hipErrorInvalidValue;
    int chunks = K * N / 16;
    hipLaunchKernelGGL(k_swizzle, dim3((chunks + 255) / 256), dim3(256), 0, s, reinterpret_cast<const uint32_t *>(W),
                       reinterpret_cast<v4i *>(Wf), K, N, B, nat);
    return hipGetLastError();
}

// ---------------------------------------------------------------- Newton-Schulz (muon_internal.cuh:182-342)
typedef float v16f __attribute__((ext_vector_type(16)));

// Every kernel of the chain takes a batch of same-shape matrices, one per blockIdx.y (matrix b's operands sit b strides
// further on); what is computed for a matrix does not depend on the batch it runs in.
// sum of squares in two deterministic stages (cublasSnrm2 in the reference): 256 partial sums per matrix
__global__ void __launch_bounds__(256) k_sumsq_partial(const float *x, int n, float *partials) {
    __shared__ float sh[256];
    x += (size_t)blockIdx.y * n; partials += (size_t)blockIdx.y * 256;
    float s = 0.f;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) { float v = x[i]; s += v * v; }
    sh[threadIdx.x] = s; __syncthreads();
    for (int o = 128; o > 0; o >>= 1) { if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o]; __syncthreads(); }
    if (threadIdx.x == 0) partials[blockIdx.x] = sh[0];
}
__global__ void __launch_bounds__(256) k_norm_finish(const float *partials, int n, float *norm) {
    __shared__ float sh[256];
    partials += (size_t)blockIdx.y * 256;
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += 256) s += partials[i];
    sh[threadIdx.x] = s; __syncthreads();
    for (int o = 128; o > 0; o >>= 1) { if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o]; __syncthreads(); }
    if (threadIdx.x == 0) norm[blockIdx.y] = sqrtf(sh[0]);
}
// muon_scale_by_norm_kernel (muon_internal.cuh:77-87)
__global__ void k_scale_by_norm(float *x, const float *norm, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { float nv = norm[blockIdx.y]; if (nv > 1e-6f) x[(size_t)blockIdx.y * n + i] /= nv; }
}

// C[M][N] (row-major, ldc = N) = epilogue(sum_k A(i,k) B(k,j)), one workgroup per 32x32 tile on
// v_mfma_f32_32x32x2_f32.  Each operand is given by two strides of which one is 1 (a row-major matrix or its
// transpose); AK / BK say that it is the k stride.  An operand whose k stride is 1 is read with one 16-byte load per lane
// (four consecutive k of the lane's row or column); the other kind has its rows or columns side by side in memory and is
// read with fully coalesced 4-byte loads.  The k range is dealt to the four waves in blocks of eight (wave w takes blocks
// w, w + 4, ...); within a block, MFMA e multiplies the k pair {8c + e, 8c + 4 + e}.  The partial tiles are added in wave
// order in LDS, so the summation order is fixed and results are reproducible; wave q writes rows 8q + 4g + e of the
// tile.  mode 0: C = alpha * acc.  mode 1: C = (i == j ? 3 : 0) - acc  (3I - G, muon_internal.cuh:91-109).

template <bool AK, bool BK>
__global__ void __launch_bounds__(EGG_THREADS) k_sgemm(const float *A, long lda, long batch_a, const float *B, long ldb, long batch_b,
                                                      float *C, int M, int N, int K, float alpha, int mode) {
    __shared__ float red[EGG_WAVES][16][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 5, j = lane & 31;
    const int tiles_n = N / 32, tile = blockIdx.x;
    const int i0 = (tile / tiles_n) * 32, j0 = (tile % tiles_n) * 32;
    A += (long)blockIdx.y * batch_a; B += (long)blockIdx.y * batch_b; C += (size_t)blockIdx.y * M * N;
    v16f acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    // lane (j, g) supplies A(i0 + j, k) and B(k, j0 + j) for k = 8c + 4g + e
    const float *ap = AK ? A + (long)(i0 + j) * lda + 4 * g : A + (long)(4 * g) * lda + i0 + j;
    const float *bp = BK ? B + (long)(j0 + j) * ldb + 4 * g : B + (long)(4 * g) * ldb + j0 + j;
#pragma unroll 4
    for (int c = wave; c < K / 8; c += EGG_WAVES) {
        v4f a4, b4;
        if (AK) a4 = *reinterpret_cast<const v4f *>(ap + 8 * c);
        else {
#pragma unroll
            for (int e = 0; e < 4; e++) a4[e] = ap[(long)(8 * c + e) * lda];
        }
        if (BK) b4 = *reinterpret_cast<const v4f *>(bp + 8 * c);
        else {
#pragma unroll
            for (int e = 0; e < 4; e++) b4[e] = bp[(long)(8 * c + e) * ldb];
        }
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a4[e], b4[e], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; r++) red[wave][r][lane] = acc[r];
    __syncthreads();
    const int q = wave;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float v = red[0][4 * q + e][lane];
#pragma unroll
        for (int w = 1; w < EGG_WAVES; w++) v += red[w][4 * q + e][lane];
        const int i = i0 + 8 * q + 4 * g + e, jj = j0 + j;
        C[(size_t)i * N + jj] = (mode == 1) ? ((i == jj ? 3.0f : 0.0f) - v) : alpha * v;
    }
}
// The same product for M and N that are multiples of 64, with the operands staged once per workgroup through LDS and every
// output element summed by one wave over the whole of K (no partial tiles to add up).  A workgroup owns a TILE x TILE
// block of C, TILE = 64 WT: wave (wm, wn) owns the 32 WT x 32 WT quarter as WT x WT MFMA tiles.  A TILE x 32 chunk of A
// and a 32 x TILE chunk of B go global -> registers -> LDS (the next chunk's loads are in flight while the MFMAs of the
// current one run, and those of the one behind it).
// The float32 matrix instruction does 64 multiplications a clock and SIMD, the bf16 one 1,024, so every operand is taken apart on its
// way into LDS: x = x0 + x1 + x2, each the nearest bf16 of what is left (8 + 8 + 8 bits: 24, the float's own), and a product is
// eight exact partial products: all but x2 y2, which is below 2^-34 of it.  (x1 y2 and x2 y1 reach 2^-24, half a unit of the last place.)
// The bf16 instruction aligns its sixteen products and its addend to the largest of them, so a product that meets a smaller sum can be off by
// a whole unit of the last place and a long sum is rounded once for each instruction.  Therefore the sum over k does not pass through
// it: x0 y0 of a chunk of 32 k and the seven others, smallest first, each start from zero, and their sum is added to the accumulator by the
// vector unit, one rounding for 32 k where the float32 instruction has sixteen; a single product is rounded as float32 multiplication rounds it.
// Relative errors of five iterations against 64 bits, float32 instruction -> this: random matrices 9.1e-7 -> 2.7e-7 at 512 x 512, 4.2e-7 -> 1.3e-7 at
// 512 x 2048, 3.3e-7 -> 1.7e-7 at 64 x 64; rank one 6.2e-6 -> 1.4e-6; rows scaled over e^4 9.7e-7 -> 2.7e-7 and 3.9e-7 -> 1.6e-7, columns 3.5e-7 -> 2.3e-7 and
// 1.05e-6 -> 3.8e-7; two elements a row, where hardly anything is summed, 1.3e-7 -> 1.3e-7 (0.83 to 1.03 of it over the sizes).  (One
// accumulator through all instructions: 6.0e-7, 2.7e-7, 2.5e-7, 3.9e-6; 1.6 times the float32 instruction's for columns scaled over e^4 at 2048 x 512, 1.3 times for
// two elements a row.)  Parts below 2^-126, so of elements below 2^-110 of the matrix' norm, are lost.
// Times, float32 instruction -> this: G (upper half) of 32 matrices of 512 x 512 56 -> 61 us, X B of them 80 -> 69, G of nine 512 x 2048 83 -> 76 and
// 2048 x 512 84 -> 87, their X P 111 and 123 -> 102, products of nine 512 x 512 30 -> 25, of eighteen 41 -> 34: those are 16 chunks one after the other, at one to three workgroups a CU.
// The whole chain of a model of hidden 64 / 128 / 256 / 512: 0.26 / 0.33 / 0.48 / 1.76 -> 0.25 / 0.32 / 0.47 / 1.60 ms.
// An operand sits in LDS as three planes [row][k] of bf16 with rows 80 bytes apart (a lane reads eight consecutive k of its row as 16
// bytes; 16 such rows fall on all banks once).  One whose k stride is not 1 is turned over on the way: a thread
// takes four rows at two consecutive k.
// What an output element is summed from, and in which order, does not depend on WT: the two tile sizes give bit-identical
// results, so the host may pick by the size of the grid.
// SYM: C is symmetric; only tiles on and above the diagonal are computed, elements above it are stored twice (36 of 64 tiles
// at 512 columns).
// A launch may multiply two left sides with the same B (blockIdx.z).  Epilogues, v the sum over k, e0 and e1 elements of
// other matrices at the same place:
enum { NS_SCALE, NS_B, NS_GRAM, NS_STEP, NS_FACTOR };
struct SgemmJob {
    const float *A; long batch_a; float *C; const float *e0, *e1; float *C2; int mode; float alpha;
};
struct SgemmJobs { SgemmJob j[2]; };
// v of the 16 elements (i + 8q + e, jj) of a lane (at: the first one's place) -> what is stored.  All reads of the other matrices come first: left
// between the stores, which may alias them as far as the compiler knows, each would be waited for by itself.
__device__ __forceinline__ void ns_epilogue(const SgemmJob &job, v16f &v, int i, int jj, size_t at, int N) {
    v16f x, y;
    if (job.mode == NS_STEP || job.mode == NS_FACTOR)
#pragma unroll
        for (int r = 0; r < 16; r++) x[r] = job.e0[at + (size_t)(8 * (r >> 2) + (r & 3)) * N];
    if (job.mode == NS_STEP)
#pragma unroll
        for (int r = 0; r < 16; r++) y[r] = job.e1[at + (size_t)(8 * (r >> 2) + (r & 3)) * N];
#pragma unroll
    for (int r = 0; r < 16; r++)
        switch (job.mode) {
            case NS_B: v[r] = (i + 8 * (r >> 2) + (r & 3) == jj ? 3.0f : 0.0f) - v[r]; break;       // 3I - G (muon_internal.cuh:91-109)
            case NS_STEP: v[r] = 0.25f * ((9.0f * x[r] - 6.0f * y[r]) + v[r]); break;               // G (3I - G)^2 / 4 from G, G^2, G^3
            case NS_FACTOR: v[r] = 0.5f * (3.0f * x[r] - v[r]); break;                              // P (3I - G) / 2
            default: v[r] = job.alpha * v[r];
        }
}
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
constexpr int NS_PLANES = 3;
// two values as NS_PLANES pairs of bf16
__device__ __forceinline__ void split_bf16(float a, float b, uint32_t *pl) {
#pragma unroll
    for (int p = 0; p < NS_PLANES; p++) {
        const v2f x = {a, b};
        pl[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, v2bf));
        a -= __uint_as_float(pl[p] << 16);
        b -= __uint_as_float(pl[p] & 0xffff0000u);
    }
}
template <bool AK, bool BK, int WT, bool SYM>
__global__ void __launch_bounds__(EGG_THREADS, WT == 1 ? 3 : 2) k_sgemm_lds(SgemmJobs jobs, long lda, const float *B, long ldb, long batch_b, int M, int N, int K) {
    constexpr int TILE = 64 * WT, KC = 32, ROW = 80, PLANE = TILE * ROW, PIECES = TILE * KC / 4 / EGG_THREADS;
    constexpr int AHEAD = WT == 2 ? 1 : 2;      // (two chunks ahead do not fit the registers beside WT = 2's accumulators)
    __shared__ __align__(16) int8_t As[NS_PLANES * PLANE];
    __shared__ __align__(16) int8_t Bs[NS_PLANES * PLANE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 5, j = lane & 31, tid = threadIdx.x;
    const int wm = wave >> 1, wn = wave & 1;
    const int tiles_n = N / TILE;
    int ti = blockIdx.x / tiles_n, tj = blockIdx.x % tiles_n;
    if (SYM) {
        ti = 0; tj = blockIdx.x;
        while (tj >= tiles_n - ti) { tj -= tiles_n - ti; ti++; }
        tj += ti;
    }
    const int i0 = ti * TILE, j0 = tj * TILE;
    const SgemmJob job = jobs.j[blockIdx.z];
    const float *const A = job.A + (long)blockIdx.y * job.batch_a;
    B += (long)blockIdx.y * batch_b;
    const size_t out = (size_t)blockIdx.y * M * N;
    v16f acc[WT][WT];
#pragma unroll
    for (int a = 0; a < WT; a++)
#pragma unroll
        for (int b = 0; b < WT; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] = 0.f;
    // global -> registers: PIECES 16-byte pieces of each operand's chunk per thread, AHEAD chunks early.  k stride 1: four k of a row a piece; otherwise four rows at k, and the next piece at
    // k + 1, sixteen such pairs of k in sixteen lanes (their writes fall on different banks).
    v4f ra[AHEAD][PIECES], rb[AHEAD][PIECES];
    auto load_operand = [&](auto kone, const float *X, long ld, int x0, int k0, v4f *r) {
#pragma unroll
        for (int p = 0; p < PIECES; p++) {
            constexpr bool KONE = decltype(kone)::value;
            const int idx = tid + EGG_THREADS * (KONE ? p : p >> 1);
            r[p] = KONE ? *reinterpret_cast<const v4f *>(X + (long)(x0 + (idx >> 3)) * ld + k0 + 4 * (idx & 7))
                        : *reinterpret_cast<const v4f *>(X + (long)(k0 + 2 * (idx & 15) + (p & 1)) * ld + x0 + 4 * (idx >> 4));
        }
    };
    auto store_operand = [&](auto kone, int8_t *X, const v4f *r) {
        constexpr bool KONE = decltype(kone)::value;
        if constexpr (KONE) {
#pragma unroll
            for (int p = 0; p < PIECES; p++) {
                const int idx = tid + EGG_THREADS * p;
                uint32_t lo[NS_PLANES], hi[NS_PLANES];
                split_bf16(r[p][0], r[p][1], lo);
                split_bf16(r[p][2], r[p][3], hi);
#pragma unroll
                for (int pl = 0; pl < NS_PLANES; pl++)
                    *reinterpret_cast<uint64_t *>(X + pl * PLANE + (idx >> 3) * ROW + 8 * (idx & 7)) = (uint64_t)hi[pl] << 32 | lo[pl];
            }
        } else {
#pragma unroll
            for (int p = 0; p < PIECES; p += 2) {
                const int idx = tid + EGG_THREADS * (p >> 1);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t w[NS_PLANES];
                    split_bf16(r[p][e], r[p + 1][e], w);
#pragma unroll
                    for (int pl = 0; pl < NS_PLANES; pl++) *reinterpret_cast<uint32_t *>(X + pl * PLANE + (4 * (idx >> 4) + e) * ROW + 4 * (idx & 15)) = w[pl];
                }
            }
        }
    };
    const std::integral_constant<bool, AK> a_kone{};
    const std::integral_constant<bool, BK> b_kone{};
    // (loads behind the last chunk ask for it again: with a load on one path only, the compiler's wait for a chunk would count on none in flight)
    auto load_chunk = [&](int n, int k0) {
        const int k = min(k0, K - KC);
        load_operand(a_kone, A, lda, i0, k, ra[n]);
        load_operand(b_kone, B, ldb, j0, k, rb[n]);
    };
    auto chunk = [&](int n, int k0) {
        __syncthreads();                    // every wave has finished reading the previous chunk
        store_operand(a_kone, As, ra[n]);
        store_operand(b_kone, Bs, rb[n]);
        __syncthreads();
        load_chunk(n, k0 + AHEAD * KC);
        constexpr int STEPS = KC / 16, LOW = 7, PA[LOW] = {2, 1, 2, 0, 1, 1, 0}, PB[LOW] = {1, 2, 0, 2, 1, 0, 1};      // the partial products below x0 y0, smallest first
        v8bf a[STEPS][WT][NS_PLANES], b[STEPS][WT][NS_PLANES];
#pragma unroll
        for (int c = 0; c < STEPS; c++)
#pragma unroll
            for (int t = 0; t < WT; t++)
#pragma unroll
                for (int pl = 0; pl < NS_PLANES; pl++) {
                    a[c][t][pl] = *reinterpret_cast<const v8bf *>(As + pl * PLANE + (32 * WT * wm + 32 * t + j) * ROW + 32 * c + 16 * g);
                    b[c][t][pl] = *reinterpret_cast<const v8bf *>(Bs + pl * PLANE + (32 * WT * wn + 32 * t + j) * ROW + 32 * c + 16 * g);
                }
#pragma unroll
        for (int ta = 0; ta < WT; ta++)
#pragma unroll
            for (int tb = 0; tb < WT; tb++) {
                v16f top = {}, low = {};
#pragma unroll
                for (int c = 0; c < STEPS; c++) top = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c][ta][0], b[c][tb][0], top, 0, 0, 0);
#pragma unroll
                for (int c = 0; c < STEPS; c++)
#pragma unroll
                    for (int m = 0; m < LOW; m++) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[c][ta][PA[m]], b[c][tb][PB[m]], low, 0, 0, 0);
                acc[ta][tb] += top + low;
            }
    };
#pragma unroll
    for (int n = 0; n < AHEAD; n++) load_chunk(n, n * KC);
    int k0 = 0;
    for (; k0 + AHEAD * KC <= K; k0 += AHEAD * KC)
#pragma unroll
        for (int n = 0; n < AHEAD; n++) chunk(n, k0 + n * KC);
#pragma unroll
    for (int n = 0; n < AHEAD - 1; n++)
        if (k0 + n * KC < K) chunk(n, k0 + n * KC);
    // accumulator register r of lane (j, g) is row 8 (r / 4) + 4 g + r % 4, column j of its 32 x 32 tile
#pragma unroll
    for (int ta = 0; ta < WT; ta++)
#pragma unroll
        for (int tb = 0; tb < WT; tb++) {
            const int i1 = i0 + 32 * WT * wm + 32 * ta + 4 * g, jj = j0 + 32 * WT * wn + 32 * tb + j;
            ns_epilogue(job, acc[ta][tb], i1, jj, out + (size_t)i1 * N + jj, N);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int i = i1 + 8 * q;
                v4f v;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const size_t at = out + (size_t)(i + e) * N + jj;
                    v[e] = acc[ta][tb][4 * q + e];
                    if (!SYM || i + e <= jj) {
                        job.C[at] = v[e];
                        if (SYM && job.mode == NS_GRAM) job.C2[at] = (i + e == jj ? 1.5f : 0.0f) - 0.5f * v[e];
                    }
                }
                if (SYM) {
                    const size_t at = out + (size_t)jj * N + i;
                    if (ti < tj) {
                        *reinterpret_cast<v4f *>(job.C + at) = v;
                        if (job.mode == NS_GRAM) *reinterpret_cast<v4f *>(job.C2 + at) = -0.5f * v;
                    } else
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (i + e < jj) {
                                job.C[at + e] = v[e];
                                if (job.mode == NS_GRAM) job.C2[at + e] = -0.5f * v[e];
                            }
                }
            }
        }
}
template <int WT, bool SYM>
static hipError_t sgemm_lds(bool ak, bool bk, const SgemmJobs &jobs, int n_jobs, long lda, const float *B, long ldb, long batch_b, int M, int N, int K, int batch, hipStream_t s) {
    const int tm = M / (64 * WT), tn = N / (64 * WT);
    const dim3 grid(SYM ? tn * (tn + 1) / 2 : tm * tn, batch, n_jobs), block(EGG_THREADS);
    if (ak && bk) hipLaunchKernelGGL((k_sgemm_lds<true, true, WT, SYM>), grid, block, 0, s, jobs, lda, B, ldb, batch_b, M, N, K);
    else if (ak) hipLaunchKernelGGL((k_sgemm_lds<true, false, WT, SYM>), grid, block, 0, s, jobs, lda, B, ldb, batch_b, M, N, K);
    else if (bk) hipLaunchKernelGGL((k_sgemm_lds<false, true, WT, SYM>), grid, block, 0, s, jobs, lda, B, ldb, batch_b, M, N, K);
    else hipLaunchKernelGGL((k_sgemm_lds<false, false, WT, SYM>), grid, block, 0, s, jobs, lda, B, ldb, batch_b, M, N, K);
    return hipGetLastError();
}
static int egg_update_cu_count() {
    static int n = 0;
    if (!n) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) n = v;
        else n = 256;
    }
    return n;
}
// A(i,k) at A[i * sa_i + k * sa_k], B(k,j) at B[k * sb_k + j * sb_j]; one stride of each pair must be 1 and the other a
// multiple of 4 (16-byte loads).  sym: the result is symmetric.
static hipError_t sgemm(const SgemmJobs &jobs, int n_jobs, long sa_i, long sa_k, const float *B, long sb_k, long sb_j, long batch_b, int M, int N, int K,
                        bool sym, int batch, hipStream_t s) {
    const bool ak = sa_k == 1, bk = sb_k == 1;
    if ((!ak && sa_i != 1) || (!bk && sb_j != 1) || M % 32 || N % 32 || K % 32) return hipErrorInvalidValue;
    const long lda = ak ? sa_i : sa_k, ldb = bk ? sb_j : sb_k;
    if (lda % 4 || ldb % 4 || jobs.j[0].batch_a % 4 || batch_b % 4) return hipErrorInvalidValue;
    // The LDS-staged kernel where the shape allows it: 128 x 128 tiles when they still fill the GPU, 64 x 64 tiles otherwise
    // (bit-identical results, so the choice may depend on the batch)
    if (M % 64 == 0 && N % 64 == 0) {
        const long tiles = sym ? (long)(N / 128) * (N / 128 + 1) / 2 : (long)(M / 128) * (N / 128);
        const bool big = M % 128 == 0 && N % 128 == 0 && tiles * batch * n_jobs >= 2 * egg_update_cu_count();
        if (sym) return big ? sgemm_lds<2, true>(ak, bk, jobs, n_jobs, lda, B, ldb, batch_b, M, N, K, batch, s)
                            : sgemm_lds<1, true>(ak, bk, jobs, n_jobs, lda, B, ldb, batch_b, M, N, K, batch, s);
        return big ? sgemm_lds<2, false>(ak, bk, jobs, n_jobs, lda, B, ldb, batch_b, M, N, K, batch, s)
                   : sgemm_lds<1, false>(ak, bk, jobs, n_jobs, lda, B, ldb, batch_b, M, N, K, batch, s);
    }
    const SgemmJob &j = jobs.j[0];
    if (n_jobs != 1 || j.mode > NS_B) return hipErrorInvalidValue;
    const dim3 grid((M / 32) * (N / 32), batch), block(EGG_THREADS);
    if (ak && bk) hipLaunchKernelGGL((k_sgemm<true, true>), grid, block, 0, s, j.A, lda, j.batch_a, B, ldb, batch_b, j.C, M, N, K, j.alpha, j.mode);
    else if (ak) hipLaunchKernelGGL((k_sgemm<true, false>), grid, block, 0, s, j.A, lda, j.batch_a, B, ldb, batch_b, j.C, M, N, K, j.alpha, j.mode);
    else if (bk) hipLaunchKernelGGL((k_sgemm<false, true>), grid, block, 0, s, j.A, lda, j.batch_a, B, ldb, batch_b, j.C, M, N, K, j.alpha, j.mode);
    else hipLaunchKernelGGL((k_sgemm<false, false>), grid, block, 0, s, j.A, lda, j.batch_a, B, ldb, batch_b, j.C, M, N, K, j.alpha, j.mode);
    return hipGetLastError();
}
static SgemmJobs one_job(const float *A, long batch_a, float *C, int mode, float alpha = 1.f) { return SgemmJobs{{{A, batch_a, C, nullptr, nullptr, nullptr, mode, alpha}, {}}}; }
__global__ void k_copy_f32(float *dst, const float *src, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// `batch` matrices of rows x cols, matrix b at w.x + b * rows * cols (w.swap likewise), its 3I - G term at
// w.bterm + b * K * K (K = min(rows, cols)), its 256 norm partials at w.partials + 256 b, its norm at w.norm + b.  The result goes back to
// w.x, or stays where it is, in w.x or w.swap, and *result says where.
hipError_t egg_launch_newton_schulz_batched(const MuonWork &w, int rows, int cols, int iters, int batch, hipStream_t s, const float **result) {
    if (rows % 32 || cols % 32 || batch < 1 || batch > 65535) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(w.x) | reinterpret_cast<uintptr_t>(w.swap) | reinterpret_cast<uintptr_t>(w.bterm)) & 15) return hipErrorInvalidValue;   // 16-byte loads
    const int n = rows * cols;
    const bool use_rows = rows < cols;
    const int K = use_rows ? rows : cols;
    const long kk = (long)K * K;
    hipLaunchKernelGGL(k_sumsq_partial, dim3(256, batch), dim3(256), 0, s, w.x, n, w.partials);
    hipLaunchKernelGGL(k_norm_finish, dim3(1, batch), dim3(256), 0, s, w.partials, 256, w.norm);
    hipLaunchKernelGGL(k_scale_by_norm, dim3((n + 255) / 256, batch), dim3(256), 0, s, w.x, w.norm, n);
    float *cur = w.x, *nxt = w.swap;          // ping-pong instead of copying back after every iteration
    hipError_t e = hipSuccess;
    // The Gram form.  An iteration X <- X (3I - G) / 2 with G = X^T X changes G to G (3I - G)^2 / 4, so the factors of all
    // iterations can be multiplied up among short x short matrices and X once with their product: with k = the short side
    // and r = long / short, 3/2 r + 6 products of k^3 for five iterations where each one on X itself takes 15/2 r (counting
    // a symmetric product as half).  Used from r = 4 on, which is also where the second matrix buffer holds the four
    // k x k matrices it needs; r = 1, the other shape of the models, would gain nothing.  With the products above it is closer to the
    // exact iteration than that on X for dense matrices (512 x 2048: relative error 1.3e-7 against 2.8e-7 for random ones, 7.0e-7 against 1.4e-6 at rank
    // one) and further with the long side scaled over e^4 (3.7e-7 against 2.8e-7); but G is not computed from X again, and an eigenvalue that should be 0 grows 9/4-fold
    // an iteration, so it is kept to eight iterations.  9 matrices of 512 x 2048, 5 iterations: 0.85 -> 0.43 ms; the products of 32 of 512 x 512 (G from its upper
    // half): 0.71 -> 0.65 ms.
    if (K % 64 == 0 && iters >= 1 && iters <= 8 && (long)rows * cols >= 4 * kk) {
        float *G = w.swap, *S = w.swap + kk * batch, *next = w.swap + 2 * kk * batch;
        float *P = iters & 1 ? w.bterm : w.swap + 3 * kk * batch, *Pn = iters & 1 ? w.swap + 3 * kk * batch : w.bterm;      // the last one in bterm
        SgemmJobs gram = one_job(cur, n, G, NS_GRAM);
        gram.j[0].C2 = P;
        e = use_rows ? sgemm(gram, 1, cols, 1, cur, 1, cols, n, K, K, cols, true, batch, s)
                     : sgemm(gram, 1, 1, cols, cur, cols, 1, n, K, K, rows, true, batch, s);
        for (int it = 1; it < iters && e == hipSuccess; it++) {
            // G^2, and the factor of this iteration onto P (the first is its P as it stands)
            SgemmJobs square = one_job(G, kk, S, NS_SCALE);
            if (it > 1) {
                square.j[1] = SgemmJob{P, kk, Pn, P, nullptr, nullptr, NS_FACTOR, 0.f};
                float *t = P; P = Pn; Pn = t;
            }
            e = sgemm(square, it > 1 ? 2 : 1, K, 1, G, 1, K, kk, K, K, K, true, batch, s);
            if (e != hipSuccess) break;
            const SgemmJobs step = {{{S, kk, next, G, S, nullptr, NS_STEP, 0.f}, {}}};
            e = sgemm(step, 1, K, 1, G, 1, K, kk, K, K, K, true, batch, s);
            float *t = G; G = next; next = t;
        }
        if (e == hipSuccess && iters > 1) {
            const SgemmJobs last = {{{P, kk, Pn, P, nullptr, nullptr, NS_FACTOR, 0.f}, {}}};
            e = sgemm(last, 1, K, 1, G, 1, K, kk, K, K, K, true, batch, s);
            P = Pn;
        }
        if (e == hipSuccess && P != w.bterm) e = hipErrorUnknown;
        if (e == hipSuccess) e = use_rows ? sgemm(one_job(P, kk, nxt, NS_SCALE), 1, K, 1, cur, cols, 1, n, rows, cols, K, false, batch, s)
                                          : sgemm(one_job(cur, n, nxt, NS_SCALE), 1, cols, 1, P, 1, K, kk, rows, cols, K, false, batch, s);
        cur = nxt;
    } else
    for (int it = 0; it < iters && e == hipSuccess; it++) {
        const bool sym = K % 64 == 0;
        if (use_rows) {
            // G = X X^T (rows x rows); X <- 0.5 (3I - G) X
            e = sgemm(one_job(cur, n, w.bterm, NS_B), 1, cols, 1, cur, 1, cols, n, K, K, cols, sym, batch, s);
            if (e == hipSuccess) e = sgemm(one_job(w.bterm, kk, nxt, NS_SCALE, 0.5f), 1, K, 1, cur, cols, 1, n, rows, cols, K, false, batch, s);
        } else {
            // G = X^T X (cols x cols); X <- 0.5 X (3I - G)
            e = sgemm(one_job(cur, n, w.bterm, NS_B), 1, 1, cols, cur, cols, 1, n, K, K, rows, sym, batch, s);
            if (e == hipSuccess) e = sgemm(one_job(cur, n, nxt, NS_SCALE, 0.5f), 1, cols, 1, w.bterm, K, 1, kk, rows, cols, K, false, batch, s);
        }
        float *t = cur; cur = nxt; nxt = t;
    }
    if (e != hipSuccess) return e;
    const size_t total = (size_t)n * batch;
    if (result) { *result = cur; return hipGetLastError(); }
    if (cur != w.x) hipLaunchKernelGGL(k_copy_f32, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, w.x, cur, total);
    return hipGetLastError();
}
hipError_t egg_launch_newton_schulz(const MuonWork &w, int rows, int cols, int iters, hipStream_t s) {
    return egg_launch_newton_schulz_batched(w, rows, cols, iters, 1, s, nullptr);
}

// ---------------------------------------------------------------- Newton-Schulz for callers that cannot allocate
// The same kernels with their workspace (ping-pong matrix, 3I - G term, norm partials) in a file-scope device array
// instead of a context's hipMalloc'd buffers.  Each GPU holds its own copy of the array; its address on a device is
// looked up once per device with hipGetSymbolAddress and used from then on in place of the array's name.
struct NsScratch {
    float swap[EGG_NS_STATIC_MAX_ELEMS];
    float bterm[EGG_NS_STATIC_MAX_SHORT * EGG_NS_STATIC_MAX_SHORT];
    float partials[1024];
    float norm[4];
};
static __device__ __align__(256) unsigned char scratch[sizeof(NsScratch)];
static NsScratch *g_ns_scratch[EGG_MAX_DEVICES];      // per device; written once, under g_ns_mutex
static std::mutex g_ns_mutex;

static hipError_t ns_scratch_on_current_device(NsScratch **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= EGG_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_ns_mutex);
    if (!g_ns_scratch[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!ptr) return hipErrorInvalidSymbol;
        g_ns_scratch[dev] = static_cast<NsScratch *>(ptr);
    }
    *out = g_ns_scratch[dev];
    return hipSuccess;
}

extern "C" int egg_newton_schulz_static(float *d_X, int rows, int cols, int iters, void *hip_stream) {
    if (!d_X || (reinterpret_cast<uintptr_t>(d_X) & 15) || rows < 32 || cols < 32 || rows % 32 || cols % 32 || iters < 0 || iters > 64) {
        egg_set_thread_error("egg_newton_schulz_static: need a 16-byte aligned device matrix with rows and cols multiples of 32 and 0 <= iters <= 64");
        return EGG_E_INVALID;
    }
    if ((long long)rows * cols > EGG_NS_STATIC_MAX_ELEMS || (rows < cols ? rows : cols) > EGG_NS_STATIC_MAX_SHORT) {
        egg_set_thread_error("egg_newton_schulz_static: matrix exceeds the static workspace (rows * cols <= 1,048,576 and min(rows, cols) <= 512)");
        return EGG_E_INVALID;
    }
    NsScratch *sc = nullptr;
    hipError_t e = ns_scratch_on_current_device(&sc);
    if (e == hipSuccess) {
        // nothing in the workspace has to start at zero: every partial, the norm, the 3I - G term and the ping-pong
        // matrix are written in full before they are read
        MuonWork w = {d_X, sc->swap, nullptr, sc->bterm, sc->partials, sc->norm};
        e = egg_launch_newton_schulz(w, rows, cols, iters, static_cast<hipStream_t>(hip_stream));
    }
    if (e != hipSuccess) {
        egg_set_thread_error((std::string("egg_newton_schulz_static: ") + hipGetErrorString(e)).c_str());
        return EGG_E_HIP;
    }
    return EGG_OK;
}
