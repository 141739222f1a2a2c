// Kernels of the decoder's prompt pass (llama.cpp, prefill): the same math as a decode step
// (export_llama.py:284-375) for up to 512 positions at once.
//
// Feeding a prompt token by token reads all 4.1 GB of TinyLlama's weights per position
// (0.76 ms each); a chunk of positions reads them once.  Up to 64 rows the products are bound by
// that read, so they have their own kernel (skinny_kernel); above, they are matrix-core bound and
// run on the tiled GEMM kernels.  TinyLlama's shape, whole prompt: 32 ids 24.3 -> 2.45 ms,
// 384 ids 291 -> 8.6 ms; 1.8 ms is the least (2 ids, two token steps took 1.5).
#include "prefill.h"
#include "coherent.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

__device__ __forceinline__ floatx4 mfma4(f4v a, f4v b, floatx4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

// ---- skinny_kernel: out = x[M][K] w[N][K]^T for M <= 16 MT rows -------------------------------
// HBM bound: 4 N K bytes of weights, each read once.  A workgroup of four wavefronts takes 32
// weight rows over one K range; the wavefronts take 128-byte pieces of the rows in turn (so a
// workgroup reads 512 contiguous bytes of each row per step) straight into the MFMA operand
// layout, no LDS and no barrier in the loop: lane l loads 16 bytes of row l % 16, k + 4 * (l / 16).
// The x rows are read the same way and come from L2 (256 KB at 32 rows of 2,048).  Two register
// sets alternate, so a wavefront has up to 8 KB of weights in flight.  The MFMA chains are cut
// every 64 k and added to a second accumulator: the sum's rounding error is then that of the
// decode step's GEMV (lanes of ~32 terms and a tree), where one chain over K had 1.6 times it.
// The four partial tiles are summed in LDS in wavefront order.  D = w x^T puts four consecutive n of one row m in a lane:
// 16-byte stores, and gate and up of one output next to each other for the SwiGLU form.
constexpr unsigned kOob = 0x80000000u;  // past every operand range: loads return 0

template <int MT, int MODE>
__global__ __launch_bounds__(256) void skinny_kernel(const float* __restrict__ x,
                                                     const float* __restrict__ w,
                                                     float* __restrict__ out, int M, int N, int K,
                                                     int kper) {
    constexpr int NT = 2, WV = 4, STEP = 32 * WV;
    __shared__ __attribute__((aligned(16))) f4v red[MT * NT][WV][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, li = lane & 15;
    const int n0 = blockIdx.x * 32;
    const int kb = blockIdx.y * kper, ke = min(K, kb + kper);
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(w, (int64_t)N * K);
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(x, (int64_t)M * K);
    const int k0 = kb + wave * 32 + 4 * g;
    unsigned wo[NT], xo[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int n = n0 + 16 * i + li;
        wo[i] = n < N ? (unsigned)(((int64_t)n * K + k0) * 4) : kOob;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = 16 * i + li;
        xo[i] = m < M ? (unsigned)(((int64_t)m * K + k0) * 4) : kOob;
    }
    struct Set { f4v w[2][NT], x[2][MT]; };
    auto load = [&](int it, Set& s) __attribute__((always_inline)) {
        const unsigned so = (unsigned)(it * STEP * 4);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const bool in = k0 + it * STEP + 16 * u < ke;
#pragma unroll
            for (int i = 0; i < NT; ++i)
                s.w[u][i] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(
                    wr, in ? wo[i] + 64u * u : kOob, so, 0));
#pragma unroll
            for (int i = 0; i < MT; ++i)
                s.x[u][i] = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(
                    xr, in ? xo[i] + 64u * u : kOob, so, 0));
        }
    };
    floatx4 acc[MT][NT], sum[MT][NT];
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = sum[i][j] = zero;
    auto flush = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                sum[i][j] += acc[i][j];
                acc[i][j] = zero;
            }
    };
    auto mul = [&](const Set& s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = mfma4(s.w[u][j], s.x[u][i], acc[i][j]);
    };
    const int nit = (ke - kb + STEP - 1) / STEP;
    Set a, b;
    load(0, a);
    int it = 0;
    for (; it + 1 < nit; it += 2) {
        load(it + 1, b);
        mul(a);
        if (it + 2 < nit) load(it + 2, a);
        mul(b);
        flush();
    }
    if (it < nit) {
        mul(a);
        flush();
    }

#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            red[i * NT + j][wave][lane] = f4v{sum[i][j][0], sum[i][j][1], sum[i][j][2], sum[i][j][3]};
    __syncthreads();
    for (int t = wave; t < MT * NT; t += WV) {
        f4v v = red[t][0][lane];
#pragma unroll
        for (int u = 1; u < WV; ++u) v += red[t][u][lane];
        const int m = 16 * (t / NT) + li, n = n0 + 16 * (t % NT) + 4 * g;
        if (m >= M || n >= N) continue;
        if constexpr (MODE == shp::SK_SWIGLU) {
            float2 r;
            r.x = (v.x * (1.0f / (1.0f + expf(-v.x)))) * v.y;
            r.y = (v.z * (1.0f / (1.0f + expf(-v.z)))) * v.w;
            *reinterpret_cast<float2*>(out + ((int64_t)m * N + n) / 2) = r;
        } else {
            *reinterpret_cast<f4v*>(out + ((int64_t)blockIdx.y * M + m) * N + n) = v;
        }
    }
}

__global__ __launch_bounds__(256) void prefill_embed_kernel(const float* __restrict__ embed,
                                                            int h4, shp::PrefillIds ids,
                                                            float* __restrict__ x) {
    const f4v* row = reinterpret_cast<const f4v*>(embed) + (int64_t)ids.id[blockIdx.x] * h4;
    f4v* o = reinterpret_cast<f4v*>(x) + (int64_t)blockIdx.x * h4;
    for (int i = threadIdx.x; i < h4; i += 256) o[i] = row[i];
}

// One workgroup per row (xout may be x); the partials of the product before (Wo or down) are added here, in
// split order, so that product needs no pass of its own to sum them.
__global__ __launch_bounds__(256) void prefill_norm_kernel(const float* x,
                                                           const float* __restrict__ part,
                                                           int splits, int64_t sstride,
                                                           float* xout,
                                                           const float* __restrict__ w, float eps,
                                                           float* __restrict__ h, int h4) {
    __shared__ float red[4];
    const int64_t base = (int64_t)blockIdx.x * h4;
    const f4v* xr = reinterpret_cast<const f4v*>(x) + base;
    f4v* xo = reinterpret_cast<f4v*>(xout) + base;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < h4; i += 256) {
        f4v v = xr[i];
        if (splits) {
            f4v t = {0.f, 0.f, 0.f, 0.f};
            for (int s = 0; s < splits; ++s)
                t += *(reinterpret_cast<const f4v*>(part + s * sstride) + base + i);
            v += t;
            xo[i] = v;
        }
        ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)(h4 * 4) + eps);
    const f4v* src = splits ? xo : xr;  // a thread re-reads what it stored
    const f4v* wv = reinterpret_cast<const f4v*>(w);
    f4v* ho = reinterpret_cast<f4v*>(h) + base;
    for (int i = threadIdx.x; i < h4; i += 256) ho[i] = (src[i] * inv) * wv[i];
}

// One workgroup per row and head block: thread = one (head, j < 32) pair of rotated columns.
__global__ __launch_bounds__(256) void prefill_rope_kernel(const float* __restrict__ part,
                                                           int splits, int64_t sstride,
                                                           float* __restrict__ q,
                                                           float* __restrict__ kc,
                                                           float* __restrict__ vc, int n_heads,
                                                           int n_kv, int max_seq, int pos0,
                                                           float theta) {
    const int row = blockIdx.x, heads = n_heads + 2 * n_kv;
    const int e = blockIdx.y * 256 + threadIdx.x, hd = e >> 5, j = e & 31;
    if (hd >= heads) return;
    const int64_t o = (int64_t)row * heads * 64 + hd * 64 + j;
    float a = 0.0f, b = 0.0f;
    for (int s = 0; s < splits; ++s) {
        a += part[s * sstride + o];
        b += part[s * sstride + o + 32];
    }
    const int pos = pos0 + row;
    if (hd >= n_heads + n_kv) {
        float* d = vc + ((int64_t)(hd - n_heads - n_kv) * max_seq + pos) * 64 + j;
        d[0] = a;
        d[32] = b;
        return;
    }
    // RoPE (rotate-half): x * cos + rotate_half(x) * sin, angle = pos * theta^(-2j/64)
    const float inv_freq = 1.0f / powf(theta, (float)(2 * j) / 64.0f);
    const float ang = (float)pos * inv_freq;
    const float c = cosf(ang), s = sinf(ang);
    const float ra = a * c + -b * s, rb = b * c + a * s;
    float* d = hd < n_heads ? q + ((int64_t)row * n_heads + hd) * 64 + j
                            : kc + ((int64_t)(hd - n_heads) * max_seq + pos) * 64 + j;
    d[0] = ra;
    d[32] = rb;
}

__global__ __launch_bounds__(256) void prefill_swiglu_kernel(const f4v* __restrict__ gu,
                                                             float2* __restrict__ act,
                                                             int64_t n2) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n2;
         i += (int64_t)gridDim.x * 256) {
        const f4v v = gu[i];
        float2 r;
        r.x = (v.x * (1.0f / (1.0f + expf(-v.x)))) * v.y;
        r.y = (v.z * (1.0f / (1.0f + expf(-v.z)))) * v.w;
        act[i] = r;
    }
}

__global__ __launch_bounds__(1024) void prefill_argmax_kernel(const float* __restrict__ logits,
                                                              int vocab, int32_t* log,
                                                              float* last_logits, int32_t* token,
                                                              int32_t* pos, int32_t* step,
                                                              int new_pos) {
    __shared__ float bv[16];
    __shared__ int bi[16];
    const float* x = logits + (int64_t)blockIdx.x * vocab;
    const bool last = last_logits && blockIdx.x == gridDim.x - 1;
    float best = -3.4028234663852886e+38f;
    int idx = 0x7fffffff;
    for (int i = threadIdx.x; i < vocab; i += 1024) {
        const float v = x[i];
        if (v > best) { best = v; idx = i; }
        if (last) last_logits[i] = v;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(best, o);
        const int oi = __shfl_xor(idx, o);
        if (ov > best || (ov == best && oi < idx)) { best = ov; idx = oi; }
    }
    if ((threadIdx.x & 63) == 0) { bv[threadIdx.x >> 6] = best; bi[threadIdx.x >> 6] = idx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w)
            if (bv[w] > best || (bv[w] == best && bi[w] < idx)) { best = bv[w]; idx = bi[w]; }
        if (idx == 0x7fffffff) idx = 0;
        log[blockIdx.x] = idx;
        if (last) {
            *token = idx;
            *pos = new_pos;
            *step = new_pos;
        }
    }
}

}  // namespace

namespace shp {

int skinny_splits(int N, int K) {
    // Enough workgroups for two or three per CU (each holds up to 32 KB of weights in flight),
    // but at least one 128-deep step per wavefront set.
    const int groups = (N + 31) / 32, steps = (K + 127) / 128;
    int s = 1;
    while (s < kSkinnySplits && groups * s < 512 && s * 2 <= steps) s *= 2;
    return s;
}

int skinny_launch(hipStream_t st, const float* x, int M, const float* w, int N, int K, int mode,
                  int splits, float* out) {
    if (M <= 0 || M > kSkinnyRows || N <= 0 || N % 8 || K <= 0 || K % 4 || splits < 1 ||
        (mode == SK_SWIGLU && splits != 1) || (int64_t)N * K * 4 >= (1ll << 31))
        return fail(SHP_ERR_SHAPE, "skinny product: shape");
    const int kper = (((K + splits - 1) / splits) + 127) / 128 * 128;
    const dim3 grid((unsigned)((N + 31) / 32), (unsigned)splits);
    const int mt = (M + 15) / 16;
#define SHP_SKINNY(MT)                                                                        \
    if (mode == SK_SWIGLU)                                                                    \
        hipLaunchKernelGGL((skinny_kernel<MT, SK_SWIGLU>), grid, dim3(256), 0, st, x, w, out, \
                           M, N, K, kper);                                                    \
    else                                                                                      \
        hipLaunchKernelGGL((skinny_kernel<MT, SK_PARTIAL>), grid, dim3(256), 0, st, x, w, out, \
                           M, N, K, kper);
    if (mt == 1) { SHP_SKINNY(1) }
    else if (mt == 2) { SHP_SKINNY(2) }
    else if (mt == 3) { SHP_SKINNY(3) }
    else { SHP_SKINNY(4) }
#undef SHP_SKINNY
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

int prefill_embed_launch(hipStream_t s, const float* embed, int hidden, const PrefillIds& ids,
                         int rows, float* x) {
    hipLaunchKernelGGL(prefill_embed_kernel, dim3(rows), dim3(256), 0, s, embed, hidden / 4, ids, x);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

int prefill_norm_launch(hipStream_t s, const float* x, const float* part, int splits, float* xout,
                        const float* w, float eps, float* h, int rows, int hidden) {
    hipLaunchKernelGGL(prefill_norm_kernel, dim3(rows), dim3(256), 0, s, x, part, splits,
                       (int64_t)rows * hidden, xout, w, eps, h, hidden / 4);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

int prefill_rope_launch(hipStream_t s, const float* part, int splits, float* q, float* k_cache,
                        float* v_cache, int rows, int n_heads, int n_kv, int max_seq, int pos0,
                        float theta) {
    const int heads = n_heads + 2 * n_kv;
    hipLaunchKernelGGL(prefill_rope_kernel, dim3(rows, (heads * 32 + 255) / 256), dim3(256), 0, s,
                       part, splits, (int64_t)rows * heads * 64, q, k_cache, v_cache, n_heads,
                       n_kv, max_seq, pos0, theta);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

int prefill_swiglu_launch(hipStream_t s, const float* gu, float* act, int rows, int ffn) {
    const int64_t n2 = (int64_t)rows * ffn / 2;
    const unsigned g = (unsigned)std::min<int64_t>((n2 + 255) / 256, 8192);
    hipLaunchKernelGGL(prefill_swiglu_kernel, dim3(g), dim3(256), 0, s,
                       reinterpret_cast<const f4v*>(gu), reinterpret_cast<float2*>(act), n2);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

int prefill_argmax_launch(hipStream_t s, const float* logits, int rows, int vocab, int32_t* log,
                          float* last_logits, int32_t* token, int32_t* pos, int32_t* step,
                          int new_pos) {
    hipLaunchKernelGGL(prefill_argmax_kernel, dim3(rows), dim3(1024), 0, s, logits, vocab, log,
                       last_logits, token, pos, step, new_pos);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

}  // namespace shp
