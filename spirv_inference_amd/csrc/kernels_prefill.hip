// Kernels of the decoder's prompt pass (llama.cpp, prefill): the same math as a decode step
// (export_llama.py:284-375) for up to 512 positions at once.
//
// Feeding a prompt token by token reads all 4.1 GB of TinyLlama's weights per position
// (0.76 ms each); a chunk of positions reads them once.  Up to 64 rows the products are bound by
// that read, so they have their own kernel (skinny_kernel); above, they are matrix-core bound and
// run on the tiled GEMM kernels.  TinyLlama's shape, whole prompt: 32 ids 24.3 -> 2.41 ms,
// 384 ids 291 -> 9.1 ms; 1.7 ms is the least (two token steps take 1.6).
#include "prefill.h"
#include "coherent.h"

#include <type_traits>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Eight products of a column: two matrix instructions from zero.
__device__ __forceinline__ floatx4 mfma2(float a0, float a1, float b0, float b1) {
    floatx4 c = {0.f, 0.f, 0.f, 0.f};
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, c, 0, 0, 0);
}

// ---- skinny_kernel: out = x[M][K] w[N][K]^T for M <= 16 MT rows -------------------------------
// HBM bound: 4 N K bytes of weights, each read once, so what counts is bytes in flight.  A
// workgroup of eight wavefronts takes 32 weight rows over one K range (gridDim.y of them); each
// wavefront takes an eighth of the range and loads its 16-deep steps straight into the MFMA operand
// layout, no LDS and no barrier in the loop: lane l loads 16 bytes of row l % 16 at k + 4 * (l / 16).
// The x rows are read the same way and come from L2 (256 KB at 32 rows of 2,048).  Four steps ahead
// of the products, so a wavefront has 8 KB of weights in flight and a CU about 100 (TinyLlama at 32
// rows: gate/up 43 us for 92 MB, the others 14 us; a form with x stationary in registers and 128 KB in
// flight took 34 and 19, loading x into every CU first costs the small ones more).  The sums are built
// to round no worse than the decode step's GEMV (lanes of few terms and a tree): MFMA chains of 8 k
// from zero, up to ten of them added in fp32 before their sum is (up to 16 rows, where registers are
// left, every two in fp64), and the eight wavefronts' partial tiles added in LDS as a tree.  With chains of 32 k and the wavefronts added in order the KV cache of
// 32 ids was 8.24e-7 off 64 bits where token steps are 7.11e-7 (four seeds); so it is 7.02e-7, for 1 %
// of the 32-id generation (16.77 -> 16.93 ms).
// D = w x^T puts four consecutive n of one row m in a lane: 16-byte stores, and gate and up of one
// output next to each other for the SwiGLU form.
constexpr unsigned kOob = 0x80000000u;  // past every operand range: loads return 0
constexpr int kSkWaves = 8;

template <int MT, int MODE>
__global__ __launch_bounds__(kSkWaves * 64, MT <= 2 ? 4 : 2) void skinny_kernel(
    const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N,
    int K, int kper) {
    constexpr int NT = 2, ST = 5;
    typedef typename std::conditional<MT == 1, doublex4, floatx4>::type Sum;
    __shared__ __attribute__((aligned(16))) f4v red[MT * NT][kSkWaves][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, li = lane & 15;
    const int n0 = blockIdx.x * 32;
    const int kb = blockIdx.y * kper, ke = min(K, kb + kper);
    const int steps = max(0, (ke - kb + 15) >> 4);
    const int s0 = steps * wave / kSkWaves, ns = steps * (wave + 1) / kSkWaves - s0;
    const int k0 = kb + 16 * s0 + 4 * g;
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(w, (int64_t)N * K);
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(x, (int64_t)M * K);
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
    struct Set { f4v w[NT], x[MT]; };
    Set st[ST];
    auto load = [&](int s, Set& d) __attribute__((always_inline)) {
        // K % 4 == 0, so a lane's 16 bytes lie on one side of the end; past it (also the steps
        // beyond ns) nothing is read: the vector offset is past every range, the scalar one never
        const bool in = s < ns && k0 + 16 * s < ke;
        const unsigned so = s < ns ? (unsigned)(s * 64) : 0u;
#pragma unroll
        for (int i = 0; i < NT; ++i)
            d.w[i] = __builtin_bit_cast(
                f4v, __builtin_amdgcn_raw_buffer_load_b128(wr, in ? wo[i] : kOob, so, 0));
#pragma unroll
        for (int i = 0; i < MT; ++i)
            d.x[i] = __builtin_bit_cast(
                f4v, __builtin_amdgcn_raw_buffer_load_b128(xr, in ? xo[i] : kOob, so, 0));
    };
    floatx4 acc[MT][NT];
    Sum sum[MT][NT];
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            acc[i][j] = zero;
            sum[i][j] = Sum{0, 0, 0, 0};
        }
    auto mul = [&](const Set& s, bool cut) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                acc[i][j] += mfma2(s.w[j].x, s.w[j].y, s.x[i].x, s.x[i].y) +
                             mfma2(s.w[j].z, s.w[j].w, s.x[i].z, s.x[i].w);
                if (cut || MT == 1) {
                    sum[i][j] += __builtin_convertvector(acc[i][j], Sum);
                    acc[i][j] = zero;
                }
            }
    };
#pragma unroll
    for (int u = 0; u < ST - 1; ++u) load(u, st[u]);
    int s = 0;
    for (; s + ST <= ns; s += ST) {
#pragma unroll
        for (int u = 0; u < ST; ++u) {
            load(s + u + ST - 1, st[(u + ST - 1) % ST]);
            __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
            mul(st[u], u == ST - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < ST - 1; ++u)
        if (s + u < ns) mul(st[u], false);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const floatx4 v = __builtin_convertvector(sum[i][j] + __builtin_convertvector(acc[i][j], Sum), floatx4);
            red[i * NT + j][wave][lane] = f4v{v[0], v[1], v[2], v[3]};
        }
    __syncthreads();
    const int t = wave;
    if (t >= MT * NT) return;
    f4v p[kSkWaves];
#pragma unroll
    for (int u = 0; u < kSkWaves; ++u) p[u] = red[t][u][lane];
    const f4v v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    const int m = 16 * (t / NT) + li, n = n0 + 16 * (t % NT) + 4 * g;
    if (m >= M || n >= N) return;
    if constexpr (MODE == shp::SK_SWIGLU) {
        float2 r;
        r.x = (v.x * (1.0f / (1.0f + expf(-v.x)))) * v.y;
        r.y = (v.z * (1.0f / (1.0f + expf(-v.z)))) * v.w;
        *reinterpret_cast<float2*>(out + ((int64_t)m * N + n) / 2) = r;
    } else {
        *reinterpret_cast<f4v*>(out + ((int64_t)blockIdx.y * M + m) * N + n) = v;
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
            f4v t[shp::kSkinnySplits];  // every partial in flight before the first is added
#pragma unroll
            for (int s = 0; s < shp::kSkinnySplits; ++s)
                if (s < splits) t[s] = *(reinterpret_cast<const f4v*>(part + s * sstride) + base + i);
            f4v sum = t[0];
#pragma unroll
            for (int s = 1; s < shp::kSkinnySplits; ++s)
                if (s < splits) sum += t[s];
            v += sum;
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
    float ta[shp::kSkinnySplits], tb[shp::kSkinnySplits];
#pragma unroll
    for (int s = 0; s < shp::kSkinnySplits; ++s)
        if (s < splits) {
            ta[s] = part[s * sstride + o];
            tb[s] = part[s * sstride + o + 32];
        }
    float a = ta[0], b = tb[0];
#pragma unroll
    for (int s = 1; s < shp::kSkinnySplits; ++s)
        if (s < splits) {
            a += ta[s];
            b += tb[s];
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

// Splits grow while every CU still gets at most about one workgroup and a wavefront keeps two
// steps (TinyLlama: QKV 80 row groups x 3, Wo 64 x 4, down 64 x 4; gate/up's 352 need none).
int skinny_splits(int N, int K) {
    const int groups = (N + 31) / 32, steps = (K + 15) / 16;
    int s = 1;
    while (s < kSkinnySplits && groups * (s + 1) <= 256 && steps / (s + 1) >= 2 * kSkWaves) ++s;
    return s;
}

int skinny_launch(hipStream_t st, const float* x, int M, const float* w, int N, int K, int mode,
                  int splits, float* out) {
    if (M <= 0 || M > kSkinnyRows || N <= 0 || N % 8 || K <= 0 || K % 4 || splits < 1 ||
        (mode == SK_SWIGLU && splits != 1) || (int64_t)N * K * 4 >= (1ll << 31))
        return fail(SHP_ERR_SHAPE, "skinny product: shape");
    const int kper = ((K + 15) / 16 + splits - 1) / splits * 16;
    const dim3 grid((unsigned)((N + 31) / 32), (unsigned)splits), block(kSkWaves * 64);
    const int mt = (M + 15) / 16;
    const bool sw = mode == SK_SWIGLU;
    auto kern = mt == 1   ? (sw ? skinny_kernel<1, SK_SWIGLU> : skinny_kernel<1, SK_PARTIAL>)
                : mt == 2 ? (sw ? skinny_kernel<2, SK_SWIGLU> : skinny_kernel<2, SK_PARTIAL>)
                : mt == 3 ? (sw ? skinny_kernel<3, SK_SWIGLU> : skinny_kernel<3, SK_PARTIAL>)
                          : (sw ? skinny_kernel<4, SK_SWIGLU> : skinny_kernel<4, SK_PARTIAL>);
    hipLaunchKernelGGL(kern, grid, block, 0, st, x, w, out, M, N, K, kper);
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
