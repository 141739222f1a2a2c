// Attention of a block of queries over any number of keys, head dim 64, on the fp32 matrix
// cores: one launch instead of scores product, row softmax and context product, so neither the
// scores nor the probabilities reach memory (they are 4 * heads * n * n bytes each).
//
// Latency and the MFMA chain bound it at the sequence lengths of the encoder and of a decoder's
// prompt (16-512).  Two wavefronts own 16 queries of one head; the workgroup stages the keys in LDS
// 128 at a time (rows padded by 4 floats) and each wavefront of the pair takes 64 of them, so a long
// row's serial chain is halved, and the pair's results meet in LDS at the end.  The next keys load into
// registers while these are multiplied.  The scores are computed transposed, S^T = K Q^T, with
// v_mfma_f32_16x16x4_f32: lane l then holds query l % 16 and keys 16j + 4 * (l / 16) + r, which is
// already the B operand of O^T = V^T P^T (the four k slots of step r are keys 4g + r of group g on
// both sides), so P never goes through LDS, a row's maximum and sum are two lane exchanges away,
// and the running rescale of a query is one factor per lane.  Four consecutive output columns
// land in one lane, so stores are 16 bytes wide.
//
// Measured (MI355X, graph-replayed): 96 heads x 128 queries 14.1 -> 10.6 us against a kernel that
// staged a whole head's K and V and sent P through LDS, 36 x 200 27 (three operators) -> 11.7 us; a
// causal prompt of 384 (32 heads on 4 KV heads) 23 us in the kernel trace.
//
// The arithmetic is the three-operator chain's apart from the order of the sums: the maximum
// starts at the lowest finite float, a row whose every key is masked with that value is uniform,
// and with minus infinity it is NaN, as in softmax_rows.  Under the causal mask a hidden key's
// weight is an exact 0, so a non-finite V row still reaches earlier queries of its 64-key tile as
// 0 * inf, as it does in the reference's masked recompute of every position.
#include "attention.h"
#include "coherent.h"

namespace {

using shp::AttnArgs;
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kKeys = 64;       // keys per wavefront and tile
constexpr int kRs = 64 + 4;     // LDS row stride

__device__ __forceinline__ floatx4 mfma4(f4v a, f4v b, floatx4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

// c plus 16 products, with SHORT as a chain of their own: the prompt's sums must not round worse than
// the token steps', which add by lanes of few terms (the KV cache of 32 ids 7.40e-7 off 64 bits with
// chains over a whole row, 7.02e-7 so, 7.11e-7 by token steps; 384 ids 22.7 -> 23.4 us a layer).  The
// encoder's products were chains of 64 before too, and the additions cost it 0.7 %.
template <bool SHORT>
__device__ __forceinline__ floatx4 mfma_add(f4v a, f4v b, floatx4 c) {
    if constexpr (SHORT) return c + mfma4(a, b, floatx4{0.f, 0.f, 0.f, 0.f});
    else return mfma4(a, b, c);
}

// U query units per workgroup, two wavefronts each; grid batch x kv_heads x wgs, the last fastest,
// wgs = ceil(units / U), where a unit is one 16-query block of one query head, the heads of a block next to each other (so a
// workgroup's units share the KV head and, under the causal mask, nearly the same key range).  The
// units with the longest causal rows come first.
template <int U, bool CAUSAL, bool MASK>
__global__ __launch_bounds__(U * 128) void attention_kernel(AttnArgs a, int wgs, int vec_out) {
    constexpr int T = U * 128;
    __shared__ __attribute__((aligned(16))) float Ks[2 * kKeys * kRs];
    __shared__ __attribute__((aligned(16))) float Vs[2 * kKeys * kRs];
    __shared__ __attribute__((aligned(16))) float Ms[MASK ? 2 * kKeys : 4];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, li = lane & 15;
    const int half = wave & 1, us = wave >> 1;
    const int qblocks = (a.n_queries + 15) >> 4;
    const int units = qblocks * a.group;
    const int bk = blockIdx.x / wgs, wx = blockIdx.x - bk * wgs;
    const int wg = CAUSAL ? wgs - 1 - wx : wx;
    const bool live = wg * U + us < units;
    const int unit = live ? wg * U + us : units - 1;
    const int qb = unit / a.group, hg = unit - qb * a.group;
    const int b = bk / a.kv_heads, kv = bk - b * a.kv_heads, h = kv * a.group + hg;
    const int query = qb * 16 + li;
    const float* kp = a.k + b * a.k_b + kv * a.k_h;
    const float* vp = a.v + b * a.v_b + kv * a.v_h;

    // keys this workgroup walks: all, or up to the last one its last query block sees
    int nk = a.n_keys;
    if constexpr (CAUSAL) {
        const int last = min(wg * U + U, units) - 1;
        nk = min(nk, a.pos0 + (last / a.group) * 16 + 16);
    }
    const int limit = CAUSAL ? min(a.n_keys, a.pos0 + query + 1) : a.n_keys;   // keys < limit
    const int open = CAUSAL ? min(a.n_keys, a.pos0 + qb * 16 + 1) : a.n_keys;  // seen by every query
    const int ntiles = (nk + 2 * kKeys - 1) / (2 * kKeys);

    f4v qf[4];
    {
        const float* qp = a.q + b * a.q_b + h * a.q_h + (int64_t)min(query, a.n_queries - 1) * a.q_r;
#pragma unroll
        for (int s = 0; s < 4; ++s) qf[s] = *reinterpret_cast<const f4v*>(qp + 16 * s + 4 * g);
    }
    // staging: 128 rows x 16 float4 of K and of V, NST of each per thread
    constexpr int NST = 2 * kKeys * 16 / T;
    f4v ks[NST], vs[NST];
    float ms = 0.0f;
    auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int e = i * T + tid, row = e >> 4, d = (e & 15) * 4;
            const int64_t key = min(t * 2 * kKeys + row, a.n_keys - 1);
            ks[i] = *reinterpret_cast<const f4v*>(kp + key * a.k_r + d);
            vs[i] = *reinterpret_cast<const f4v*>(vp + key * a.v_r + d);
        }
        if constexpr (MASK)
            if (tid < 2 * kKeys) ms = a.mask[min(t * 2 * kKeys + tid, a.n_keys - 1)];
    };
    load(0);

    constexpr float kLowest = -3.4028234663852886e+38f;
    float m = kLowest, l = 0.0f;
    floatx4 o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};

    const float* const Kh = Ks + half * kKeys * kRs;
    const float* const Vh = Vs + half * kKeys * kRs;
    for (int t = 0; t < ntiles; ++t) {
        __syncthreads();  // every wavefront has read the previous tile
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int e = i * T + tid, row = e >> 4, d = (e & 15) * 4;
            *reinterpret_cast<f4v*>(&Ks[row * kRs + d]) = ks[i];
            // past the last key the weight is 0, which must not meet the last row's infinity
            *reinterpret_cast<f4v*>(&Vs[row * kRs + d]) =
                t * 2 * kKeys + row < a.n_keys ? vs[i] : f4v{0.f, 0.f, 0.f, 0.f};
        }
        if constexpr (MASK)
            if (tid < 2 * kKeys) Ms[tid] = ms;
        __syncthreads();
        if (t + 1 < ntiles) load(t + 1);
        const int key0 = (2 * t + half) * kKeys;  // this wavefront's first key
        if (key0 >= nk) continue;                 // uniform; the last tile's second half

        floatx4 s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            f4v kf[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                kf[j] = *reinterpret_cast<const f4v*>(&Kh[(16 * j + li) * kRs + 16 * c + 4 * g]);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = mfma_add<CAUSAL>(kf[j], qf[c], s[j]);
        }
        // s[j][r]: key key0 + 16 j + 4 g + r, query li
        float mx = m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] *= a.scale;
            if constexpr (MASK) {
                const f4v mv = *reinterpret_cast<const f4v*>(&Ms[half * kKeys + 16 * j + 4 * g]);
                s[j] += floatx4{mv.x, mv.y, mv.z, mv.w};
            }
        }
        if (key0 + kKeys > open) {  // uniform: some key is hidden from some query
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    s[j][r] = key0 + 16 * j + 4 * g + r < limit ? s[j][r] : -__builtin_inff();
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[j][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float alpha = expf(m - mx);
        m = mx;
        float ps = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[j][r] = expf(s[j][r] - mx);
                ps += s[j][r];
            }
        }
        l = l * alpha + ps;  // this lane's keys; the groups are added at the end
#pragma unroll
        for (int d = 0; d < 4; ++d) o[d] *= alpha;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float vf[4][4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int d = 0; d < 4; ++d) vf[r][d] = Vh[(16 * j + 4 * g + r) * kRs + 16 * d + li];
#pragma unroll
            for (int d = 0; d < 4; ++d)
                o[d] = mfma_add<CAUSAL>(f4v{vf[0][d], vf[1][d], vf[2][d], vf[3][d]},
                                        f4v{s[j][0], s[j][1], s[j][2], s[j][3]}, o[d]);
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);

    // the second half's maximum, sum and output, through the keys' LDS
    __syncthreads();
    float* ex = Ks + us * (64 * 16);  // [16 float4 slots of d and lane]
    float2* es = reinterpret_cast<float2*>(Vs) + us * 64;
    if (half) {
#pragma unroll
        for (int d = 0; d < 4; ++d)
            *reinterpret_cast<f4v*>(&ex[(d * 64 + lane) * 4]) = f4v{o[d][0], o[d][1], o[d][2], o[d][3]};
        es[lane] = make_float2(m, l);
    }
    __syncthreads();
    if (half || !live || query >= a.n_queries) return;
    const float2 e = es[lane];
    const float mm = fmaxf(m, e.x), f0 = expf(m - mm), f1 = expf(e.x - mm);
    const float inv = 1.0f / (l * f0 + e.y * f1);
    float* op = a.out + b * a.o_b + h * a.o_h + (int64_t)query * a.o_r;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const f4v p = *reinterpret_cast<const f4v*>(&ex[(d * 64 + lane) * 4]);
        f4v r;
#pragma unroll
        for (int c = 0; c < 4; ++c) r[c] = (o[d][c] * f0 + p[c] * f1) * inv;
        float* q = op + 16 * d + 4 * g;
        if (vec_out) {
            *reinterpret_cast<f4v*>(q) = r;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) q[c] = r[c];
        }
    }
}

}  // namespace

namespace shp {

int attention_launch(hipStream_t s, const AttnArgs& a) {
    if (a.batch <= 0 || a.kv_heads <= 0 || a.group <= 0 || a.n_queries <= 0 || a.n_keys <= 0 ||
        a.pos0 < 0)
        return fail(SHP_ERR_SHAPE, "attention: dims");
    const int64_t units = (int64_t)((a.n_queries + 15) / 16) * a.group;
    if (units > (1 << 30)) return fail(SHP_ERR_SHAPE, "attention: too many queries");
    if (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v) & 15 ||
        (a.q_b | a.q_h | a.q_r | a.k_b | a.k_h | a.k_r | a.v_b | a.v_h | a.v_r) & 3)
        return fail(SHP_ERR_SHAPE, "attention: Q/K/V rows must be 16-byte aligned");
    const int vec = ((uintptr_t)a.out & 15) == 0 && ((a.o_b | a.o_h | a.o_r) & 3) == 0;
    // Four units share a staged tile; two where that would leave most CUs without a workgroup.
    const int u = (units + 3) / 4 * a.kv_heads * a.batch >= 192 ? 4 : 2;
    const int64_t wgs = (units + u - 1) / u, grid = wgs * a.kv_heads * a.batch;
    if (grid > 0x7fffffff) return fail(SHP_ERR_SHAPE, "attention: grid");
    auto kern = u == 4 ? (a.causal ? attention_kernel<4, true, false>
                                   : a.mask ? attention_kernel<4, false, true> : attention_kernel<4, false, false>)
                       : (a.causal ? attention_kernel<2, true, false>
                                   : a.mask ? attention_kernel<2, false, true> : attention_kernel<2, false, false>);
    if (a.causal && a.mask) return fail(SHP_ERR_UNSUPPORTED, "attention: causal with a mask");
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(u * 128), 0, s, a, (int)wgs, vec);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

}  // namespace shp
