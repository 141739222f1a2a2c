// Attention of a block of queries over any number of keys, head dim 64, on the fp32 matrix
// cores: one launch instead of scores product, row softmax and context product, so neither the
// scores nor the probabilities reach memory (they are 4 * heads * n * n bytes each).
//
// Latency and the MFMA chain bound it at the sequence lengths of the encoder and of a decoder's
// prompt (16-512).  A wavefront owns 16 queries of one head and walks the keys in tiles of 64 that
// the workgroup stages in LDS (rows padded by 4 floats); the next tile's rows load into registers
// while this one is multiplied.  The scores are computed transposed, S^T = K Q^T, with
// v_mfma_f32_16x16x4_f32: lane l then holds query l % 16 and keys 16j + 4 * (l / 16) + r, which is
// already the B operand of O^T = V^T P^T (the four k slots of step r are keys 4g + r of group g on
// both sides), so P never goes through LDS, a row's maximum and sum are two lane exchanges away,
// and the running rescale of a query is one factor per lane.  Four consecutive output columns
// land in one lane, so stores are 16 bytes wide.
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

constexpr int kKeys = 64;       // keys per tile
constexpr int kRs = 64 + 4;     // LDS row stride

__device__ __forceinline__ floatx4 mfma4(f4v a, f4v b, floatx4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

// NW wavefronts per workgroup; grid (ceil(units / NW), kv_heads, batch) where a unit is one
// 16-query block of one query head, the heads of a block next to each other (so a workgroup's
// wavefronts share the KV head and, under the causal mask, nearly the same key range).
template <int NW>
__global__ __launch_bounds__(NW * 64) void attention_kernel(AttnArgs a) {
    __shared__ __attribute__((aligned(16))) float Ks[kKeys * kRs];
    __shared__ __attribute__((aligned(16))) float Vs[kKeys * kRs];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, li = lane & 15;
    const int qblocks = (a.n_queries + 15) >> 4;
    const int units = qblocks * a.group;
    const int unit = min((int)blockIdx.x * NW + wave, units - 1);
    const bool live = (int)blockIdx.x * NW + wave < units;
    const int qb = unit / a.group, hg = unit - qb * a.group;
    const int kv = blockIdx.y, h = kv * a.group + hg, b = blockIdx.z;
    const int query = qb * 16 + li;
    const float* kp = a.k + b * a.k_b + kv * a.k_h;
    const float* vp = a.v + b * a.v_b + kv * a.v_h;

    // keys this workgroup walks: all, or up to the last one its last query block sees
    int nk = a.n_keys;
    if (a.causal) {
        const int last = min((int)blockIdx.x * NW + NW, units) - 1;
        nk = min(nk, a.pos0 + (last / a.group) * 16 + 16);
    }
    const int limit = a.causal ? min(a.n_keys, a.pos0 + query + 1) : a.n_keys;  // keys < limit
    const int ntiles = (nk + kKeys - 1) / kKeys;

    f4v qf[4];
    {
        const float* qp = a.q + b * a.q_b + h * a.q_h + (int64_t)min(query, a.n_queries - 1) * a.q_r;
#pragma unroll
        for (int s = 0; s < 4; ++s) qf[s] = *reinterpret_cast<const f4v*>(qp + 16 * s + 4 * g);
    }
    // staging: 64 rows x 16 float4 of K and of V, NST of each per thread
    constexpr int NST = kKeys * 16 / (NW * 64);
    f4v ks[NST], vs[NST];
    auto load = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int e = i * NW * 64 + tid, row = e >> 4, d = (e & 15) * 4;
            const int64_t key = min(t * kKeys + row, a.n_keys - 1);
            ks[i] = *reinterpret_cast<const f4v*>(kp + key * a.k_r + d);
            vs[i] = *reinterpret_cast<const f4v*>(vp + key * a.v_r + d);
        }
    };
    load(0);

    constexpr float kLowest = -3.4028234663852886e+38f;
    float m = kLowest, l = 0.0f;
    floatx4 o[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};

    for (int t = 0; t < ntiles; ++t) {
        __syncthreads();  // every wavefront has read the previous tile
#pragma unroll
        for (int i = 0; i < NST; ++i) {
            const int e = i * NW * 64 + tid, row = e >> 4, d = (e & 15) * 4;
            *reinterpret_cast<f4v*>(&Ks[row * kRs + d]) = ks[i];
            *reinterpret_cast<f4v*>(&Vs[row * kRs + d]) = vs[i];
        }
        __syncthreads();
        if (t + 1 < ntiles) load(t + 1);

        floatx4 s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const f4v kf = *reinterpret_cast<const f4v*>(&Ks[(16 * j + li) * kRs + 16 * c + 4 * g]);
                s[j] = mfma4(kf, qf[c], s[j]);
            }
        }
        // s[j][r]: key t * 64 + 16 j + 4 g + r, query li
        float mx = m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = t * kKeys + 16 * j + 4 * g + r;
                float v = s[j][r] * a.scale;
                if (a.mask) v += a.mask[min(key, a.n_keys - 1)];
                s[j][r] = key < limit ? v : -__builtin_inff();
                mx = fmaxf(mx, s[j][r]);
            }
        }
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
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float* vr = &Vs[(16 * j + 4 * g + r) * kRs + li];
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[16 * d], s[j][r], o[d], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (live && query < a.n_queries) {
        const float inv = 1.0f / l;
        float* op = a.out + b * a.o_b + h * a.o_h + (int64_t)query * a.o_r;
#pragma unroll
        for (int d = 0; d < 4; ++d)
            *reinterpret_cast<f4v*>(op + 16 * d + 4 * g) =
                f4v{o[d][0] * inv, o[d][1] * inv, o[d][2] * inv, o[d][3] * inv};
    }
}

}  // namespace

namespace shp {

int attention_launch(hipStream_t s, const AttnArgs& a) {
    if (a.batch <= 0 || a.kv_heads <= 0 || a.group <= 0 || a.n_queries <= 0 || a.n_keys <= 0 ||
        a.batch > 65535 || a.kv_heads > 65535 || a.pos0 < 0)
        return fail(SHP_ERR_SHAPE, "attention: dims");
    const int64_t units = (int64_t)((a.n_queries + 15) / 16) * a.group;
    if (units > (1 << 30)) return fail(SHP_ERR_SHAPE, "attention: too many queries");
    // Two wavefronts share a staged tile where four would leave fewer workgroups than CUs.
    const int64_t wgs4 = (units + 3) / 4 * a.kv_heads * a.batch;
    if (wgs4 >= 256)
        hipLaunchKernelGGL((attention_kernel<4>), dim3((unsigned)((units + 3) / 4), a.kv_heads, a.batch),
                           dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((attention_kernel<2>), dim3((unsigned)((units + 1) / 2), a.kv_heads, a.batch),
                           dim3(128), 0, s, a);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

}  // namespace shp
