// Products and convolutions too small to fill the GPU with 64x64 tiles (gemm_direct_kernel).
//
// What bounds them is not the matrix rate but the length of the serial chain: with less than a
// 64x64 tile per CU the tiled kernels run one workgroup per CU or fewer, whose four wavefronts
// step through K together, two LDS barriers per K tile, with two tiles of loads in flight.  Here
// a workgroup owns a 32x64 tile and its eight wavefronts split the tile's K between them: each
// multiplies its own K range for the whole tile on v_mfma_f32_16x16x4_f32, its operands loaded from
// global memory (the XCD's L2, mostly) straight into the MFMA layout, two to three 16-deep steps
// ahead.  No LDS and no barrier until the eight partial tiles are summed in LDS, in wavefront
// order.  K can be split over workgroups too; the last arrival of a tile sums the partials in split
// order, as in the other kernels.  A lane of a 16-deep step loads 16 bytes of one A row (k + 4 *
// (l / 16)) and, from a [K][N] operand, 16 bytes of four k rows, so the four products of a column
// block give it four consecutive columns and its stores are 16 bytes wide.
//
// Measured (MI355X, operands in L2, against the tiled kernels' best plan): 98x512x4608 15.6 -> 10.7
// us, 980x256x2304 23.0 -> 15.2, 600x768x3072 35.4 -> 32.4; from one 64x64 tile per CU and long K
// on the tiled kernels win (1568x512x4608: 69 against 71), since eight tile-wide operand reads per
// CU cost more L2 traffic than one shared LDS tile.
#include "gemm.h"
#include "coherent.h"

namespace {

using shp::GemmParams;
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr unsigned kOob = 0x80000000u;  // past every operand range: loads return 0
constexpr int kTm = 32, kTn = 64, kWaves = 8, kStages = 3, kMaxSplits = 8;
constexpr int kFm = kTm / 16, kFn = kTn / 16;

__device__ __forceinline__ f4v load4(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
    return __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// AM: A_KVEC rows or A_CONV_NHWC4 with IC % 16 == 0; BMD: B_NVEC ([K][N]) or B_KVEC ([N][K]).
// K % 16 == 0.  Grid (tiles, splits).
template <int AM, int BMD>
__global__ __launch_bounds__(kWaves * 64, 4) void gemm_direct_kernel(GemmParams p, int tiles_m,
                                                                  int tiles_n) {
    constexpr bool CONV = AM == shp::A_CONV_NHWC4, BT = BMD == shp::B_KVEC;
    constexpr int IDX = kFm * kFn;  // 16-byte results of a lane
    __shared__ __attribute__((aligned(16))) f4v red[kWaves * IDX * 64];
    __shared__ int last;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, li = lane & 15;
    // Workgroup x runs on XCD x % 8: each XCD takes a contiguous run of the tiles, along the
    // larger operand's panels' other side, so that operand is fetched by as few L2s as possible.
    int pos = blockIdx.x;
    const int full = (int)(gridDim.x / 8) * 8;
    if (pos < full) pos = (pos % 8) * (full / 8) + pos / 8;
    const bool by_rows = p.M > p.N;
    const int tm = by_rows ? pos / tiles_n : pos % tiles_m;
    const int tn = by_rows ? pos % tiles_n : pos / tiles_m;
    const int m0 = tm * kTm, n0 = tn * kTn;

    const int kb = blockIdx.y * p.k_per_split, ke = min(p.K, kb + p.k_per_split);
    const int steps = (ke - kb) >> 4;                      // 16-deep steps of this workgroup
    const int s0 = steps * wave / kWaves, s1 = steps * (wave + 1) / kWaves;
    const int ns = s1 - s0, k0 = kb + 16 * s0;

    const int64_t a_span = CONV ? (int64_t)p.cn * p.cih * p.ciw * p.cic : (int64_t)(p.M - 1) * p.sam + p.K;
    const int64_t b_span = BT ? (int64_t)(p.N - 1) * p.sbn + p.K : (int64_t)(p.K - 1) * p.sbk + p.N;
    const __amdgpu_buffer_rsrc_t ar = buffer_rsrc(p.a, a_span), br = buffer_rsrc(p.b, b_span);

    // A: byte offset of each row's next chunk; a convolution's rows are recomputed per tap
    unsigned va[kFm];
    int abase[CONV ? kFm : 1], iy0[CONV ? kFm : 1], ix0[CONV ? kFm : 1];
    int ky = 0, kx = 0, ic = 0;
    auto tap = [&]() __attribute__((always_inline)) {
        if constexpr (CONV) {
#pragma unroll
            for (int i = 0; i < kFm; ++i) {
                const bool ok = (unsigned)(iy0[i] + ky) < (unsigned)p.cih &&
                                (unsigned)(ix0[i] + kx) < (unsigned)p.ciw;
                va[i] = ok ? (unsigned)(abase[i] + (ky * p.ciw + kx) * p.cic + 4 * g) * 4u : kOob;
            }
        }
    };
#pragma unroll
    for (int i = 0; i < kFm; ++i) {
        const int m = m0 + 16 * i + li;
        if constexpr (CONV) {
            const int mm = min(m, p.M - 1);
            const int ox = mm % p.cow, t = mm / p.cow, oy = t % p.coh, img = t / p.coh;
            iy0[i] = m < p.M ? oy * p.csh - p.cpt : -(1 << 28);  // rows past M fail every check
            ix0[i] = ox * p.csw - p.cpl;
            abase[i] = (img * p.cih * p.ciw + (oy * p.csh - p.cpt) * p.ciw + ix0[i]) * p.cic;
        } else {
            va[i] = (unsigned)(((int64_t)min(m, p.M - 1) * p.sam + k0 + 4 * g) * 4);
        }
    }
    if constexpr (CONV) {
        ic = k0 % p.cic;
        const int t = k0 / p.cic;
        kx = t % p.ckw;
        ky = t / p.ckw;
        tap();
    }
    unsigned vb[kFn];
#pragma unroll
    for (int j = 0; j < kFn; ++j) {
        if constexpr (BT)
            vb[j] = (unsigned)(((int64_t)min(n0 + 16 * j + li, p.N - 1) * p.sbn + k0 + 4 * g) * 4);
        else
            vb[j] = (unsigned)(((int64_t)(k0 + 4 * g + j) * p.sbk + min(n0 + 4 * li, p.N - 4)) * 4);
    }
    const unsigned b_step = BT ? 64u : (unsigned)(64 * p.sbk);

    // This thread's result: four columns of one row (4 li .. + 3 of a [K][N] operand's tile, li + 16 c
    // of an [N][K] operand's).  Its bias and residual load with the operands.
    constexpr int CS = BT ? 16 : 1;
    const int om = m0 + 16 * (wave >> 2) + 4 * g + (wave & 3), on = n0 + (BT ? li : 4 * li);
    const bool own = om < p.M && on < p.N;
    const int64_t oo = (int64_t)om * p.scm + on;
    f4v bias = {0.f, 0.f, 0.f, 0.f}, resid = bias;
    if (own) {
        if constexpr (!BT) {
            if (p.bias) bias = *reinterpret_cast<const f4v*>(p.bias + on);
            if (p.residual) resid = *reinterpret_cast<const f4v*>(p.residual + oo);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (on + CS * c < p.N) {
                    if (p.bias) bias[c] = p.bias[on + CS * c];
                    if (p.residual) resid[c] = p.residual[oo + CS * c];
                }
        }
    }

    struct Stage { f4v a[kFm], b[kFn]; };
    Stage st[kStages];
    int at = 0;  // next step to load
    auto load = [&](Stage& s) __attribute__((always_inline)) {
        const bool in = at < ns;  // uniform over the wavefront
        if constexpr (CONV) {
#pragma unroll
            for (int i = 0; i < kFm; ++i) s.a[i] = load4(ar, in ? va[i] : kOob, in ? (unsigned)(ic * 4) : 0u);
            ic += 16;
            if (ic == p.cic) {
                ic = 0;
                if (++kx == p.ckw) { kx = 0; ++ky; }
                tap();
            }
        } else {
#pragma unroll
            for (int i = 0; i < kFm; ++i) s.a[i] = load4(ar, in ? va[i] : kOob, in ? (unsigned)(at * 64) : 0u);
        }
#pragma unroll
        for (int j = 0; j < kFn; ++j) s.b[j] = load4(br, in ? vb[j] : kOob, in ? (unsigned)at * b_step : 0u);
        ++at;
    };
    floatx4 acc[kFm][kFn];
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
        for (int j = 0; j < kFn; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto mul = [&](const Stage& s) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < kFm; ++i)
#pragma unroll
                for (int j = 0; j < kFn; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.a[i][q], BT ? s.b[j][q] : s.b[q][j],
                                                                    acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < kStages - 1; ++u) load(st[u]);
    int k = 0;
    for (; k + kStages <= ns; k += kStages) {
#pragma unroll
        for (int u = 0; u < kStages; ++u) {
            load(st[(u + kStages - 1) % kStages]);
            __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the products
            mul(st[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < kStages - 1; ++u)
        if (k + u < ns) mul(st[u]);

    // Result e = (i * 4 + r): row 16 i + 4 g + r, columns 4 li .. + 3 ([K][N]) or li + 16 c.
#pragma unroll
    for (int i = 0; i < kFm; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            red[(wave * IDX + i * 4 + r) * 64 + lane] =
                f4v{acc[i][0][r], acc[i][1][r], acc[i][2][r], acc[i][3][r]};
    __syncthreads();
    static_assert(IDX == kWaves, "one result row per wavefront");
    f4v v = red[wave * 64 + lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) v += red[(w * IDX + wave) * 64 + lane];

    if (p.splits > 1) {
        const int S = p.splits, tile = tm * tiles_n + tn;
        const __amdgpu_buffer_rsrc_t pr =
            buffer_rsrc(p.partial + (int64_t)tile * S * (kTm * kTn), (int64_t)S * kTm * kTn);
        st_coh16(pr, (unsigned)((blockIdx.y * kWaves * 64 + tid) * 16), make_float4(v.x, v.y, v.z, v.w));
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this thread's partial is stored
        __syncthreads();
        if (tid == 0)
            last = __hip_atomic_fetch_add((SHP_GLOBAL int*)(p.counters + tile), 1, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT) == S - 1;
        __syncthreads();
        if (!last) return;
        if (tid == 0)  // every split has arrived: the counter is free for the next launch
            __hip_atomic_store((SHP_GLOBAL int*)(p.counters + tile), 0, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        float4 q[kMaxSplits];
#pragma unroll
        for (int u = 0; u < kMaxSplits; ++u)
            if (u < S) q[u] = ld_coh16(pr, (unsigned)((u * kWaves * 64 + tid) * 16), 0);
        v = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < kMaxSplits; ++u)
            if (u < S) v += f4v{q[u].x, q[u].y, q[u].z, q[u].w};
    }
    if (!own) return;
    if (p.bias) v += bias;
    if (p.residual) v += resid;
    if (p.act) {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = shpd::apply_act(v[c], p.act, p.alpha);
    }
    if constexpr (!BT) {
        *reinterpret_cast<f4v*>(p.c + oo) = v;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (on + CS * c < p.N) p.c[oo + CS * c] = v[c];
    }
}

}  // namespace

namespace shp {

bool direct_eligible(const GemmParams& p, int amode, int bmode, int cmode) {
    if (cmode != C_STRIDED || p.batch_outer * p.batch_inner != 1 || p.K < 16 || p.K % 16 ||
        p.N < 4 || p.N % 4 || p.M <= 0 || p.scn != 1 || p.scm % 4 || p.short_chains)
        return false;
    if (((uintptr_t)p.a | (uintptr_t)p.b | (uintptr_t)p.c | (uintptr_t)p.bias | (uintptr_t)p.residual) & 15)
        return false;
    const int64_t lim = (int64_t)1 << 29;  // floats: byte offsets stay below 2 GiB
    if (amode == A_CONV_NHWC4) {
        if (p.cic % 16 || (int64_t)p.cn * p.cih * p.ciw * p.cic > lim) return false;
    } else if (amode != A_KVEC || p.sak != 1 || p.sam % 4 || (int64_t)(p.M - 1) * p.sam + p.K > lim) {
        return false;
    }
    if (bmode == B_NVEC)
        return p.sbn == 1 && p.sbk % 4 == 0 && (int64_t)(p.K - 1) * p.sbk + p.N <= lim;
    return bmode == B_KVEC && p.sbk == 1 && p.sbn % 4 == 0 && (int64_t)(p.N - 1) * p.sbn + p.K <= lim;
}

// Splits the direct kernel takes the problem with, 0 for the tiled kernels (`tune` < 0 never, > 0
// always, with that many splits).  The line lies at one workgroup per CU: with at most 256 tiles
// the direct kernel won on all 114 of the swept shapes (1x1 and 3x3 convolutions of CNN layers at
// batches 1-32, BERT's and TinyLlama's products with 1-2,048 rows) by 1.08-1.82 times, 1.35 at the
// median (512x768x768 16.3 -> 10.4 us); above it the tiled kernels did on 57 of 80, and gemm_launch
// compares both estimates.  K is split while every CU
// still gets at most one workgroup and a split keeps 128 k: a second round of workgroups costs more
// than the shorter chains give (200x2304x768, 252 tiles: 10.5 us unsplit, 13.2 in two).
//
// A further sweep (840 products and convolutions up to K = 51,200, both operand orders) found where
// that ends: where the workgroups' own K is long and they leave CUs idle, the tiled kernels' splits
// fill the GPU better, and an [N][K] operand, whose loads are 64 bytes of 16 rows, earlier still:
//  - [K][N]: from 4,000 k a workgroup while these fill less than three quarters of the CUs
//    (1000x300x16384 124 us, tiled 90; at 192 workgroups and more direct still wins);
//  - [N][K] products: from 3,000 k, or 2,000 while they fill less than that (265x952x11376 94 us,
//    tiled 67; 1164x264x2080 26.6, 24.3);
//  - [N][K] convolutions with taps: from 300 k, 700 under 160 workgroups and 4,000 under 64
//    (2x32x32x2048 to 192 channels, 3x3: 237 us, tiled 143; 7x28x28x256 to 192, stride 2: 38, 30);
//    1x1 with a stride, which the tiled kernel reads as rows: from 300 k, and with K under 512
//    (12x16x16x2048 to 256: 23.5, 16.4; 9x33x33x48 to 128: 7.6, 5.9; 7x32x32x512 to 16: 9.8, 14.6).
// Over 930 shapes this is within 0.4 % of the faster of the two on average.
int direct_splits(const GemmParams& p, int amode, int bmode, int tune) {
    if (tune < 0) return 0;
    const int64_t tiles = (int64_t)((p.M + kTm - 1) / kTm) * ((p.N + kTn - 1) / kTn);
    const int steps = p.K / 16;
    if (tiles > (int64_t)(kSplitCounterBytes / sizeof(int))) return 0;
    int s = 1;
    if (tune > 0) {
        s = std::min(tune, kMaxSplits);
    } else {
        if (tiles > 256) return 0;
        for (int t : {2, 3, 4, 6, 8})
            if (tiles * t <= 256 && p.K / t >= 128) s = t;
        const int64_t wgs = tiles * s;
        const int k = p.K / s;
        const bool conv = amode == A_CONV_NHWC4;
        if (bmode == B_NVEC) {
            if (!conv && k > 4000 && wgs < 192) return 0;
        } else if (conv && p.ckh * p.ckw > 1) {
            if (k > (wgs < 64 ? 4000 : wgs < 160 ? 700 : 300)) return 0;
        } else if (conv && (p.csh > 1 || p.csw > 1)) {
            if (p.K < 512 || k > 300) return 0;
        } else if (k > (wgs < 192 ? 2000 : 3000)) {
            return 0;
        }
    }
    const int per = (steps + s - 1) / s;
    return (steps + per - 1) / per;
}

// Above one tile per CU, by time estimates: [K][N] operands only.  With [N][K] ones the direct kernel
// lost on 141 of 143 swept shapes, by up to 1.9 times (3x56x56x192 to 512 channels, 3x3: 244 us, tiled 153).
bool direct_may_exceed(const GemmParams& p, int bmode) {
    const int64_t tiles = (int64_t)((p.M + kTm - 1) / kTm) * ((p.N + kTn - 1) / kTn);
    return tiles > 256 && bmode == B_NVEC;
}

size_t direct_workspace(const GemmParams& p, int splits) {
    if (splits <= 1) return 0;
    const size_t tiles = (size_t)((p.M + kTm - 1) / kTm) * ((p.N + kTn - 1) / kTn);
    return kSplitCounterBytes + tiles * splits * kTm * kTn * sizeof(float);
}

int direct_launch(hipStream_t stream, GemmParams p, int amode, int bmode, int splits,
                  float* workspace) {
    const int tiles_m = (p.M + kTm - 1) / kTm, tiles_n = (p.N + kTn - 1) / kTn;
    p.splits = splits;
    p.k_per_split = (p.K / 16 + splits - 1) / splits * 16;
    p.partial = splits > 1 ? workspace + kSplitCounterBytes / sizeof(float) : nullptr;
    p.counters = splits > 1 ? reinterpret_cast<int*>(workspace) : nullptr;
    const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)splits);
    auto kern = amode == A_KVEC
                    ? (bmode == B_NVEC ? gemm_direct_kernel<A_KVEC, B_NVEC> : gemm_direct_kernel<A_KVEC, B_KVEC>)
                    : (bmode == B_NVEC ? gemm_direct_kernel<A_CONV_NHWC4, B_NVEC>
                                       : gemm_direct_kernel<A_CONV_NHWC4, B_KVEC>);
    hipLaunchKernelGGL(kern, grid, dim3(kWaves * 64), 0, stream, p, tiles_m, tiles_n);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

}  // namespace shp
