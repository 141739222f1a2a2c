// The HLO path's shape ops that the reference runs on the host CPU between its Vulkan
// dispatches, as device kernels so tensors stay resident in HBM:
//   broadcast / broadcast_in_dim  source/xla_hlo/src/compiler.rs:336-347, broadcast_tensor :1361-1393
//   transpose (any rank)          compiler.rs:374-386, transpose_tensor :1395-1418
//   slice                         compiler.rs:570-582, parse_slice_spec :1897-1929, cpu_slice :1931-1952
//   concatenate                   compiler.rs:554-569, cpu_concatenate :1879-1895
//   compare (predicate as f32)    compiler.rs:511-537, binary_tensor :1521-1564, infer_broadcast_dims :1566-1572
//   select                        compiler.rs:538-553, select_tensor :1574-1620
//   reduce over any rank          compiler.rs:939-1007 (rank > 4 -> reduce_tensor :1730-1759), reduce_kind :1722-1728
//   strided copy                  no counterpart: materialises a view of the compiled HLO program
// The reference has no GLSL kernel (so no push layout) for these; the i32 push vectors
// below carry the HLO attributes directly (shapes, `dimensions`, slice starts/limits/strides,
// compare direction), so a host lowering passes what it parsed.  Ranks up to 8.
//
// Broadcast, transpose and slice are one strided gather: output coordinate c reads source
// element base + sum_k c_k * stride_k (stride 0 on broadcast axes, permuted strides for a
// transpose, start/step for a slice).  All are HBM-bound copies: one thread per output
// element, consecutive threads on consecutive outputs.
#include <cstring>

#include "coherent.h"
#include "common.h"
#include "fastdiv.h"

namespace {

constexpr int kBlock = 256;
constexpr int kMaxRank = 8;

unsigned hlo_grid(uint64_t n) {
    uint64_t g = (n + kBlock - 1) / kBlock;
    if (g > 256 * 32) g = 256 * 32;
    return g == 0 ? 1u : (unsigned)g;
}

struct Gather {
    int r;
    int dims[kMaxRank];         // output dims
    int64_t stride[kMaxRank];   // source element stride per output axis
    int64_t base;               // source offset of output coordinate 0
    int check;                  // slice: zero where first + c*step >= lim on some axis
    int64_t first[kMaxRank], step[kMaxRank], lim[kMaxRank];
};

__global__ __launch_bounds__(kBlock) void gather_kernel(const float* __restrict__ x,
                                                        float* __restrict__ y, Gather g,
                                                        uint64_t total) {
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += stride) {
        uint64_t rem = i;
        int64_t off = g.base;
        bool ok = true;
        for (int k = g.r - 1; k >= 0; --k) {
            const int64_t c = (int64_t)(rem % (uint64_t)g.dims[k]);
            rem /= (uint64_t)g.dims[k];
            off += c * g.stride[k];
            if (g.check) ok = ok && (g.first[k] + c * g.step[k] < g.lim[k]);
        }
        float v = 0.0f;
        if (ok) v = x[off];
        y[i] = v;
    }
}

// Row-major element strides of a shape.
void strides_of(const int* dims, int r, int64_t* st) {
    int64_t s = 1;
    for (int k = r - 1; k >= 0; --k) {
        st[k] = s;
        s *= dims[k];
    }
}

int64_t elems_of(const int* dims, int r) {
    int64_t n = 1;
    for (int k = 0; k < r; ++k) n *= dims[k];
    return n;
}

int read_dims(const int32_t* q, int r, int* dims, const char* kernel) {
    for (int k = 0; k < r; ++k) {
        if (q[k] <= 0) return shp::fail(SHP_ERR_SHAPE, std::string(kernel) + ": dims must be > 0");
        dims[k] = q[k];
    }
    return SHP_OK;
}

// ---- the gather's fast forms (fewer than 2^31 elements, no coordinate outside the source).  The
// generic kernel above spends a 64-bit division per axis and moves 4 bytes per thread, and reads one
// line per element where a transpose moves the contiguous axis.  After dropping axes of size 1 and
// merging axes that stay neighbours:
// * rows (the innermost output axis is contiguous in the source, or a broadcast): 16 bytes per thread,
//   four in flight, divisions by multiplication (8x384x32x128 to 8x32x384x128: 52 -> 19 us); single
//   elements where length or alignment do not allow 16 bytes;
// * a transpose (some other axis is the contiguous one): tiles of both axes through LDS, so reads run
//   along the source's contiguous axis and writes along the output's (8x306x32x64 to 8x32x64x306:
//   31 -> 12 us); single elements where the matrices or the tensor are small.
using shpd::FastDiv;
using shpd::fast_div;
using shpd::fdiv;

struct Rows {
    int r;                        // axes outside the innermost, outermost first
    FastDiv d[kMaxRank];          // their sizes; d[r]: 16-byte (or single) elements of a row
    int64_t stride[kMaxRank];     // source strides in floats; [r]: along a row of single elements
    int64_t base;
};
enum { ROWS_VEC = 0, ROWS_SPLAT = 1, ROWS_SINGLE = 2 };

template <int MODE, int U>
__global__ __launch_bounds__(kBlock) void gather_rows_kernel(const float* __restrict__ x,
                                                             float* __restrict__ y, Rows g,
                                                             unsigned total) {
    typedef float elem __attribute__((ext_vector_type(MODE == ROWS_SINGLE ? 1 : 4)));
    elem* const ye = reinterpret_cast<elem*>(y);
    for (unsigned b0 = blockIdx.x * (kBlock * U) + threadIdx.x; b0 < total;
         b0 += gridDim.x * (kBlock * U)) {
        elem v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned i = min(b0 + u * kBlock, total - 1);
            unsigned q = fdiv(i, g.d[g.r]);
            const int64_t c = i - q * g.d[g.r].d;
            int64_t off = g.base + (MODE == ROWS_VEC ? c * 4 : MODE == ROWS_SINGLE ? c * g.stride[g.r] : 0);
            for (int k = g.r - 1; k >= 0; --k) {
                const unsigned n = fdiv(q, g.d[k]);
                off += (int64_t)(q - n * g.d[k].d) * g.stride[k];
                q = n;
            }
            if constexpr (MODE == ROWS_SPLAT) v[u] = x[off];
            else v[u] = *reinterpret_cast<const elem*>(x + off);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (b0 + u * kBlock < total) ye[b0 + u * kBlock] = v[u];
    }
}

struct Tiles {
    int a, b;                     // sizes of the output's innermost axis and the source's
    int ta, tb;                   // tile: ta * tb <= 4096
    int64_t sa, ob;               // source stride along a, output stride along b (both others 1)
    FastDiv fta, ftb;             // by the tile's sizes
    FastDiv na, nb;               // tiles along a and b
    int r;                        // the other axes, outermost first
    FastDiv d[kMaxRank];
    int64_t in[kMaxRank], out[kMaxRank];
    int64_t base;
};

__global__ __launch_bounds__(256) void gather_tiles_kernel(const float* __restrict__ x,
                                                           float* __restrict__ y, Tiles g) {
    __shared__ float tile[4096 + 256];
    unsigned q = fdiv(blockIdx.x, g.na);
    const int a0 = (int)(blockIdx.x - q * g.na.d) * g.ta;
    const unsigned q2 = fdiv(q, g.nb);
    const int b0 = (int)(q - q2 * g.nb.d) * g.tb;
    q = q2;
    int64_t in = g.base, out = 0;
    for (int k = g.r - 1; k >= 0; --k) {
        const unsigned n = fdiv(q, g.d[k]);
        const int64_t c = q - n * g.d[k].d;
        in += c * g.in[k];
        out += c * g.out[k];
        q = n;
    }
    const int ls = g.ta | 1;  // odd: a column of the tile touches every bank
    const int n = g.ta * g.tb;
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i * 256 >= n) break;  // uniform
        const unsigned e = i * 256 + threadIdx.x;
        const unsigned ea = fdiv(e, g.ftb), eb = e - ea * g.ftb.d;
        if ((int)e < n && a0 + (int)ea < g.a && b0 + (int)eb < g.b)
            v[i] = x[in + (int64_t)(a0 + (int)ea) * g.sa + b0 + (int)eb];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i * 256 >= n) break;
        const unsigned e = i * 256 + threadIdx.x;
        const unsigned ea = fdiv(e, g.ftb), eb = e - ea * g.ftb.d;
        if ((int)e < n) tile[eb * ls + ea] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (i * 256 >= n) break;
        const unsigned e = i * 256 + threadIdx.x;
        const unsigned eb = fdiv(e, g.fta), ea = e - eb * g.fta.d;
        if ((int)e < n && a0 + (int)ea < g.a && b0 + (int)eb < g.b)
            y[out + (int64_t)(b0 + (int)eb) * g.ob + a0 + (int)ea] = tile[eb * ls + ea];
    }
}

int launch_gather(const shp::Launch& l, const Gather& g0) {
    // An output coordinate can leave the source only where a slice's limit does.
    Gather g = g0;
    if (g.check) {
        bool inside = true;
        for (int k = 0; k < g.r; ++k) inside &= g.first[k] + (g.dims[k] - 1) * g.step[k] < g.lim[k];
        if (inside) g.check = 0;
    }
    const float* x = (const float*)l.in0;
    float* y = (float*)l.out;
    if (!g.check && l.out_elems < (1ull << 31)) {
        int d[kMaxRank], r = 0;
        int64_t st[kMaxRank];
        for (int k = 0; k < g.r; ++k) {
            if (g.dims[k] == 1) continue;
            if (r && st[r - 1] == g.stride[k] * g.dims[k]) {
                d[r - 1] *= g.dims[k];
                st[r - 1] = g.stride[k];
            } else {
                d[r] = g.dims[k];
                st[r++] = g.stride[k];
            }
        }
        if (!r) {
            d[0] = 1;
            st[0] = 1;
            r = 1;
        }
        const int n = d[r - 1];
        bool rows = n % 4 == 0 && ((uintptr_t)y & 15) == 0;
        if (st[r - 1] == 1) {
            rows = rows && ((uintptr_t)(x + g.base) & 15) == 0;
            for (int k = 0; k < r - 1; ++k) rows = rows && st[k] % 4 == 0;
        } else {
            rows = rows && st[r - 1] == 0;
        }
        auto launch_rows = [&](bool vec) {
            Rows p{};
            p.r = r - 1;
            p.base = g.base;
            for (int k = 0; k < r; ++k) {
                p.d[k] = fast_div((unsigned)(k < r - 1 || !vec ? d[k] : n / 4));
                p.stride[k] = st[k];
            }
            const unsigned total = (unsigned)(vec ? l.out_elems / 4 : l.out_elems);
            // four per thread once that still leaves four workgroups per CU
            const bool many = total >= (1u << 20);
            const unsigned grid = many ? std::min<unsigned>((total + kBlock * 4 - 1) / (kBlock * 4), 256 * 32)
                                       : (total + kBlock - 1) / kBlock;
            auto kern = !vec ? (many ? gather_rows_kernel<ROWS_SINGLE, 4> : gather_rows_kernel<ROWS_SINGLE, 1>)
                        : st[r - 1] == 1
                            ? (many ? gather_rows_kernel<ROWS_VEC, 4> : gather_rows_kernel<ROWS_VEC, 1>)
                            : (many ? gather_rows_kernel<ROWS_SPLAT, 4> : gather_rows_kernel<ROWS_SPLAT, 1>);
            hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, l.stream, x, y, p, total);
            SHP_HIP_CHECK(hipGetLastError());
            return (int)SHP_OK;
        };
        if (rows) return launch_rows(true);
        int bx = -1;  // the source's contiguous axis
        for (int k = 0; k < r - 1; ++k)
            if (st[k] == 1) bx = k;
        Tiles p{};
        if (bx >= 0 && st[r - 1] > 1) {
            p.a = n;
            p.b = d[bx];
            // up to 64 of each, or one axis longer where the other is short
            p.ta = std::min(n, 64);
            p.tb = std::min(p.b, std::min(256, 4096 / p.ta));
            p.ta = std::min(n, std::min(256, 4096 / p.tb));
        }
        // A tile pays a load, LDS and store latency of its own: it wins from 1,024 elements a tile on
        // (200,000 matrices of 32x32 329 us, 606 as single elements, but of 16x32 235 against 212 and of
        // 4x8 134 against 11), once there are 1.25 M elements, which fill the GPU with tiles (8x384x7x64
        // 7.8 against 10.7; 256 matrices of 64x64 6.6 against 4.9, one 300x33 5.8 against 2.6).  So a
        // launch has fewer than 2^24 tiles.
        if (p.ta * p.tb >= 1024 && l.out_elems >= (5u << 18)) {
            p.sa = st[r - 1];
            p.base = g.base;
            p.fta = fast_div(p.ta);
            p.ftb = fast_div(p.tb);
            const int na = (n + p.ta - 1) / p.ta, nb = (p.b + p.tb - 1) / p.tb;
            p.na = fast_div(na);
            p.nb = fast_div(nb);
            int64_t os = 1, wgs = (int64_t)na * nb;
            int64_t ost[kMaxRank];
            for (int k = r - 1; k >= 0; --k) {
                ost[k] = os;
                os *= d[k];
            }
            p.ob = ost[bx];
            for (int k = 0; k < r - 1; ++k) {
                if (k == bx) continue;
                p.d[p.r] = fast_div(d[k]);
                p.in[p.r] = st[k];
                p.out[p.r++] = ost[k];
                wgs *= d[k];
            }
            hipLaunchKernelGGL(gather_tiles_kernel, dim3((unsigned)wgs), dim3(256), 0, l.stream, x,
                               y, p);
            SHP_HIP_CHECK(hipGetLastError());
            return SHP_OK;
        }
        return launch_rows(false);
    }
    hipLaunchKernelGGL(gather_kernel, dim3(hlo_grid(l.out_elems)), dim3(kBlock), 0, l.stream, x, y, g,
                       l.out_elems);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

// Operand broadcast as binary_tensor / select_tensor do it: an operand with as many
// elements as the output is taken flat; one element is splatted; otherwise its axes align
// with the trailing output axes (infer_broadcast_dims) and size-1 axes broadcast
// (broadcast_tensor).  Fills per-output-axis strides.
int operand_strides(const int* sd, int rs, const int* od, int ro, int64_t* st,
                    const char* kernel) {
    const int64_t n = elems_of(sd, rs), total = elems_of(od, ro);
    if (n == total) {
        strides_of(od, ro, st);
        return SHP_OK;
    }
    for (int k = 0; k < ro; ++k) st[k] = 0;
    if (n == 1) return SHP_OK;
    if (rs > ro) return shp::fail(SHP_ERR_SHAPE, std::string(kernel) + ": operand rank > output rank");
    int64_t sst[kMaxRank];
    strides_of(sd, rs, sst);
    const int offset = ro - rs;
    for (int a = 0; a < rs; ++a) {
        if (sd[a] == 1) continue;
        if (sd[a] != od[a + offset])
            return shp::fail(SHP_ERR_SHAPE, std::string(kernel) + ": operand does not broadcast");
        st[a + offset] = sst[a];
    }
    return SHP_OK;
}

// ---- hlo_broadcast: push {r_src, r_out, total, src_dims[r_src], out_dims[r_out],
//      dimensions[r_src]} (dimensions[a] = output axis of source axis a, as in HLO).
int launch_broadcast(const shp::Launch& l) {
    const int32_t* q = l.push;
    const int rs = q[0], ro = q[1];
    if (rs < 0 || rs > kMaxRank || ro < 1 || ro > kMaxRank)
        return shp::fail(SHP_ERR_SHAPE, "hlo_broadcast: rank out of range (0..8 / 1..8)");
    if ((int64_t)l.n_push < 3 + 2 * rs + ro)
        return shp::fail(SHP_ERR_PUSH, "hlo_broadcast needs 3 + 2*r_src + r_out push constants");
    int sd[kMaxRank], od[kMaxRank];
    int rc = read_dims(q + 3, rs, sd, "hlo_broadcast");
    if (!rc) rc = read_dims(q + 3 + rs, ro, od, "hlo_broadcast");
    if (rc) return rc;
    const int32_t* map = q + 3 + rs + ro;
    if (elems_of(od, ro) != q[2]) return shp::fail(SHP_ERR_SHAPE, "hlo_broadcast: total != product of out dims");
    rc = shp::check_total(l, q[2], "hlo_broadcast");
    if (rc) return rc;
    Gather g{};
    g.r = ro;
    for (int k = 0; k < ro; ++k) g.dims[k] = od[k];
    const int64_t n = elems_of(sd, rs);
    bool same = (rs == ro);
    for (int k = 0; same && k < rs; ++k) same = sd[k] == od[k];
    if (same) {  // broadcast_tensor: identical shape -> copy
        strides_of(od, ro, g.stride);
    } else if (n == 1) {  // one element -> splat (strides stay 0)
    } else {
        int64_t sst[kMaxRank];
        strides_of(sd, rs, sst);
        for (int a = 0; a < rs; ++a) {
            if (map[a] < 0 || map[a] >= ro)
                return shp::fail(SHP_ERR_SHAPE, "hlo_broadcast: dimensions entry out of range");
            if (sd[a] == 1) continue;
            if (sd[a] != od[map[a]])
                return shp::fail(SHP_ERR_SHAPE, "hlo_broadcast: source dim != mapped output dim");
            g.stride[map[a]] += sst[a];
        }
    }
    return launch_gather(l, g);
}

// ---- hlo_transpose: push {r, total, src_dims[r], perm[r]}; output axis i is source axis
//      perm[i] (HLO `dimensions`), so out dims are src_dims[perm[i]].
int launch_transpose_nd(const shp::Launch& l) {
    const int32_t* q = l.push;
    const int r = q[0];
    if (r < 1 || r > kMaxRank) return shp::fail(SHP_ERR_SHAPE, "hlo_transpose: rank out of range 1..8");
    if ((int64_t)l.n_push < 2 + 2 * r) return shp::fail(SHP_ERR_PUSH, "hlo_transpose needs 2 + 2*r push constants");
    int sd[kMaxRank];
    int rc = read_dims(q + 2, r, sd, "hlo_transpose");
    if (rc) return rc;
    const int32_t* perm = q + 2 + r;
    int seen = 0;
    for (int i = 0; i < r; ++i) {
        if (perm[i] < 0 || perm[i] >= r || (seen >> perm[i]) & 1)
            return shp::fail(SHP_ERR_SHAPE, "hlo_transpose: dimensions is not a permutation");
        seen |= 1 << perm[i];
    }
    if (elems_of(sd, r) != q[1]) return shp::fail(SHP_ERR_SHAPE, "hlo_transpose: total != product of dims");
    rc = shp::check_total(l, q[1], "hlo_transpose");
    if (rc) return rc;
    Gather g{};
    g.r = r;
    int64_t sst[kMaxRank];
    strides_of(sd, r, sst);
    for (int i = 0; i < r; ++i) {
        g.dims[i] = sd[perm[i]];
        g.stride[i] = sst[perm[i]];
    }
    return launch_gather(l, g);
}

// ---- hlo_slice: push {r, total, src_dims[r], starts[r], limits[r], strides[r]}; output dim
//      k is ceil((limit - start) / stride).  As cpu_slice, an output whose source coordinate
//      falls outside the source is 0.
int launch_slice(const shp::Launch& l) {
    const int32_t* q = l.push;
    const int r = q[0];
    if (r < 1 || r > kMaxRank) return shp::fail(SHP_ERR_SHAPE, "hlo_slice: rank out of range 1..8");
    if ((int64_t)l.n_push < 2 + 4 * r) return shp::fail(SHP_ERR_PUSH, "hlo_slice needs 2 + 4*r push constants");
    int sd[kMaxRank];
    int rc = read_dims(q + 2, r, sd, "hlo_slice");
    if (rc) return rc;
    const int32_t *st = q + 2 + r, *lim = q + 2 + 2 * r, *sp = q + 2 + 3 * r;
    Gather g{};
    g.r = r;
    g.check = 1;
    int64_t sst[kMaxRank];
    strides_of(sd, r, sst);
    for (int k = 0; k < r; ++k) {
        if (st[k] < 0 || sp[k] < 1 || lim[k] <= st[k])
            return shp::fail(SHP_ERR_SHAPE, "hlo_slice: need 0 <= start < limit and stride >= 1");
        g.dims[k] = (lim[k] - st[k] + sp[k] - 1) / sp[k];
        g.first[k] = st[k];
        g.step[k] = sp[k];
        g.lim[k] = sd[k];
        g.stride[k] = sst[k] * sp[k];
        if (st[k] < sd[k]) g.base += st[k] * sst[k];
    }
    if (elems_of(g.dims, r) != q[1]) return shp::fail(SHP_ERR_SHAPE, "hlo_slice: total != product of slice dims");
    rc = shp::check_total(l, q[1], "hlo_slice");
    if (rc) return rc;
    // a start past the source end leaves only zeros on that axis: keep the gather in range
    for (int k = 0; k < r; ++k)
        if (st[k] >= sd[k]) g.stride[k] = 0;
    return launch_gather(l, g);
}

// ---- hlo_concatenate_into: writes one operand (in0) into its slab of the output.
//      push {r, dim, offset, out_dims[r], in_dims[r]}; the operand's coordinate along `dim`
//      is shifted by `offset` (the summed extents of the operands before it); coordinates
//      past the output are dropped, as cpu_concatenate does.  N operands = N launches.
struct Slab {
    int r, dim, offset;
    int in_dims[kMaxRank], out_dims[kMaxRank];
    int64_t out_stride[kMaxRank];
};

__global__ __launch_bounds__(kBlock) void concat_into_kernel(const float* __restrict__ x,
                                                             float* __restrict__ y, Slab s,
                                                             uint64_t n_in) {
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n_in; i += stride) {
        uint64_t rem = i;
        int64_t off = 0;
        bool ok = true;
        for (int k = s.r - 1; k >= 0; --k) {
            int64_t c = (int64_t)(rem % (uint64_t)s.in_dims[k]);
            rem /= (uint64_t)s.in_dims[k];
            if (k == s.dim) c += s.offset;
            ok = ok && c < s.out_dims[k];
            off += c * s.out_stride[k];
        }
        if (ok) y[off] = x[i];
    }
}

int launch_concatenate_into(const shp::Launch& l) {
    const int32_t* q = l.push;
    const int r = q[0];
    if (r < 1 || r > kMaxRank) return shp::fail(SHP_ERR_SHAPE, "hlo_concatenate_into: rank out of range 1..8");
    if ((int64_t)l.n_push < 3 + 2 * r)
        return shp::fail(SHP_ERR_PUSH, "hlo_concatenate_into needs 3 + 2*r push constants");
    Slab s{};
    s.r = r;
    s.dim = q[1];
    s.offset = q[2];
    if (s.dim < 0 || s.dim >= r || s.offset < 0)
        return shp::fail(SHP_ERR_SHAPE, "hlo_concatenate_into: bad dim/offset");
    int rc = read_dims(q + 3, r, s.out_dims, "hlo_concatenate_into");
    if (!rc) rc = read_dims(q + 3 + r, r, s.in_dims, "hlo_concatenate_into");
    if (rc) return rc;
    rc = shp::check_total(l, elems_of(s.out_dims, r), "hlo_concatenate_into");
    if (rc) return rc;
    strides_of(s.out_dims, r, s.out_stride);
    const uint64_t n_in = (uint64_t)elems_of(s.in_dims, r);
    hipLaunchKernelGGL(concat_into_kernel, dim3(hlo_grid(n_in)), dim3(kBlock), 0, l.stream,
                       (const float*)l.in0, (float*)l.out, s, n_in);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

// ---- hlo_compare: y = (a <dir> b) ? 1 : 0 with binary_tensor's operand broadcast.
//      push {direction, total, r_out, r_a, r_b, out_dims[r_out], a_dims[r_a], b_dims[r_b]};
//      direction 0 LT, 1 LE, 2 EQ, 3 NE, 4 GE, 5 GT (the reference's default).
// ---- hlo_select: y = pred != 0 ? on_true : y, where y holds on_false (already broadcast
//      to the output shape) on entry: the ABI has two inputs, so on_false rides in the
//      output buffer.  push {total, r_out, r_p, r_t, out_dims, pred_dims, true_dims}.
struct Bin {
    int r, dir;
    int dims[kMaxRank];
    int64_t as[kMaxRank], bs[kMaxRank];
};

template <bool SELECT>
__global__ __launch_bounds__(kBlock) void compare_select_kernel(const float* __restrict__ a,
                                                                const float* __restrict__ b,
                                                                float* __restrict__ y, Bin p,
                                                                uint64_t total) {
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += stride) {
        uint64_t rem = i;
        int64_t ai = 0, bi = 0;
        for (int k = p.r - 1; k >= 0; --k) {
            const int64_t c = (int64_t)(rem % (uint64_t)p.dims[k]);
            rem /= (uint64_t)p.dims[k];
            ai += c * p.as[k];
            bi += c * p.bs[k];
        }
        const float u = a[ai], v = b[bi];
        if constexpr (SELECT) {
            if (u != 0.0f) y[i] = v;
        } else {
            bool t;
            switch (p.dir) {
                case 0: t = u < v; break;
                case 1: t = u <= v; break;
                case 2: t = u == v; break;
                case 3: t = u != v; break;
                case 4: t = u >= v; break;
                default: t = u > v; break;
            }
            y[i] = t ? 1.0f : 0.0f;
        }
    }
}

template <bool SELECT>
int launch_compare_select(const shp::Launch& l) {
    const char* kernel = SELECT ? "hlo_select" : "hlo_compare";
    // field k of the compare layout; select's layout lacks the leading direction
    auto q = [&](int k) { return l.push[SELECT ? k - 1 : k]; };
    const int ro = q(2), ra = q(3), rb = q(4);
    if (ro < 1 || ro > kMaxRank || ra < 0 || ra > kMaxRank || rb < 0 || rb > kMaxRank)
        return shp::fail(SHP_ERR_SHAPE, std::string(kernel) + ": rank out of range");
    const int64_t need = (SELECT ? 4 : 5) + ro + ra + rb;
    if ((int64_t)l.n_push < need)
        return shp::fail(SHP_ERR_PUSH, std::string(kernel) + " needs " + std::to_string(need) +
                                           " push constants");
    int od[kMaxRank], ad[kMaxRank], bd[kMaxRank];
    const int32_t* dims = &l.push[SELECT ? 4 : 5];
    int rc = read_dims(dims, ro, od, kernel);
    if (!rc) rc = read_dims(dims + ro, ra, ad, kernel);
    if (!rc) rc = read_dims(dims + ro + ra, rb, bd, kernel);
    if (rc) return rc;
    if (elems_of(od, ro) != q(1)) return shp::fail(SHP_ERR_SHAPE, std::string(kernel) + ": total != product of out dims");
    rc = shp::check_total(l, q(1), kernel);
    if (rc) return rc;
    Bin p{};
    p.r = ro;
    p.dir = SELECT ? 0 : q(0);
    if (!SELECT && (p.dir < 0 || p.dir > 5)) return shp::fail(SHP_ERR_INVALID, "hlo_compare: direction 0..5");
    for (int k = 0; k < ro; ++k) p.dims[k] = od[k];
    rc = operand_strides(ad, ra, od, ro, p.as, kernel);
    if (!rc) rc = operand_strides(bd, rb, od, ro, p.bs, kernel);
    if (rc) return rc;
    hipLaunchKernelGGL((compare_select_kernel<SELECT>), dim3(hlo_grid(l.out_elems)), dim3(kBlock),
                       0, l.stream, (const float*)l.in0, (const float*)l.in1, (float*)l.out, p,
                       l.out_elems);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

// ---- hlo_reduce: push {kind, r, total_out, init (f32 bits), src_dims[r], reduce[r]};
//      kind 0 sum, 1 max (reduce_kind); reduce[k] != 0 marks a reduced axis; the output
//      keeps the other axes in order.  Each output folds its inputs in increasing source
//      index from `init`, as reduce_tensor does (so sums match it bit for bit); max is
//      fmaxf, the NaN-ignoring maximum of Rust's f32::max.
struct Red {
    int kind, rk, rr;
    float init;
    int kdims[kMaxRank], rdims[kMaxRank];
    int64_t kstride[kMaxRank], rstride[kMaxRank];
    int64_t rcount;
};

// Any reduced axes (after merging): one thread per output, the last reduced axis in batches of 16
// loads that are all issued before the first of them is folded.
__global__ __launch_bounds__(kBlock) void reduce_nd_kernel(const float* __restrict__ x,
                                                           float* __restrict__ y, Red p,
                                                           uint64_t total) {
    constexpr int U = 16;
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    const int inner = p.rr ? p.rdims[p.rr - 1] : 1;
    const int64_t step = p.rr ? p.rstride[p.rr - 1] : 0;
    const int64_t outer = p.rcount / inner;
    for (uint64_t o = (uint64_t)blockIdx.x * kBlock + threadIdx.x; o < total; o += stride) {
        uint64_t rem = o;
        int64_t off = 0;
        for (int k = p.rk - 1; k >= 0; --k) {
            off += (int64_t)(rem % (uint64_t)p.kdims[k]) * p.kstride[k];
            rem /= (uint64_t)p.kdims[k];
        }
        float acc = p.init;
        int c[kMaxRank] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int64_t j = 0; j < outer; ++j) {
            const float* xp = x + off;
            int i = 0;
            for (; i + U <= inner; i += U) {
                float v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = xp[(i + u) * step];
#pragma unroll
                for (int u = 0; u < U; ++u) acc = p.kind ? fmaxf(acc, v[u]) : acc + v[u];
            }
            for (; i < inner; ++i) {
                const float v = xp[i * step];
                acc = p.kind ? fmaxf(acc, v) : acc + v;
            }
            // next reduced coordinate in row-major order (last reduced axis fastest)
            for (int k = p.rr - 2; k >= 0; --k) {
                off += p.rstride[k];
                if (++c[k] < p.rdims[k]) break;
                off -= (int64_t)p.rdims[k] * p.rstride[k];
                c[k] = 0;
            }
        }
        y[o] = acc;
    }
}

// Contiguous rows of n elements, one output per row.  The order of a sum is fixed (increasing
// index), so an output's adds are one chain in one lane; what can be parallel is the memory.
// 256 threads stage a tile of 8,192 floats, `rows` rows of 8192 / rows columns, with coalesced
// loads into registers and then LDS (rows padded by 4 floats, so 16-byte reads down a column of
// rows are free of bank conflicts), while the tile before it is folded by the first `rows`
// threads.  Few rows per workgroup when there are few rows at all: 1,024 rows of 768 take four
// each, one per CU: 114 us with a thread walking each row, 5.4 us so (10.5 before the LDS reads
// were kept a batch ahead of the adds).
constexpr int kRedTile = 8192;

template <bool VEC, bool MAX>
__global__ __launch_bounds__(256) void reduce_rows_kernel(const float* __restrict__ x,
                                                          float* __restrict__ y,
                                                          float init, int64_t nrows, int n,
                                                          int rows) {
    __shared__ __attribute__((aligned(16))) float tile[kRedTile + 256 * 4];
    constexpr int W = VEC ? 4 : 1, NL = kRedTile / 256 / W;  // loads per thread and tile
    const int tid = threadIdx.x;
    const int cols = kRedTile / rows, ls = cols + 4;
    const int64_t r0 = (int64_t)blockIdx.x * rows;
    // Load i of a thread is a fixed distance from its load 0: a tile row is cols / W loads, a
    // power of two, so 256 threads cover whole rows or a part of one.  The buffer range is the
    // check: rows past the end lie outside it (the whole distance is in the vector offset, which is
    // what the range bounds), columns past n are another row's or outside, and never folded.
    const int cw = cols / W, sh = 31 - __clz(cw);
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(x + r0 * n, min((int64_t)rows, nrows - r0) * n);
    const int row = cw < 256 ? tid >> sh : 0, col = (cw < 256 ? tid & (cw - 1) : tid) * W;
    const unsigned voff = (unsigned)(row * n + col) * 4u;
    float* const lp = tile + row * ls + col;
    float st[NL][W];
    auto load = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int di = cw < 256 ? i * (256 >> sh) : (i * 256) >> sh;  // rows from load 0
            const int dc = cw < 256 ? 0 : ((i * 256) & (cw - 1)) * W;
            const unsigned off = voff + (unsigned)(di * n + dc + c0) * 4u;
            if constexpr (VEC) {
                const f4v v = __builtin_bit_cast(f4v, __builtin_amdgcn_raw_buffer_load_b128(xr, off, 0, 0));
                st[i][0] = v.x; st[i][1] = v.y; st[i][2] = v.z; st[i][3] = v.w;
            } else {
                st[i][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, off, 0, 0));
            }
        }
    };
    load(0);
    float acc = init;
    for (int c0 = 0; c0 < n; c0 += cols) {
        __syncthreads();  // the previous tile has been folded
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int di = cw < 256 ? i * (256 >> sh) : (i * 256) >> sh;
            const int dc = cw < 256 ? 0 : ((i * 256) & (cw - 1)) * W;
            float* d = lp + di * ls + dc;
            if constexpr (VEC)
                *reinterpret_cast<float4*>(d) = make_float4(st[i][0], st[i][1], st[i][2], st[i][3]);
            else
                *d = st[i][0];
        }
        __syncthreads();
        if (c0 + cols < n) load(c0 + cols);
        if (tid < rows) {
            const float* t = tile + tid * ls;
            const int m = min(cols, n - c0);
            auto fold = [&](float4 v) __attribute__((always_inline)) {
                if constexpr (MAX) {
                    acc = fmaxf(fmaxf(fmaxf(fmaxf(acc, v.x), v.y), v.z), v.w);
                } else {
                    acc += v.x; acc += v.y; acc += v.z; acc += v.w;
                }
            };
            // 32 elements at a time, the next 32 read while these are folded
            int c = 0;
            if (m >= 32) {
                float4 a[8], b[8];
                auto read = [&](float4 (&d)[8], int at) __attribute__((always_inline)) {
                    const float* q = t + (at + 32 <= m ? at : 0);
#pragma unroll
                    for (int u = 0; u < 8; ++u) d[u] = *reinterpret_cast<const float4*>(q + 4 * u);
                    __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the adds
                };
                read(a, 0);
                for (; c + 64 <= m; c += 64) {
                    read(b, c + 32);
#pragma unroll
                    for (int u = 0; u < 8; ++u) fold(a[u]);
                    read(a, c + 64);
#pragma unroll
                    for (int u = 0; u < 8; ++u) fold(b[u]);
                }
                if (c + 32 <= m) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) fold(a[u]);
                    c += 32;
                }
            }
            for (; c + 4 <= m; c += 4) fold(*reinterpret_cast<const float4*>(t + c));
            for (; c < m; ++c) acc = MAX ? fmaxf(acc, t[c]) : acc + t[c];
        }
    }
    if (tid < rows && r0 + tid < nrows) y[r0 + tid] = acc;
}

// Outputs along a kept innermost axis, [outer][n][inner] -> [outer][inner], where there are too
// few outputs for a thread each to keep memory busy: a workgroup takes 64 adjacent outputs, its
// four wavefronts load every fourth element of the reduced axis, 16 deep, into LDS, and the first
// wavefront folds the 64 elements of each output in order while the next 64 load.
__global__ __launch_bounds__(256) void reduce_cols_kernel(const float* __restrict__ x,
                                                          float* __restrict__ y, int kind,
                                                          float init, int n, int inner,
                                                          int blocks) {
    __shared__ float tile[64 * 64];
    constexpr int NL = 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int outer = blockIdx.x / blocks, i0 = (blockIdx.x - outer * blocks) * 64;
    const bool ok = i0 + lane < inner;
    const float* xp = x + (int64_t)outer * n * inner + i0 + (ok ? lane : 0);
    float st[NL];
    auto load = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int r = r0 + i * 4 + wave;
            st[i] = ok && r < n ? xp[(int64_t)r * inner] : 0.0f;
        }
    };
    load(0);
    float acc = init;
    for (int r0 = 0; r0 < n; r0 += 64) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NL; ++i) tile[(i * 4 + wave) * 64 + lane] = st[i];
        __syncthreads();
        if (r0 + 64 < n) load(r0 + 64);
        if (wave == 0) {
            const int m = min(64, n - r0);
#pragma unroll 8
            for (int r = 0; r < m; ++r) {
                const float v = tile[r * 64 + lane];
                acc = kind ? fmaxf(acc, v) : acc + v;
            }
        }
    }
    if (wave == 0 && ok) y[(int64_t)outer * inner + i0 + lane] = acc;
}

// ---- hlo_strided_copy: push {r, total, dims[r], strides[r]}: out (row-major over dims) =
//      in0[sum_k c_k * strides[k]].  Materialises a strided view (a transpose, slice or
//      broadcast the HLO program kept as a view) into a contiguous tensor; in0 points at the
//      view's first element.  Strides >= 0 (0 on broadcast axes).
int launch_strided_copy(const shp::Launch& l) {
    const int32_t* q = l.push;
    const int r = q[0];
    if (r < 1 || r > kMaxRank) return shp::fail(SHP_ERR_SHAPE, "hlo_strided_copy: rank out of range 1..8");
    if ((int64_t)l.n_push < 2 + 2 * r) return shp::fail(SHP_ERR_PUSH, "hlo_strided_copy needs 2 + 2*r push constants");
    int dims[kMaxRank];
    int rc = read_dims(q + 2, r, dims, "hlo_strided_copy");
    if (rc) return rc;
    if (elems_of(dims, r) != q[1]) return shp::fail(SHP_ERR_SHAPE, "hlo_strided_copy: total != product of dims");
    rc = shp::check_total(l, q[1], "hlo_strided_copy");
    if (rc) return rc;
    Gather g{};
    g.r = r;
    for (int k = 0; k < r; ++k) {
        if (q[2 + r + k] < 0) return shp::fail(SHP_ERR_SHAPE, "hlo_strided_copy: negative stride");
        g.dims[k] = dims[k];
        g.stride[k] = q[2 + r + k];
    }
    return launch_gather(l, g);
}

int launch_reduce_nd(const shp::Launch& l) {
    const int32_t* q = l.push;
    const int r = q[1];
    if (r < 1 || r > kMaxRank) return shp::fail(SHP_ERR_SHAPE, "hlo_reduce: rank out of range 1..8");
    if ((int64_t)l.n_push < 4 + 2 * r) return shp::fail(SHP_ERR_PUSH, "hlo_reduce needs 4 + 2*r push constants");
    if (q[0] != 0 && q[0] != 1) return shp::fail(SHP_ERR_INVALID, "hlo_reduce: kind 0 (sum) or 1 (max)");
    int sd[kMaxRank];
    int rc = read_dims(q + 4, r, sd, "hlo_reduce");
    if (rc) return rc;
    Red p{};
    p.kind = q[0];
    std::memcpy(&p.init, &q[3], sizeof(float));
    int64_t sst[kMaxRank];
    strides_of(sd, r, sst);
    p.rcount = 1;
    int64_t kept = 1;
    // Axes in order, neighbours of one kind merged into one (sizes of 1 belong to either), which
    // leaves the fold order and the output layout as they are.
    int64_t outer = 1, inner = 1;  // kept elements before and after the reduced axes
    int last = -1;                 // kind of the axis before: 1 reduced, 0 kept
    for (int k = 0; k < r; ++k) {
        const int red = q[4 + r + k] ? 1 : 0;
        if (!red) kept *= sd[k];
        else p.rcount *= sd[k];
        if (sd[k] == 1) continue;
        int& cnt = red ? p.rr : p.rk;
        int* dims = red ? p.rdims : p.kdims;
        int64_t* st = red ? p.rstride : p.kstride;
        if (last == red && (int64_t)dims[cnt - 1] * sd[k] < (1ll << 31)) {
            dims[cnt - 1] *= sd[k];
        } else {
            dims[cnt] = sd[k];
            ++cnt;
        }
        st[cnt - 1] = sst[k];
        if (!red) (p.rr ? inner : outer) *= sd[k];
        last = red;
    }
    if (kept != q[2]) return shp::fail(SHP_ERR_SHAPE, "hlo_reduce: total != product of kept dims");
    rc = shp::check_total(l, q[2], "hlo_reduce");
    if (rc) return rc;
    // One reduced run: rows of contiguous elements go through LDS tiles (the fewest rows per
    // workgroup that still give every CU one), from 16 elements on, or 8 in 16-byte loads (30,000 rows
    // of 9 take 5.2 us so and 3.9 with a thread each).  Columns do where a thread per output, which
    // batches 16 loads, is short of them: up to 64 elements (16 x 40 x 130 over axis 1: 3.3 us
    // against 4.0; 16 x 200 x 130 8.4 against 6.9) or with so few columns in many places that its
    // loads hardly coalesce (300 x 200 x 2: 8.6 against 24; 16 of them 8.4 against 7.0), and not past 1,024 workgroups (30,000 x 40 x 2, two
    // lanes of a workgroup each: 30 us against 7.3).
    const float* x = (const float*)l.in0;
    float* y = (float*)l.out;
    const bool row_vec = p.rcount % 4 == 0 && ((uintptr_t)x & 15) == 0;
    if (p.rr == 1 && p.rk <= 1 && inner == 1 && p.rcount >= (row_vec ? 8 : 16)) {
        int rows = 256;
        while (rows > 4 && (outer + rows - 1) / rows < 256) rows /= 2;
        while (rows > 4 && rows * p.rcount >= (1ll << 28)) rows /= 2;  // 32-bit offsets
        const int64_t wgs = (outer + rows - 1) / rows;
        if (wgs < (1ll << 31) && rows * p.rcount < (1ll << 28)) {
            const int n = (int)p.rcount;
            auto kern = p.kind ? (row_vec ? reduce_rows_kernel<true, true> : reduce_rows_kernel<false, true>)
                               : (row_vec ? reduce_rows_kernel<true, false> : reduce_rows_kernel<false, false>);
            hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(256), 0, l.stream, x, y, p.init, outer,
                               n, rows);
            SHP_HIP_CHECK(hipGetLastError());
            return SHP_OK;
        }
    }
    const int64_t col_wgs = outer * ((inner + 63) / 64);
    if (p.rr == 1 && inner > 1 && p.rcount > 16 && col_wgs <= 1024 &&
        (p.rcount < 64 || (inner <= 3 && outer >= 64))) {
        const int blocks = (int)((inner + 63) / 64);
        hipLaunchKernelGGL(reduce_cols_kernel, dim3((unsigned)(outer * blocks)), dim3(256), 0,
                           l.stream, x, y, p.kind, p.init, (int)p.rcount, (int)inner, blocks);
        SHP_HIP_CHECK(hipGetLastError());
        return SHP_OK;
    }
    hipLaunchKernelGGL(reduce_nd_kernel, dim3(hlo_grid(l.out_elems)), dim3(kBlock), 0, l.stream,
                       x, y, p, l.out_elems);
    SHP_HIP_CHECK(hipGetLastError());
    return SHP_OK;
}

}  // namespace

namespace shp {

KernelEntry kHloOpKernels[] = {
    {"hlo_broadcast", 3, false, launch_broadcast},
    {"hlo_transpose", 2, false, launch_transpose_nd},
    {"hlo_slice", 2, false, launch_slice},
    {"hlo_concatenate_into", 3, false, launch_concatenate_into},
    {"hlo_compare", 5, false, launch_compare_select<false>},
    {"hlo_select", 4, false, launch_compare_select<true>},
    {"hlo_reduce", 4, false, launch_reduce_nd},
    {"hlo_strided_copy", 2, false, launch_strided_copy},
};
const int kHloOpKernelCount = sizeof(kHloOpKernels) / sizeof(kHloOpKernels[0]);

}  // namespace shp
