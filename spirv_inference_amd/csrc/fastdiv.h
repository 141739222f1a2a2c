// Division by a launch-constant divisor as a multiply-high and a shift: the index arithmetic of the
// strided kernels, where a 64-bit division per axis cost more than the memory access it served.
#pragma once
#include <hip/hip_runtime.h>

namespace shpd {

struct FastDiv {
    unsigned m, l, d;
};

inline FastDiv fast_div(unsigned d) {
    FastDiv f{0, 0, d};
    while ((1ull << f.l) < d) ++f.l;
    f.m = (unsigned)((((1ull << f.l) - d) << 32) / d + 1);
    return f;
}

// n / d for n < 2^31
__device__ __forceinline__ unsigned fdiv(unsigned n, const FastDiv& f) {
    return (__umulhi(n, f.m) + n) >> f.l;
}

}  // namespace shpd
