// quick_math.hpp -- division and indexing helpers of the device code (gfx950).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace gdtk {

// a / b correctly rounded from y = RN(1 / b): q = RN(a y) lies within an ulp of a / b, the
// remainder a - b q is exact in one fma, and RN(q + r y) is the correctly rounded quotient
// (Markstein's theorem; P. Markstein, IA-64 and Elementary Functions, 2000).  Bit for bit
// a / b for the normal operands met here; a true division costs ~10 instructions, this 3,
// and a divisor shared by several quotients needs its reciprocal once.
__host__ __device__ inline double div_by(double a, double b, double y) {
    const double q = a * y;
    const double r = fma(-b, q, a);
    return fma(r, y, q);
}

// a / b for normal operands: the hardware reciprocal refined by one cubic step (residual e:
// y (1 + e + e^2), relative error e^3), the quotient and one remainder correction: a / b within
// an ulp (the reciprocal is not always the rounded one).  A divisor of zero or infinity gives a
// NaN, where the division's result may be 0 or an infinity.  7 instructions, where the compiler's
// division takes 11 to scale operands that none of the quotients here needs scaled.
__device__ __forceinline__ double quick_rcp(double b) {
    const double y = __builtin_amdgcn_rcp(b);
    const double e = fma(-b, y, 1.0);
    return fma(y, fma(e, e, e), y);
}
__device__ __forceinline__ double quick_div(double a, double b) { return div_by(a, b, quick_rcp(b)); }

// Unsigned division by a divisor known on the host (Granlund & Montgomery, Division by
// Invariant Integers using Multiplication, 1994, the round-up multiplier): 4 instructions.
struct FastDiv {
    unsigned d, mul, shift;  // shift = ceil(log2 d) - 1, and 0 with mul = 0 for d = 1
    static FastDiv of(unsigned d) {
        FastDiv f{d, 0u, 0u};
        if (d <= 1) return f;
        unsigned l = 0;
        while (((uint64_t)1 << l) < d) ++l;
        f.mul = (unsigned)((((uint64_t)1 << 32) * (((uint64_t)1 << l) - d)) / d + 1);
        f.shift = l - 1;
        return f;
    }
    // n / d and the remainder
    __host__ __device__ unsigned divmod(unsigned n, unsigned& rem) const {
        unsigned q = n;
        if (d > 1) {
            const unsigned t = (unsigned)(((uint64_t)mul * n) >> 32);
            q = (t + ((n - t) >> 1)) >> shift;
        }
        rem = n - q * d;
        return q;
    }
};

// The index of the wave's first active lane: the origin that the lanes' 32-bit offsets count
// from, where a lane's index never is below that of a lane before it.
__device__ __forceinline__ unsigned wave_origin(unsigned i) { return (unsigned)__builtin_amdgcn_readfirstlane((int)i); }

// Element i of an array at a wave-uniform address: base in scalar registers, a 32-bit byte
// offset (i < 2^29: count it from wave_origin) and the global address space, so that the access
// needs one vector register for its address where a flat one needs two and their arithmetic.
__device__ __forceinline__ double ld_plane(const double* base, unsigned i) {
    typedef __attribute__((address_space(1))) const char* gptr;
    typedef __attribute__((address_space(1))) const double* dptr;
    return *(dptr)((gptr)base + i * 8u);
}
__device__ __forceinline__ void st_plane(double* base, unsigned i, double v) {
    typedef __attribute__((address_space(1))) char* gptr;
    typedef __attribute__((address_space(1))) double* dptr;
    *(dptr)((gptr)base + i * 8u) = v;
}

}  // namespace gdtk
