// Quotients by a divisor known in advance.  Plain C++, shared by the kernels
// and their CPU checks.
#pragma once

#ifdef __HIPCC__
#define SSGPU_QUOT __host__ __device__ inline
#else
#define SSGPU_QUOT inline
#endif

namespace ssgpu {

// Operands of quot_from: neither the divisor nor the dividend beyond 2^400 nor
// below 2^-400 (the dividend may be zero), so that no intermediate leaves the
// normal range.
SSGPU_QUOT bool quot_divisor(double d) {
    const double a = __builtin_fabs(d);
    return (a >= 0x1p-400) & (a <= 0x1p400);
}
SSGPU_QUOT bool quot_dividend(double s) {
    const double a = __builtin_fabs(s);
    return (s == 0.0) | ((a >= 0x1p-400) & (a <= 0x1p400));
}
// s / d for y = 1 / d rounded to nearest: two Newton corrections of s * y, the
// second of which rounds correctly (P. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990, theorem 8.3).
SSGPU_QUOT double quot_from(double s, double d, double y) {
    const double q0 = s * y;
    const double q1 = __builtin_fma(__builtin_fma(-q0, d, s), y, q0);
    // the corrections of a zero keep its value but not its sign
    return __builtin_copysign(__builtin_fma(__builtin_fma(-q1, d, s), y, q1), q0);
}

}  // namespace ssgpu
