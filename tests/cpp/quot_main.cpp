// The kernels' quotient from a known reciprocal (ssgpu_quot.h) as they use it:
// operands outside its range take the division.  Returns how many it formed.
#include "ssgpu_quot.h"

extern "C" long quotients(long n, const double* s, const double* d, double* q) {
    long formed = 0;
    for (long i = 0; i < n; ++i) {
        const bool plain = ssgpu::quot_divisor(d[i]) & ssgpu::quot_dividend(s[i]);
        q[i] = plain ? ssgpu::quot_from(s[i], d[i], 1.0 / d[i]) : s[i] / d[i];
        formed += plain;
    }
    return formed;
}
