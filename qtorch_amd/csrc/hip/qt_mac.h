// Complex multiply-accumulate in the arithmetic forms of a contraction step.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qt {
namespace {

constexpr int kThreads = 256;

enum { MODE_PLAIN = 0, MODE_4M = 1, MODE_3M = 2, MODE_BF16X3 = 3 };

template <class V>
struct Real;
template <>
struct Real<double2> {
    using T = double;
};
template <>
struct Real<float2> {
    using T = float;
};

// Accumulator of one complex output.  The 3M form keeps the three real sums.
template <class V, int MODE>
struct Acc {
    using T = typename Real<V>::T;
    T re = 0, im = 0, p3 = 0;
};

__device__ __forceinline__ void mac_plain(Acc<double2, MODE_PLAIN>& acc, double2 a, double2 b) {
#pragma clang fp contract(off)
    // std::complex<double> product then +=, exactly as the reference evaluates it
    const double pr = a.x * b.x - a.y * b.y;
    const double pi = a.x * b.y + a.y * b.x;
    acc.re = acc.re + pr;
    acc.im = acc.im + pi;
}

__device__ __forceinline__ float bf16_round(float x) {
    // round-to-nearest-even to bfloat16, returned widened to float
    uint32_t u = __float_as_uint(x);
    const uint32_t lsb = (u >> 16) & 1u;
    u += 0x7fffu + lsb;
    u &= 0xffff0000u;
    return __uint_as_float(u);
}

template <class V, int MODE>
__device__ __forceinline__ void mac(Acc<V, MODE>& acc, V a, V b) {
    if constexpr (MODE == MODE_PLAIN) {
        mac_plain(acc, a, b);
    } else if constexpr (MODE == MODE_4M) {
        acc.re = fmaf(a.x, b.x, acc.re);
        acc.re = fmaf(-a.y, b.y, acc.re);
        acc.im = fmaf(a.x, b.y, acc.im);
        acc.im = fmaf(a.y, b.x, acc.im);
    } else if constexpr (MODE == MODE_3M) {
        acc.re = fmaf(a.x, b.x, acc.re);          // P1 = sum ar br
        acc.im = fmaf(a.y, b.y, acc.im);          // P2 = sum ai bi
        acc.p3 = fmaf(a.x + a.y, b.x + b.y, acc.p3);  // P3 = sum (ar+ai)(br+bi)
    } else {
        // bf16x3: x = hi + lo with hi, lo bfloat16; a*b ~ ah*bh + ah*bl + al*bh
        const float arh = bf16_round(a.x), arl = bf16_round(a.x - arh);
        const float aih = bf16_round(a.y), ail = bf16_round(a.y - aih);
        const float brh = bf16_round(b.x), brl = bf16_round(b.x - brh);
        const float bih = bf16_round(b.y), bil = bf16_round(b.y - bih);
        float re = acc.re, im = acc.im;
        re = fmaf(arh, brh, re); re = fmaf(arh, brl, re); re = fmaf(arl, brh, re);
        re = fmaf(-aih, bih, re); re = fmaf(-aih, bil, re); re = fmaf(-ail, bih, re);
        im = fmaf(arh, bih, im); im = fmaf(arh, bil, im); im = fmaf(arl, bih, im);
        im = fmaf(aih, brh, im); im = fmaf(aih, brl, im); im = fmaf(ail, brh, im);
        acc.re = re;
        acc.im = im;
    }
}

template <class V, int MODE>
__device__ __forceinline__ V finish(const Acc<V, MODE>& acc) {
    V r;
    if constexpr (MODE == MODE_3M) {
        r.x = acc.re - acc.im;
        r.y = acc.p3 - acc.re - acc.im;
    } else {
        r.x = acc.re;
        r.y = acc.im;
    }
    return r;
}

}  // namespace
}  // namespace qt
