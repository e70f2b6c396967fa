// fft_device.hpp -- complex FP64 transforms of a workgroup's lines in LDS.
//
// Stockham passes (no bit reversal): radix 5, 4, 3 and 2 butterflies in
// registers and a direct sum for any other prime, so that every length works.
// A workgroup holds a line or a few, so a pass lasts as long as one lane's
// butterfly: 1500 cycles at radix 4 and 2200 at radix 8, whose 273 instructions
// leave 7 of 8 lanes idle on a line of 64.  Lines sit in LDS `ld` elements
// apart with one element of padding in nine, which keeps the strided stores of
// a first pass off each other's banks.  On this card an FP64 multiply-add costs
// what an FP32 one does.
#pragma once
#include "aw_internal.hpp"

namespace aw::fft {

__device__ __forceinline__ int pad(int i) { return i + (i >> 3); }

// a / d for a, d < 2^20 by the FP32 reciprocal r of d: (a + 1/2) / d keeps 1 / (2 d)
// from every integer, far beyond the product's rounding
__device__ __forceinline__ int div_by(int a, float r) { return (int)(((float)a + 0.5f) * r); }

// one pass: radix r after the passes of product ns; m = n / r butterflies,
// twiddle stride st = n / (ns r)
struct Pass {
    int r, ns, st, m;
    float inv_ns, inv_m;
};

__device__ __forceinline__ double2 operator+(double2 a, double2 b) {
    return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 operator-(double2 a, double2 b) {
    return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
// a * (S i)
template <int S>
__device__ __forceinline__ double2 mul_i(double2 a) {
    return S > 0 ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// v[k] = sum_s v[s] exp(S 2 pi i s k / R)
template <int R, int S>
__device__ __forceinline__ void dft(double2 (&v)[R]) {
    if constexpr (R == 2) {
        const double2 a = v[0] + v[1];
        v[1] = v[0] - v[1];
        v[0] = a;
    } else if constexpr (R == 3) {
        constexpr double kS = 0.86602540378443864676;  // sin(2 pi / 3)
        const double2 t = v[1] + v[2], d = v[1] - v[2];
        const double2 m = make_double2(fma(-0.5, t.x, v[0].x), fma(-0.5, t.y, v[0].y));
        const double2 r = mul_i<S>(make_double2(kS * d.x, kS * d.y));
        v[0] = v[0] + t;
        v[1] = m + r;
        v[2] = m - r;
    } else if constexpr (R == 4) {
        const double2 a = v[0] + v[2], b = v[0] - v[2], c = v[1] + v[3],
                      d = mul_i<S>(v[1] - v[3]);
        v[0] = a + c;
        v[1] = b + d;
        v[2] = a - c;
        v[3] = b - d;
    } else {
        static_assert(R == 5);
        constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
        constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
        const double2 t1 = v[1] + v[4], t2 = v[2] + v[3], d1 = v[1] - v[4], d2 = v[2] - v[3];
        const double2 m1 = make_double2(fma(c2, t2.x, fma(c1, t1.x, v[0].x)),
                                        fma(c2, t2.y, fma(c1, t1.y, v[0].y)));
        const double2 m2 = make_double2(fma(c1, t2.x, fma(c2, t1.x, v[0].x)),
                                        fma(c1, t2.y, fma(c2, t1.y, v[0].y)));
        const double2 r1 = mul_i<S>(make_double2(fma(s2, d2.x, s1 * d1.x), fma(s2, d2.y, s1 * d1.y)));
        const double2 r2 = mul_i<S>(make_double2(fma(-s1, d2.x, s2 * d1.x), fma(-s1, d2.y, s2 * d1.y)));
        v[0] = v[0] + t1 + t2;
        v[1] = m1 + r1;
        v[2] = m2 + r2;
        v[3] = m2 - r2;
        v[4] = m1 - r1;
    }
}

template <int S>
__device__ __forceinline__ double2 twiddle(const double2* tw, int i) {
    const double2 w = tw[i];  // exp(-2 pi i i / n)
    return S > 0 ? make_double2(w.x, -w.y) : w;
}

template <int R, int S>
__device__ __forceinline__ void pass(const double2* src, double2* dst, const Pass& p,
                                     const double2* tw, int lines, int ld) {
    const int total = lines * p.m;
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        const int line = div_by(t, p.inv_m), b = t - line * p.m;
        const int q = div_by(b, p.inv_ns), k = b - q * p.ns;
        const double2* a = src + line * ld;
        double2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = a[pad(b + r * p.m)];
        if (p.ns > 1) {
            // powers of one twiddle, each of the two before it in half the steps
            double2 w[R];
            w[1] = twiddle<S>(tw, k * p.st);
#pragma unroll
            for (int r = 2; r < R; ++r) w[r] = cmul(w[r / 2], w[r - r / 2]);
#pragma unroll
            for (int r = 1; r < R; ++r) v[r] = cmul(v[r], w[r]);
        }
        dft<R, S>(v);
        double2* o = dst + line * ld;
        const int base = q * p.ns * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) o[pad(base + r * p.ns)] = v[r];
    }
}

// one output a thread, a sum of p.r terms: the prime factors without a butterfly
template <int S>
__device__ __forceinline__ void pass_any(const double2* src, double2* dst, const Pass& p,
                                         const double2* tw, int n, int lines, int ld) {
    const int total = lines * n;
    const float inv_n = 1.0f / (float)n;
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        const int line = div_by(t, inv_n), o = t - line * n;
        const int r = div_by(o, p.inv_m), b = o - r * p.m;
        const int q = div_by(b, p.inv_ns), k = b - q * p.ns;
        const double2* a = src + line * ld;
        int step = k * p.st + r * p.m;
        if (step >= n) step -= n;
        double2 acc = a[pad(b)];
        int i = 0;
        for (int s = 1; s < p.r; ++s) {
            i += step;
            if (i >= n) i -= n;
            const double2 w = twiddle<S>(tw, i), v = a[pad(b + s * p.m)];
            acc.x = fma(v.x, w.x, fma(-v.y, w.y, acc.x));
            acc.y = fma(v.x, w.y, fma(v.y, w.x, acc.y));
        }
        dst[line * ld + pad(q * p.ns * p.r + k + r * p.ns)] = acc;
    }
}

// Transforms the lines at a (b: as much scratch) with exp(S 2 pi i ..), tw their
// twiddles in LDS; the result is in the buffer returned.  Every thread calls it, after a barrier
// that follows the lines' writes; it ends with a barrier.
template <int S>
__device__ __forceinline__ double2* lines(double2* a, double2* b, const FftLine& l,
                                          const double2* tw, int nlines, int ld) {
    unsigned long long radices = l.radices;
    int ns = 1;
    for (int i = 0; i < l.npass; ++i, radices >>= 8) {
        Pass p;
        p.r = (int)(radices & 255);
        p.ns = ns;
        p.m = div_by(l.n, 1.0f / (float)p.r);
        p.inv_ns = 1.0f / (float)ns;
        p.inv_m = 1.0f / (float)p.m;
        p.st = div_by(p.m, p.inv_ns);
        ns *= p.r;
        switch (p.r) {
            case 2: pass<2, S>(a, b, p, tw, nlines, ld); break;
            case 3: pass<3, S>(a, b, p, tw, nlines, ld); break;
            case 4: pass<4, S>(a, b, p, tw, nlines, ld); break;
            case 5: pass<5, S>(a, b, p, tw, nlines, ld); break;
            default: pass_any<S>(a, b, p, tw, l.n, nlines, ld); break;
        }
        __syncthreads();
        double2* t = a;
        a = b;
        b = t;
    }
    return a;
}

}  // namespace aw::fft
