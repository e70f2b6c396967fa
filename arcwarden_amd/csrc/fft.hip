// fft.hip -- the spectral solves on the library's own transforms.
//
// A solve is three launches: rows forward, columns (forward, the k-space
// algebra, inverse) and rows inverse, with what used to be launches of its own
// fused in: the conversion of the fixed-point accumulators into the first, the
// Green's functions (include/pic/solver_es.hpp:39-78, solver_darwin.hpp:38-129)
// into the second, the field combination, pump and field maxima into the
// third.  Two real lines share a complex one (a + i b), so every length, odd
// ones too, takes the same code.  Lines are transformed in LDS in FP64
// (fft_device.hpp); between the launches the half spectra are FP32, as the
// k-space arrays of the rocFFT solves are.
//
// The solves are bound by latency, not by bytes or operations: about 2.5 us a
// launch until the first loads are back, 0.7 us a pass, three to four launches
// a step where rocFFT's took six (sides of 2^n) to nineteen (a prime factor
// above 17).  A step with two markers a cell, electrostatic / Darwin, us:
// 64x64 24 / 60 (rocFFT 25 / 71), 60x48 25 / 64 (36 / 118), 125x100 27 / 68
// (47 / 116), 190x250 33 / 94 (54 / 142), 256x256 30 / 99 (32 / 106), 300x300
// 32 / 104 (49 / 149), 600x384 43 / 174 (54 / 194), 61x61 40 / 112 (82 / 200).
// Where rocFFT is ahead the solves stay with it: ahead(), below.
#include "fft_device.hpp"

#include <algorithm>
#include <cmath>
#include <functional>
#include <vector>

namespace aw {

using namespace fft;

namespace {

constexpr double kTwoPi = 6.28318530717958647692;

struct KGeom {
    int nx, ny, nkx;
    double dkx, dky;
    const double2 *hx, *hy;  // half-cell phases exp(i pi k / n), k <= n / 2
};

KGeom geom(const aw_ctx& c) {
    const double2* h = c.fft_tw.get() + c.g.nx + c.g.ny;
    return {c.g.nx, c.g.ny, c.g.nx / 2 + 1, kTwoPi / c.g.Lx, kTwoPi / c.g.Ly, h, h + c.g.nx / 2 + 1};
}

// Grid q is paired with grid q + 1 row by row, the last of an odd number with
// itself, two rows at a time.
struct Pair {
    int q0, j0, q1, j1;
    bool two;
};

__device__ __forceinline__ Pair pair_of(int p, int nq, int ny) {
    if (nq == 2) return {0, p, 1, p, true};
    const int whole = (nq >> 1) * ny;
    if (p < whole) {
        const int a = p / ny, j = p - a * ny;
        return {2 * a, j, 2 * a + 1, j, true};
    }
    const int j = 2 * (p - whole);
    return {nq - 1, j, nq - 1, j + 1, j + 1 < ny};
}

int pair_count(int nq, int ny) { return (nq / 2) * ny + (nq % 2) * ((ny + 1) / 2); }

int line_ld(int n) { return n + (n >> 3) + 1; }

// Static LDS of the row kernels, beside their lines and twiddles: lines_set's
// word a wavefront and (kFormEl) the two floats a wavefront of block_max2.
constexpr int kMaxWaves = 16;
constexpr size_t kRowsStaticLds = kMaxWaves * (sizeof(int) + 2 * sizeof(float));

// What a workgroup's two lines hold: bit 0 and 1 something, bit 2 and 3 a value
// that is not finite.  A line of zeros comes out as zeros, not as the rounding
// of its partner.  Every thread calls it; a barrier is inside.
constexpr int kNotFinite = 4;
__device__ __forceinline__ int lines_set(bool a, bool b, bool bada = false, bool badb = false) {
    __shared__ int s_set[kMaxWaves];
    const int m = (__ballot(a) ? 1 : 0) | (__ballot(b) ? 2 : 0) |
                  (__ballot(bada) ? kNotFinite : 0) | (__ballot(badb) ? 2 * kNotFinite : 0);
    if ((threadIdx.x & 63) == 0) s_set[threadIdx.x >> 6] = m;
    __syncthreads();
    int all = 0;
    for (int w = 0; w < (int)((blockDim.x + 63) >> 6); ++w) all |= s_set[w];
    return all;
}

// A cell of grid q: its accumulator or FP32 value, and where both go.
struct Cell {
    const SpecSrc& a;
    int64_t nc;
    int r, q;
    bool first;
    __device__ __forceinline__ Cell(const SpecSrc& a_, int64_t nc_, int r_, int q_)
        : a(a_), nc(nc_), r(r_), q(q_), first(q_ < a_.split) {}
    __device__ __forceinline__ unsigned long long* acc(int64_t c) const {
        return first ? a.acc + r * a.acc_rs + q * nc + c : a.acc2 + r * a.acc2_rs + (q - a.split) * nc + c;
    }
    __device__ __forceinline__ double inv() const {
        return a.inv ? a.inv[r * a.inv_rs + q + (first ? a.inv_a : a.inv_b)] : a.inv0;
    }
    __device__ __forceinline__ long long base(int64_t c) const {
        if (q != 0) return 0;
        return a.base ? a.base[a.base_cell ? r * a.out_rs + c : r] : a.base_val;
    }
    // the cell's value into the FP32 grid, its accumulator cleared
    __device__ __forceinline__ void take(int64_t c, long long v, double s) const {
        *acc(c) = 0ull;
        a.out[r * a.out_rs + (q + (first ? a.out_a : a.out_b)) * nc + c] = (float)((double)v * s);
    }
    __device__ __forceinline__ float in(int64_t c) const { return a.in[r * a.in_rs + q * nc + c]; }
};

// Rows forward: a pair of rows as one complex line, ks[r][q][j][k] for k < nkx.
// The kernels load a thread's first elements and twiddles before they store any
// of them (elements past the end load the last one), so that one memory
// latency covers them all.
constexpr int kAhead = 2;

template <bool ACC, int NQ>
__global__ void __launch_bounds__(1024)
rows_forward_kernel(SpecSrc a, FftLine fx, int ny, float2* __restrict__ ks) {
    extern __shared__ double2 s_tw[];
    double2* s_l = s_tw + fx.ntw;
    const int nx = fx.n, nkx = nx / 2 + 1, ld = nx + (nx >> 3) + 1, r = blockIdx.y;
    const int nt = blockDim.x, tid = threadIdx.x;
    const int64_t nc = (int64_t)nx * ny;
    const Pair p = pair_of(blockIdx.x, NQ, ny);
    const Cell ca(a, nc, r, p.q0), cb(a, nc, r, p.q1);
    const int64_t ra = (int64_t)p.j0 * nx, rb = p.two ? (int64_t)p.j1 * nx : ra;
    bool seta = false, setb = false, bada = false, badb = false;
    const double2 w0 = fx.tw[min(tid, nx - 1)];
    if constexpr (ACC) {
        const double sa = ca.inv(), sb = cb.inv();
        for (int x0 = 0; x0 < nx; x0 += kAhead * nt) {
            long long va[kAhead], vb[kAhead], ba[kAhead], bb[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int x = min(x0 + u * nt + tid, nx - 1);
                va[u] = (long long)*ca.acc(ra + x);
                vb[u] = (long long)*cb.acc(rb + x);
                ba[u] = ca.base(ra + x);
                bb[u] = cb.base(rb + x);
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int x = x0 + u * nt + tid;
                if (x >= nx) continue;
                ca.take(ra + x, va[u], sa);
                if (p.two) cb.take(rb + x, vb[u], sb);
                const double2 v = make_double2((double)(va[u] - ba[u]) * sa,
                                               p.two ? (double)(vb[u] - bb[u]) * sb : 0.0);
                seta = seta || v.x != 0.0;
                setb = setb || v.y != 0.0;
                s_l[pad(x)] = v;
            }
        }
        if (blockIdx.x == 0 && r == 0)
            for (int i = tid; i < a.ncounter; i += nt) a.counter[i] = 0ull;
    } else {
        for (int x0 = 0; x0 < nx; x0 += kAhead * nt) {
            float va[kAhead], vb[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int x = min(x0 + u * nt + tid, nx - 1);
                va[u] = ca.in(ra + x);
                vb[u] = cb.in(rb + x);
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int x = x0 + u * nt + tid;
                if (x >= nx) continue;
                double2 v = make_double2(va[u], p.two ? vb[u] : 0.f);
                seta = seta || v.x != 0.0;
                setb = setb || v.y != 0.0;
                // infinities and NaN stay out of the line they would share
                if (!isfinite(v.x)) bada = true, v.x = 0.0;
                if (!isfinite(v.y)) badb = true, v.y = 0.0;
                s_l[pad(x)] = v;
            }
        }
    }
    if (tid < fx.ntw) s_tw[tid] = w0;
    for (int i = tid + nt; i < fx.ntw; i += nt) s_tw[i] = fx.tw[i];
    const int set = lines_set(seta, setb, bada, badb);
    const double2* z = lines<-1>(s_l, s_l + ld, fx, s_tw, 1, ld);
    float2* k0 = ks + (((int64_t)r * NQ + p.q0) * ny + p.j0) * nkx;
    float2* k1 = ks + (((int64_t)r * NQ + p.q1) * ny + p.j1) * nkx;
    // a line that is not finite has no finite mode; its partner is its own
    const float2 zero = make_float2(0.f, 0.f), none = make_float2(NAN, NAN);
    for (int k = tid; k < nkx; k += nt) {
        const double2 u = z[pad(k)], w = z[pad(k ? nx - k : 0)];
        // the transforms of a and b out of that of a + i b
        const float2 A = make_float2((float)(0.5 * (u.x + w.x)), (float)(0.5 * (u.y - w.y)));
        const float2 B = make_float2((float)(0.5 * (u.y + w.y)), (float)(0.5 * (w.x - u.x)));
        k0[k] = set & kNotFinite ? none : set & 1 ? A : zero;
        if (p.two) k1[k] = set & 2 * kNotFinite ? none : set & 2 ? B : zero;
    }
}

// ---- the k-space algebra, one mode (i, j) -------------------------------------------

struct Mode {
    double kx, ky, k2;
    bool nyq;
    int i, j;
};

__device__ __forceinline__ Mode mode_of(const KGeom& g, int i, int j) {
    const int m = j <= g.ny / 2 ? j : j - g.ny;
    Mode k;
    k.kx = i * g.dkx;
    k.ky = m * g.dky;
    k.k2 = k.kx * k.kx + k.ky * k.ky;
    k.nyq = ((g.nx % 2 == 0) && i == g.nx / 2) || ((g.ny % 2 == 0) && j == g.ny / 2);
    k.i = i;
    k.j = m;
    return k;
}

// phi_k = rho_k / (eps0 k^2), E_k = -i k phi_k; DC and Nyquist zero
// (es_poisson_field_kernel)
struct OpEs {
    static constexpr int kIn = 1, kOut = 2;
    double eps0;
    __device__ __forceinline__ void operator()(const KGeom&, const Mode& k, const double2* in,
                                               double2* out) const {
        const double g = k.k2 > 0.0 && !k.nyq ? 1.0 / (eps0 * k.k2) : 0.0;
        const double pr = in[0].x * g, pi = in[0].y * g;
        out[0] = make_double2(k.kx * pi, -k.kx * pr);
        out[1] = make_double2(k.ky * pi, -k.ky * pr);
    }
};

// its transpose: lrho_k = i g (kx lEx_k + ky lEy_k)
struct OpEsAdj {
    static constexpr int kIn = 2, kOut = 1;
    double eps0;
    __device__ __forceinline__ void operator()(const KGeom&, const Mode& k, const double2* in,
                                               double2* out) const {
        const double g = k.k2 > 0.0 && !k.nyq ? 1.0 / (eps0 * k.k2) : 0.0;
        out[0] = make_double2(-g * (k.kx * in[0].y + k.ky * in[1].y),
                              g * (k.kx * in[0].x + k.ky * in[1].x));
    }
};

// E_L and B_k = i mu0 (k x J) / k^2 from [rho|Jx|Jy|Jz] (darwin_b_field_kernel);
// B0 is B's DC mode.  stag: Jx, Jy sampled half a cell off the nodes.
struct OpElb {
    static constexpr int kIn = 4, kOut = 5;
    double eps0, c;
    float b0[3];
    int stag;
    __device__ __forceinline__ void operator()(const KGeom& g, const Mode& k, const double2* in,
                                               double2* out) const {
        double2 jx = in[1], jy = in[2];
        const double2 jz = in[3];
        if (stag) {
            const double2 hx = g.hx[k.i], hy = g.hy[k.j < 0 ? -k.j : k.j];
            const double cx = hx.x, sx = hx.y, cy = hy.x, sy = k.j < 0 ? -hy.y : hy.y;
            jx = make_double2(in[1].x * cx + in[1].y * sx, in[1].y * cx - in[1].x * sx);
            jy = make_double2(in[2].x * cy + in[2].y * sy, in[2].y * cy - in[2].x * sy);
        }
        const bool on = k.k2 > 0.0 && !k.nyq;
        const double e = on ? 1.0 / (eps0 * k.k2) : 0.0;
        const double G = e / (c * c);
        const double pr = in[0].x * e, pi = in[0].y * e;
        out[0] = make_double2(k.kx * pi, -k.kx * pr);
        out[1] = make_double2(k.ky * pi, -k.ky * pr);
        out[2] = make_double2(-G * k.ky * jz.y, G * k.ky * jz.x);
        out[3] = make_double2(G * k.kx * jz.y, -G * k.kx * jz.x);
        out[4] = make_double2(-G * (k.kx * jy.y - k.ky * jx.y), G * (k.kx * jy.x - k.ky * jx.x));
        if (k.i == 0 && k.j == 0) {
            const double nn = (double)g.nx * (double)g.ny;
#pragma unroll
            for (int q = 0; q < 3; ++q) out[2 + q] = make_double2((double)b0[q] * nn, 0.0);
        }
    }
};

// dJ/dt = dcu - i S(amu), its transverse part, E_T = -G (dJ/dt)_T with
// G = 1 / (eps0 c^2 k^2 + n0) (darwin_et_kernel)
struct OpEt {
    static constexpr int kIn = 7, kOut = 3;
    double eps0, c, n0;
    __device__ __forceinline__ void operator()(const KGeom&, const Mode& k, const double2* in,
                                               double2* out) const {
        const bool on = k.k2 > 0.0 && !k.nyq;
        const double G = on ? 1.0 / (eps0 * c * c * k.k2 + n0) : 0.0;
        const double inv = on ? 1.0 / k.k2 : 0.0;
        const double2 a0 = in[3], a1 = in[4], a2 = in[5], a3 = in[6];
        const double Sxr = k.kx * a0.x + k.ky * a1.x, Sxi = k.kx * a0.y + k.ky * a1.y;
        const double Syr = k.kx * a1.x - k.ky * a0.x, Syi = k.kx * a1.y - k.ky * a0.y;
        const double Szr = k.kx * a2.x + k.ky * a3.x, Szi = k.kx * a2.y + k.ky * a3.y;
        double Jxr = in[0].x + Sxi, Jxi = in[0].y - Sxr;
        double Jyr = in[1].x + Syi, Jyi = in[1].y - Syr;
        const double Jzr = in[2].x + Szi, Jzi = in[2].y - Szr;
        const double kdr = (k.kx * Jxr + k.ky * Jyr) * inv, kdi = (k.kx * Jxi + k.ky * Jyi) * inv;
        Jxr -= k.kx * kdr;
        Jxi -= k.kx * kdi;
        Jyr -= k.ky * kdr;
        Jyi -= k.ky * kdi;
        out[0] = make_double2(-G * Jxr, -G * Jxi);
        out[1] = make_double2(-G * Jyr, -G * Jyi);
        out[2] = make_double2(-G * Jzr, -G * Jzi);
    }
};

// Columns: C neighbouring kx (1 << clog) of every input grid transformed along
// y, the algebra, every output grid transformed back.  smax (OpEsAdj): slots of
// the largest |Re| + |Im| of the output modes (FP32 bit patterns).
template <class Op>
__global__ void __launch_bounds__(512)
columns_kernel(const float2* __restrict__ kin, float2* __restrict__ kout, KGeom g, FftLine fy,
               int clog, Op op, unsigned int* __restrict__ smax) {
    extern __shared__ double2 s_tw[];
    double2* s_l = s_tw + fy.ntw;
    constexpr int NI = Op::kIn, NO = Op::kOut, NM = NI > NO ? NI : NO;
    const int C = 1 << clog, ny = g.ny, ld = ny + (ny >> 3) + 1, r = blockIdx.y;
    const int k0 = blockIdx.x << clog;
    const int64_t nk = (int64_t)g.nkx * ny;
    double2 *a = s_l, *b = s_l + NM * C * ld;
    const int nt = blockDim.x, cells = ny << clog;
    const double2 w0 = fy.tw[min((int)threadIdx.x, ny - 1)];
    for (int t0 = 0; t0 < cells; t0 += nt) {
        const int t = min(t0 + (int)threadIdx.x, cells - 1), c = t & (C - 1), j = t >> clog;
        // columns past the last kx repeat it; they are not stored
        const float2* in = kin + (int64_t)r * NI * nk + (int64_t)j * g.nkx + min(k0 + c, g.nkx - 1);
        float2 v[NI];
#pragma unroll
        for (int q = 0; q < NI; ++q) v[q] = in[q * nk];
#pragma unroll
        for (int q = 0; q < NI; ++q) a[(q * C + c) * ld + pad(j)] = make_double2(v[q].x, v[q].y);
    }
    if ((int)threadIdx.x < fy.ntw) s_tw[threadIdx.x] = w0;
    for (int i = threadIdx.x + nt; i < fy.ntw; i += nt) s_tw[i] = fy.tw[i];
    __syncthreads();
    double2* z = lines<-1>(a, b, fy, s_tw, NI * C, ld);
    double2* o = z == a ? b : a;
    float top = 0.f;
    for (int t = threadIdx.x; t < (ny << clog); t += blockDim.x) {
        const int c = t & (C - 1), j = t >> clog, at = c * ld + pad(j);
        double2 in[NI], out[NO];
#pragma unroll
        for (int q = 0; q < NI; ++q) in[q] = z[q * C * ld + at];
        op(g, mode_of(g, min(k0 + c, g.nkx - 1), j), in, out);
#pragma unroll
        for (int q = 0; q < NO; ++q) o[q * C * ld + at] = out[q];
        if (NO == 1 && k0 + c < g.nkx)
            top = fmaxf(top, fabsf((float)out[0].x) + fabsf((float)out[0].y));
    }
    if (NO == 1 && smax) {
        for (int d = 32; d > 0; d >>= 1) top = fmaxf(top, __shfl_xor(top, d, 64));
        if ((threadIdx.x & 63) == 0 && top > 0.f)
            atomicMax(smax + (blockIdx.x % kSpecSlots) * kSpecSlotStride, __float_as_uint(top));
    }
    __syncthreads();
    o = lines<1>(o, z, fy, s_tw, NO * C, ld);
    for (int q = 0; q < NO; ++q)
        for (int t = threadIdx.x; t < (ny << clog); t += blockDim.x) {
            const int c = t & (C - 1), j = t >> clog;
            if (k0 + c >= g.nkx) continue;
            const double2 v = o[(q * C + c) * ld + pad(j)];
            kout[((int64_t)r * NO + q) * nk + (int64_t)j * g.nkx + k0 + c] =
                make_float2((float)v.x, (float)v.y);
        }
}

// one value of output grid q at cell c (column x) of run r, and what is formed of it
template <int FORM>
__device__ __forceinline__ void emit(const SpecDst& d, int r, int q, int64_t c, int64_t nc, float v,
                                     const float (&pump)[3], bool pumped, float& me, float& mb) {
    (q == 0 ? d.out : d.out1 + (q - 1) * nc)[r * d.out_rs + c] = v;
    if constexpr (FORM == SpecDst::kFormEl) {
        if (q >= 2) {
            mb = fmaxf(mb, fabsf(v));
            return;
        }
        const float e = pumped ? v + pump[q] : v;
        d.e[r * d.e_rs + q * nc + c] = e;
        me = fmaxf(me, fabsf(e));
        if (q == 0) {
            const float ez = pumped ? 0.0f + pump[2] : 0.0f;
            d.e[r * d.e_rs + 2 * nc + c] = ez;
            me = fmaxf(me, fabsf(ez));
        }
    } else if constexpr (FORM == SpecDst::kFormEt) {
        float e = q < 2 ? d.el[r * d.el_rs + q * nc + c] + v : v;
        if (pumped) e += pump[q];
        d.e[r * d.e_rs + q * nc + c] = e;
    }
}

// Rows inverse: two half spectra A, B as the line A + i B, its real part the
// one row and its imaginary part the other.
template <int NQ, int FORM>
__global__ void __launch_bounds__(1024)
rows_inverse_kernel(const float2* __restrict__ ks, FftLine fx, int ny, double scale, SpecDst d) {
    extern __shared__ double2 s_tw[];
    double2* s_l = s_tw + fx.ntw;
    const int nx = fx.n, nkx = nx / 2 + 1, ld = nx + (nx >> 3) + 1, r = blockIdx.y;
    const int nt = blockDim.x, tid = threadIdx.x;
    const int64_t nc = (int64_t)nx * ny;
    const Pair p = pair_of(blockIdx.x, NQ, ny);
    const float2* k0 = ks + (((int64_t)r * NQ + p.q0) * ny + p.j0) * nkx;
    const float2* k1 = p.two ? ks + (((int64_t)r * NQ + p.q1) * ny + p.j1) * nkx : k0;
    const double2 w0 = fx.tw[min(tid, nx - 1)];
    bool seta = false, setb = false;
    for (int i0 = 0; i0 < nkx; i0 += kAhead * nt) {
        float2 va[kAhead], vb[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = min(i0 + u * nt + tid, nkx - 1);
            va[u] = k0[k];
            vb[u] = k1[k];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int k = i0 + u * nt + tid;
            if (k >= nkx) continue;
            float2 A = va[u], B = p.two ? vb[u] : make_float2(0.f, 0.f);
            const bool real = k == 0 || 2 * k == nx;
            if (real) A.y = B.y = 0.f;  // a real line's DC and Nyquist
            seta = seta || A.x != 0.f || A.y != 0.f;
            setb = setb || B.x != 0.f || B.y != 0.f;
            s_l[pad(k)] = make_double2((double)A.x - B.y, (double)A.y + B.x);
            if (!real) s_l[pad(nx - k)] = make_double2((double)A.x + B.y, (double)B.x - A.y);
        }
    }
    if (tid < fx.ntw) s_tw[tid] = w0;
    for (int i = tid + nt; i < fx.ntw; i += nt) s_tw[i] = fx.tw[i];
    const int set = lines_set(seta, setb);
    const double2* z = lines<1>(s_l, s_l + ld, fx, s_tw, 1, ld);
    const bool pumped = FORM != SpecDst::kPlain && d.pump.on && d.pump.t < d.pump.toff;
    float me = 0.f, mb = 0.f;
    for (int x = tid; x < nx; x += nt) {
        const double2 v = z[pad(x)];
        float pump[3] = {0.f, 0.f, 0.f};
        if (pumped && (FORM == SpecDst::kFormEt || p.q0 < 2))
            dev::pump_at(d.pump, x, pump[0], pump[1], pump[2]);
        emit<FORM>(d, r, p.q0, (int64_t)p.j0 * nx + x, nc, set & 1 ? (float)(v.x * scale) : 0.f,
                   pump, pumped, me, mb);
        if (p.two)
            emit<FORM>(d, r, p.q1, (int64_t)p.j1 * nx + x, nc, set & 2 ? (float)(v.y * scale) : 0.f,
                       pump, pumped, me, mb);
    }
    if constexpr (FORM == SpecDst::kFormEl) {
        dev::block_max2(me, mb);
        if (tid == 0) {
            float* o = d.part + 2 * ((int64_t)r * gridDim.x + blockIdx.x);
            o[0] = me;
            o[1] = mb;
        }
    }
}

// Factors n for the line transforms; false past the largest prime whose direct
// sum was measured ahead of rocFFT's convolution (97x80, above it, takes 47 us
// a step there).  direct: the terms of the direct sums are added to it.
constexpr int kMaxPrime = 61;
bool make_line(int n, FftLine& l, int& direct) {
    int f[64], nf = 0, m = n;
    for (; m % 4 == 0; m /= 4) f[nf++] = 4;
    for (; m % 2 == 0; m /= 2) f[nf++] = 2;
    for (int p = 3; m > 1; p += 2)
        for (; m % p == 0; m /= p) {
            if (p > kMaxPrime || nf >= 40) return false;
            f[nf++] = p;
        }
    if (nf > FftLine::kMaxPass) return false;
    std::sort(f, f + nf, std::greater<int>());
    l.n = n;
    l.npass = nf;
    l.radices = 0;
    l.ntw = 0;
    int ns = 1;
    for (int i = 0; i < nf; ++i) {
        const int r = f[i];
        l.radices |= (unsigned long long)r << (8 * i);
        // a butterfly takes powers of one twiddle, a direct sum any of them
        const bool fly = r <= 5;
        if (!fly) direct += r;
        l.ntw = std::max(l.ntw, ns == 1 && fly ? 0 : fly ? n / r : n);
        ns *= r;
    }
    return true;
}

size_t rows_lds(const aw_ctx& c) {
    return ((size_t)2 * line_ld(c.g.nx) + c.fx.ntw) * sizeof(double2);
}
size_t columns_lds(const aw_ctx& c, int nmax, int C) {
    return ((size_t)2 * nmax * C * line_ld(c.g.ny) + c.fy.ntw) * sizeof(double2);
}

int threads_for(int64_t work, int most) {
    return (int)std::clamp<int64_t>((work + 63) / 64 * 64, 64, most);
}

// kx columns a workgroup takes: towards whole memory sectors, but a workgroup
// per CU before that
int columns_log(const aw_ctx& c, int nmax, int runs) {
    const int nkx = c.g.nx / 2 + 1;
    int lg = 0;
    while (lg < 5 && columns_lds(c, nmax, 2 << lg) <= (size_t)64 << 10 &&
           (int64_t)((nkx + (2 << lg) - 1) / (2 << lg)) * runs >= std::max(1, c.num_cu) &&
           ((int64_t)c.g.ny << lg) * nmax < 4096)
        ++lg;
    return lg;
}

template <class Op>
void solve(aw_ctx& c, const SpecSrc& in, const SpecDst& out, const Op& op, int runs,
           unsigned int* smax, hipStream_t s) {
    AW_REQUIRE(Op::kIn > 2 ? c.own_em : c.own_es, "the grid's solves go through rocFFT");
    constexpr int NM = std::max(Op::kIn, Op::kOut);
    const int64_t nk = nkmodes(c);
    const int ny = c.g.ny;
    // either Darwin solve allocates for both, so that the second allocates nothing
    // (a caller may capture it after a first call of the other)
    constexpr int kGrids = std::max(Op::kIn + Op::kOut, Op::kIn > 2 ? OpEt::kIn + OpEt::kOut : 0);
    c.ktmp.reserve((size_t)2 * kGrids * nk * runs);
    float2* kin = reinterpret_cast<float2*>(c.ktmp.get());
    float2* kout = kin + (size_t)Op::kIn * nk * runs;
    const int rt = threads_for(c.g.nx / kAhead, 1024);
    auto rows = in.acc ? rows_forward_kernel<true, Op::kIn> : rows_forward_kernel<false, Op::kIn>;
    rows<<<dim3(pair_count(Op::kIn, ny), runs), rt, rows_lds(c), s>>>(in, c.fx, ny, kin);
    AW_LAUNCH_CHECK();
    const int lg = columns_log(c, NM, runs), nkx = c.g.nx / 2 + 1;
    columns_kernel<Op><<<dim3((nkx + (1 << lg) - 1) >> lg, runs),
                         threads_for(((int64_t)std::max(4, NM) * ny << lg) / 4, 512),
                         columns_lds(c, NM, 1 << lg), s>>>(
        kin, kout, geom(c), c.fy, lg, op, smax);
    AW_LAUNCH_CHECK();
    auto inverse = rows_inverse_kernel<Op::kOut, SpecDst::kPlain>;
    if constexpr (Op::kOut == 5) {
        if (out.form == SpecDst::kFormEl) inverse = rows_inverse_kernel<5, SpecDst::kFormEl>;
    }
    if constexpr (Op::kOut == 3) {
        if (out.form == SpecDst::kFormEt) inverse = rows_inverse_kernel<3, SpecDst::kFormEt>;
    }
    inverse<<<dim3(pair_count(Op::kOut, ny), runs), rt, rows_lds(c), s>>>(
        kout, c.fx, ny, 1.0 / ((double)c.g.nx * (double)ny), out);
    AW_LAUNCH_CHECK();
}

// Where the own transforms are ahead of rocFFT, for the electrostatic solve (one
// grid in, two out) and the Darwin ones (em: up to seven).  They save launches,
// while rocFFT's passes are cheaper once the launches are full, so it is a
// matter of size: measured on 300 grids from 24x17 to 3600x600 at two markers a
// cell, us a step below as own / rocFFT.  A grid's choice does not ask how many
// runs a batch holds: a run equals the same run stepped alone.
bool ahead(int nx, int ny, int direct, bool em) {
    auto pow2 = [](int n) { return (n & (n - 1)) == 0; };
    const int64_t cells = (int64_t)nx * ny;
    // rocFFT takes an odd real line as a complex one and falls behind (Darwin
    // 1001x1: 69 / 123, 61x61: 112 / 200, 625x625: 246 / 320) but for a long line
    // of direct sums (3599x1, 120 terms: 236 / 212; 3111x78, 78 terms in a row:
    // 306 / 431)
    if (nx % 2) return (int64_t)nx * direct <= 400000 && cells <= (int64_t)1 << 19;
    // work that no launch hides; 24 terms of direct sums weigh as much as all
    // other passes (610x610, 122 terms: Darwin 531 / 414).  Electrostatic
    // 2500x384: 81 / 87, 2500x600: 119 / 111; Darwin 960x360: 212 / 244,
    // 600x600: 249 / 240, 1200x360: 278 / 264, 3000x600: 935 / 703
    if (cells * (24 + direct) > 24 * (em ? (int64_t)350000 : (int64_t)1 << 20)) return false;
    // rocFFT's best sides.  Electrostatic 256x256: 29.7 / 31.9, 512x64: 28.5 /
    // 29.1, 512x128: 31.6 / 28.4; Darwin 1024x64: 95 / 100, 128x512: 108 / 102,
    // 2048x1: 67 / 63
    if (pow2(nx) && pow2(ny)) {
        const int side = std::max(nx, ny);
        if (em) return nx <= 1024 && ny <= 256;
        return side <= 256 || (side <= 512 && cells <= 1 << 15);
    }
    // long rows, and too few of them for the chip.  Darwin 1300x1: 69 / 76,
    // 1400x1: 68 / 64, 3600x1: 84 / 76, 3000x17: 113 / 99, 3000x60: 137 / 143
    if (em) return nx <= 1300 || ny > 60;
    // long rows and columns that rocFFT is good at.  Electrostatic 625x1: 22 / 37,
    // 1250x128: 36.6 / 32.6, 1250x1: 24.2 / 22.9, 3000x100: 50 / 48; 1000x120:
    // 34 / 45, 3000x250: 67 / 79
    if (direct == 0 && nx > 512 && ny > 1 && pow2(ny)) return false;
    return nx <= 1200 || ny > 100;
}

}  // namespace

// The grids whose solves run here: sides made of the transforms' factors, lines
// (at most a column of E_T's seven grids) that fit LDS, and where that is ahead.
void init_own_fft(aw_ctx& c) {
    c.own_es = c.own_em = false;
    int direct = 0;
    if (!make_line(c.g.nx, c.fx, direct) || !make_line(c.g.ny, c.fy, direct)) return;
    const bool es = ahead(c.g.nx, c.g.ny, direct, false), em = ahead(c.g.nx, c.g.ny, direct, true);
    if (!es && !em) return;
    if (rows_lds(c) + kRowsStaticLds > c.lds_per_block ||
        columns_lds(c, 7, 1) > c.lds_per_block)
        return;
    // both lines' twiddles, then their half-cell phases
    std::vector<double2> tw;
    for (const int n : {c.g.nx, c.g.ny})
        for (int k = 0; k < n; ++k) {
            const double th = kTwoPi * (double)k / (double)n;
            tw.push_back(make_double2(std::cos(th), -std::sin(th)));
        }
    for (const int n : {c.g.nx, c.g.ny})
        for (int k = 0; k <= n / 2; ++k) {
            const double th = 0.5 * kTwoPi * (double)k / (double)n;
            tw.push_back(make_double2(std::cos(th), std::sin(th)));
        }
    c.fft_tw.resize(tw.size());
    AW_HIP(hipMemcpy(c.fft_tw.get(), tw.data(), tw.size() * sizeof(double2), hipMemcpyHostToDevice));
    c.fx.tw = c.fft_tw.get();
    c.fy.tw = c.fft_tw.get() + c.g.nx;
    c.own_es = es;
    c.own_em = em;
}

// workgroups a run of the rows-inverse launch (the pairs of maxima of kFormEl)
int spec_blocks(const aw_ctx& c, int nq) { return pair_count(nq, c.g.ny); }

void spec_solve_es(aw_ctx& c, const SpecSrc& in, const SpecDst& out, double eps0, int runs,
                   hipStream_t s) {
    solve(c, in, out, OpEs{eps0}, runs, nullptr, s);
}

void spec_solve_es_adj(aw_ctx& c, const SpecSrc& in, const SpecDst& out, double eps0,
                       unsigned int* rmax, hipStream_t s) {
    solve(c, in, out, OpEsAdj{eps0}, 1, rmax, s);
}

void spec_solve_elb(aw_ctx& c, const SpecSrc& in, const SpecDst& out, double eps0, double cl,
                    const float B0[3], bool stag, int runs, hipStream_t s) {
    solve(c, in, out, OpElb{eps0, cl, {B0[0], B0[1], B0[2]}, stag ? 1 : 0}, runs, nullptr, s);
}

void spec_solve_et(aw_ctx& c, const SpecSrc& in, const SpecDst& out, double eps0, double cl,
                   double n0, int runs, hipStream_t s) {
    solve(c, in, out, OpEt{eps0, cl, n0}, runs, nullptr, s);
}

}  // namespace aw
