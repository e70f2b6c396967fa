// esk_device.hpp -- the Esirkepov current's per-particle device code and
// its host set-up, shared by the deposit kernels (esirkepov.hip) and by
// kernels that deposit the current of the moves they make (yee.hip).
//
// Reference: s1_shape4, esirkepov_scatter (include/pic/yee2d.hpp:124-132,
// 310-389).  Contributions are int64 fixed point with one scale exponent per
// component, taken from a bound on the largest single contribution.
#pragma once
#include "aw_internal.hpp"

namespace aw::esk {

constexpr int kFixBits = 44;
constexpr int kSortedApron = 4;  // particles in the tile order of an earlier sort

struct EskArgs {
    const float *x0, *y0, *x1, *y1, *uz, *w;
    float *xw, *yw;  // optional: x1, y1 wrapped into the box, written back
    int n, nx, ny;
    int per_w;       // per-particle deposit weights (w, or the caller's own)
    double qm, w_uniform, dt, dx, dy;
    const unsigned int* bound;  // [0] max|w| (or 0), [1] max|w uz| (|uz| for uniform w)
};

// Scale exponents of the three components (identical in deposit and convert).
__device__ __forceinline__ void esk_exponents(const EskArgs& a, int S[3]) {
    const double wmax = a.per_w ? (double)__uint_as_float(a.bound[0]) : fabs(a.w_uniform);
    const double wuz = a.per_w ? (double)__uint_as_float(a.bound[1])
                               : fabs(a.w_uniform) * (double)__uint_as_float(a.bound[1]);
    const double b[3] = {fabs(a.qm) * wmax / (a.dt * a.dy), fabs(a.qm) * wmax / (a.dt * a.dx),
                         fabs(a.qm) * wuz / (a.dx * a.dy)};
    for (int q = 0; q < 3; ++q) {
        int e = 0;
        (void)frexp(b[q], &e);  // b < 2^e
        S[q] = kFixBits - e;
    }
}

// the current of accumulated quanta v of component q: v 2^-S_q
__device__ __forceinline__ float esk_value(long long v, int Sq) {
    return (float)ldexp((double)v, -Sq);
}

__device__ __forceinline__ void esk_scales(const EskArgs& a, double scale[3]) {
    int S[3];
    esk_exponents(a, S);
    for (int q = 0; q < 3; ++q) scale[q] = ldexp(1.0, S[q]);
}

// One particle's move: the shared stencil geometry plus its fixed-point
// scaled coefficients.
struct EskMove {
    dev::EskShape sh;
    double cJx, cJy, cJz;
};

// The coefficients' constant factors, once per thread: kc = (2^Sx/(dt dy),
// 2^Sy/(dt dx), 2^Sz/(dx dy)), so a particle's coefficients are products.
__device__ __forceinline__ void esk_coefs(const EskArgs& a, double kc[3]) {
    double scale[3];
    esk_scales(a, scale);
    kc[0] = scale[0] / (a.dt * a.dy);
    kc[1] = scale[1] / (a.dt * a.dx);
    kc[2] = scale[2] / (a.dx * a.dy);
}

// the move (x0, y0) -> (x1, y1) with deposit weight w and velocity uz:
// cJx = -q w kc0, cJy = -q w kc1, cJz = q w uz kc2
__device__ __forceinline__ void esk_prepare_v(const EskArgs& a, float x0, float y0, float x1,
                                              float y1, float uz, double w, const double kc[3],
                                              EskMove& m) {
    dev::esk_shape(x0, y0, x1, y1, a.nx, a.ny, m.sh);
    const double qw = a.qm * w;
    m.cJx = -qw * kc[0];
    m.cJy = -qw * kc[1];
    m.cJz = qw * (double)uz * kc[2];
}

__device__ __forceinline__ void esk_prepare(const EskArgs& a, int i, const double kc[3],
                                            EskMove& m) {
    esk_prepare_v(a, a.x0[i], a.y0[i], a.x1[i], a.y1[i], a.uz[i],
                  a.w ? (double)a.w[i] : a.w_uniform, kc, m);
}

// The contributions of one move.  On a one-row grid (ny = 1) the three
// stencil rows are the same row: each (component, column) sum of the
// fixed-point contributions is formed in registers (exact, int64) and added
// once, at row 1, instead of once per row.
template <bool ONE_ROW, class Add>
__device__ __forceinline__ void esk_emit(const EskMove& m, Add&& add) {
    if constexpr (!ONE_ROW) {
        dev::esk_emit(m.sh, m.cJx, m.cJy, m.cJz, add);
    } else {
        unsigned long long col[3][4] = {};
        dev::esk_emit(m.sh, m.cJx, m.cJy, m.cJz,
                      [&](int q, int k, int, unsigned long long v) { col[q][k] += v; });
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int k = 1; k < 4; ++k)
                if (col[q][k]) add(q, k, 1, col[q][k]);
    }
}

// Moves that leave their cell, set aside by a wavefront in its own LDS slots
// until cap of them fill (most of) a wavefront.  A move inside one cell has 8
// of the 21 contributions and about a third of the arithmetic; moves that
// leave theirs are a few percent, but nearly every wavefront has one, and
// handled on the spot they would cost all 64 lanes the general stencil.
// Every lane of the wavefront calls push and drain.
struct MoveQueue {
    static constexpr int kFloats = 6;  // LDS per slot
    float* s;                          // this wavefront's slots, [6][cap]
    int cap;
    int cnt = 0;                       // wave-uniform

    // body(x0, y0, x1, y1, uz, w) runs once per set-aside move
    template <class Body>
    __device__ __forceinline__ void push(bool want, float x0, float y0, float x1, float y1,
                                         float uz, float w, Body&& body) {
        unsigned long long m = __ballot(want);
        while (m) {
            const int pos = cnt + (int)__builtin_amdgcn_mbcnt_hi(
                                      (unsigned)(m >> 32),
                                      __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            const bool put = want && pos < cap;
            if (put) {
                s[pos] = x0;
                s[cap + pos] = y0;
                s[2 * cap + pos] = x1;
                s[3 * cap + pos] = y1;
                s[4 * cap + pos] = uz;
                s[5 * cap + pos] = w;
                want = false;
            }
            cnt = min(cap, cnt + (int)__popcll(m));
            m = __ballot(want);
            if (m) drain(body);
        }
    }

    template <class Body>
    __device__ __forceinline__ void drain(Body&& body) {
        // the slots are this wavefront's own: its LDS accesses complete in
        // program order, the fences keep the compiler to that order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int l = (int)(threadIdx.x & 63); l < cnt; l += 64)
            body(s[l], s[cap + l], s[2 * cap + l], s[3 * cap + l], s[4 * cap + l],
                 s[5 * cap + l]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        cnt = 0;
    }
};

// esk_emit for a move inside its cell (one-row grids: each column's rows
// summed first, at row 1)
template <bool ONE_ROW, class Add>
__device__ __forceinline__ void esk_emit_cell(const dev::EskCell& m, double cJx, double cJy,
                                              double cz, Add&& add) {
    if constexpr (!ONE_ROW) {
        dev::esk_emit_cell(m, cJx, cJy, cz, add);
    } else {
        unsigned long long col[3][3] = {};
        dev::esk_emit_cell(m, cJx, cJy, cz,
                           [&](int q, int k, int, unsigned long long v) { col[q][k] += v; });
        add(0, 1, 1, col[0][1]);
#pragma unroll
        for (int k = 1; k < 3; ++k) {
            add(1, k, 1, col[1][k]);
            add(2, k, 1, col[2][k]);
        }
    }
}

__device__ __forceinline__ int wrap_local(int l, int n) {
    if (l < 0) l += n;
    else if (l >= n) l -= n;
    return l;
}

// Host side.  args fills the kernels' arguments; setup also clears the
// accumulators and takes the scale bound from a bound pass, unless the caller
// did both (EskExtra::fixed); convert adds the accumulated current to jx, jy, jz.
EskArgs args(aw_ctx& c, const float* x0, const float* y0, const aw_particles& p, double qm,
             double dt, const EskExtra& ex);
EskArgs setup(aw_ctx& c, const float* x0, const float* y0, const aw_particles& p, double qm,
              double dt, hipStream_t s, const EskExtra& ex);
void convert(aw_ctx& c, const EskArgs& a, float* jx, float* jy, float* jz, hipStream_t s);

}  // namespace aw::esk
