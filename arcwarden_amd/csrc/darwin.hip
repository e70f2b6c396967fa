// darwin.hip -- spectral Darwin particle kernels.
//
//   em_moments_kernel  rho, J, amu of the current state (init / API):
//                      deposit_rho_j_tiled_kernel + deposit_amu_kernel
//                      (include/pic/depositor.hpp:160-270)
//   dcu_kernel         qm^2 w/area (E + v x B) with E, B gathered from an LDS
//                      field tile: deposit_dcu_kernel (:275-324)
//   em_push_kernel     E, B gathered from an LDS tile, full Boris, move, wrap,
//                      then rho, J, amu of the NEW state deposited for the next
//                      step: em_push_tiled_kernel (pusher.hpp:211-258) +
//                      particle_migrate_kernel + the next step's ρ/J/amu
//                      deposits, for 40 B of particle traffic.
//
// All eight moments (rho, Jx, Jy, Jz, amu0..amu3) and the three dcu
// components accumulate fixed-point int64 quanta: each contribution is the
// FP32 product v*W rounded to an integer, v carrying the quantity's 2^S scale.
#include "esk_device.hpp"

#include <algorithm>

namespace aw {

namespace {

constexpr int kThreads = 256;

inline int blocks_for(int64_t n) { return (int)((n + kThreads - 1) / kThreads); }

__device__ __forceinline__ int local_index(int i, int org, int n) {
    int l = i - org;
    if (l < 0) l += n;
    else if (l >= n) l -= n;
    return l;
}

struct EmArgs {
    float *x, *y, *ux, *uy, *uz;
    const float* w;
    const int32_t* off;
    const int32_t* idx;          // bin permutation (unsorted particles) or nullptr
    int ntx, tx, ty, apron, W, H, bpt;
    int nx, ny, ncell;
    // fields (E = total, B), each [ny][nx]
    const float *Ex, *Ey, *Ez, *Bx, *By, *Bz;
    unsigned long long* acc;     // nq grids of ncell int64
    const float* cq;             // device: rho, J, amu coefficients 2^S * qm/area
                                 // (* w_uniform when uniform)
    const float* c_dcu;          // device: 2^S_dcu * qm^2/area (* w_uniform)
    float qmh, cx, cy;
    double dxdt, dydt;           // dx/dt, dy/dt (Esirkepov current coefficients)
    unsigned long long* strays;
    double* ke_part;
    int qslots;                  // slots of a wavefront's move queue (ESK)
    // uniform batch (EmBatch): run blockIdx.y offsets its pointers by these
    long long bp, be, bb, ba, bk;
    int bo;
};

// Moves every per-run pointer of a to run blockIdx.y of a uniform batch.
__device__ __forceinline__ void select_run(EmArgs& a) {
    const long long r = blockIdx.y;
    if (r == 0) return;
    a.x += r * a.bp;
    a.y += r * a.bp;
    a.ux += r * a.bp;
    a.uy += r * a.bp;
    a.uz += r * a.bp;
    if (a.w) a.w += r * a.bp;
    a.off += r * a.bo;
    if (a.Ex) {
        a.Ex += r * a.be;
        a.Ey += r * a.be;
        a.Ez += r * a.be;
        a.Bx += r * a.bb;
        a.By += r * a.bb;
        a.Bz += r * a.bb;
    }
    if (a.acc) a.acc += r * a.ba;
    if (a.c_dcu) a.c_dcu += r;
    if (a.ke_part) a.ke_part += r * a.bk;
}

// Range guard of the fixed-point moments: the static scales put the largest
// contribution allowed by |u| <= 2 max(1, c) at 2^48.  A moment beyond 2^50
// (|u| four times that bound for J, twice for amu) marks the thread's stray
// count with kRangeBit; the count reaches the host as stray_count +
// kRangeFlag, and the simulation reports the overflow instead of letting
// saturated (clamped) contributions pile up into a wrapped int64 sum.
constexpr float kRangeLimit = 1125899906842624.0f;  // 2^50
constexpr unsigned int kRangeBit = 0x80000000u;

__device__ __forceinline__ unsigned long long stray_word(unsigned int nstray) {
    return (unsigned long long)(nstray & ~kRangeBit) + ((nstray & kRangeBit) ? kRangeFlag : 0ull);
}

// the 8 moment values of one particle (already scaled); cq = a.cq
__device__ __forceinline__ void moments8(const float cq[3], float mw, float ux, float uy, float uz,
                                         float v[8]) {
    const float br = cq[0] * mw, bj = cq[1] * mw, ba = cq[2] * mw;
    v[0] = br;
    v[1] = bj * ux;
    v[2] = bj * uy;
    v[3] = bj * uz;
    v[4] = ba * (0.5f * (ux * ux - uy * uy));
    v[5] = ba * (ux * uy);
    v[6] = ba * (uz * ux);
    v[7] = ba * (uz * uy);
}

// the NQ moment values, clamped for fix_mul; notes one out of range
template <int NQ>
__device__ __forceinline__ void fix_values(const float* v_in, double* v, unsigned int& nstray) {
    float top = 0.f;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        top = fmaxf(top, fabsf(v_in[q]));
        v[q] = (double)dev::clamp_fix_f32(v_in[q]);
    }
    if (top > kRangeLimit) nstray |= kRangeBit;
}

// Deposits v[q] for the q < NQ selected by MASK (grid q of the tile / global
// accumulators): 4 CIC contributions rint(v[q] * W_k) per moment, with the
// FP64 weights of cic_d (exact products) and one fma per contribution.
template <int NQ, unsigned MASK = (1u << NQ) - 1u>
__device__ __forceinline__ void deposit_q(unsigned long long* s_acc, int R, int W, int H,
                                          unsigned long long* g_acc, int ncell, int nx, int ny,
                                          int orgx, int orgy, const dev::CicD& d,
                                          const float* v_in, unsigned int& nstray) {
    double v[NQ];
    fix_values<NQ>(v_in, v, nstray);
    const int mi = local_index(d.i0, orgx, nx), mj = local_index(d.j0, orgy, ny);
    if (dev::in_tile(mi, W - 2) && dev::in_tile(mj, H - 2)) {
        const int b = mj * W + mi;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (!((MASK >> q) & 1u)) continue;
            unsigned long long* s = s_acc + q * R;
            atomicAdd(&s[b], dev::fix_mul(v[q], d.w0));
            atomicAdd(&s[b + 1], dev::fix_mul(v[q], d.w1));
            atomicAdd(&s[b + W], dev::fix_mul(v[q], d.w2));
            atomicAdd(&s[b + W + 1], dev::fix_mul(v[q], d.w3));
        }
    } else {
        int i0, i1, j0, j1;
        dev::wrap_pair(d.i0, nx, i0, i1);
        dev::wrap_pair(d.j0, ny, j0, j1);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (!((MASK >> q) & 1u)) continue;
            unsigned long long* g = g_acc + (size_t)q * ncell;
            atomicAdd(&g[j0 * nx + i0], dev::fix_mul(v[q], d.w0));
            atomicAdd(&g[j0 * nx + i1], dev::fix_mul(v[q], d.w1));
            atomicAdd(&g[j1 * nx + i0], dev::fix_mul(v[q], d.w2));
            atomicAdd(&g[j1 * nx + i1], dev::fix_mul(v[q], d.w3));
        }
        ++nstray;
    }
}

template <int NQ>
__device__ __forceinline__ void flush_q(const unsigned long long* s_acc, int R, int W,
                                        unsigned long long* g_acc, int ncell, int nx, int ny,
                                        int orgx, int orgy) {
    for (int c = threadIdx.x; c < R; c += kThreads) {
        const int gc = dev::wrapfar(orgy + c / W, ny) * nx + dev::wrapfar(orgx + c % W, nx);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const unsigned long long v = s_acc[q * R + c];
            if (v) atomicAdd(&g_acc[(size_t)q * ncell + gc], v);
        }
    }
}

struct Frame {
    int W, H, R, orgx, orgy, r0, r1;
};

__device__ __forceinline__ Frame frame(const EmArgs& a) {
    Frame f;
    f.W = a.W;
    f.H = a.H;
    f.R = a.W * a.H;
    const int tile = blockIdx.x / a.bpt, part = blockIdx.x % a.bpt;
    f.orgx = (tile % a.ntx) * a.tx - a.apron;
    f.orgy = (tile / a.ntx) * a.ty - a.apron;
    dev::split_range(a.off[tile], a.off[tile + 1], part, a.bpt, f.r0, f.r1);
    return f;
}

// field tile: node c -> (Ex, Ey, Ez, Bx) float4 + (By, Bz) float2
__device__ __forceinline__ void load_fields(const EmArgs& a, const Frame& f, float4* fa,
                                            float2* fb) {
    for (int c = threadIdx.x; c < f.R; c += kThreads) {
        const int gc =
            dev::wrapfar(f.orgy + c / f.W, a.ny) * a.nx + dev::wrapfar(f.orgx + c % f.W, a.nx);
        fa[c] = make_float4(a.Ex[gc], a.Ey[gc], a.Ez[gc], a.Bx[gc]);
        fb[c] = make_float2(a.By[gc], a.Bz[gc]);
    }
}

// gather (E, B) at a particle: LDS tile when inside, global otherwise
__device__ __forceinline__ bool gather6(const EmArgs& a, const Frame& f, const float4* fa,
                                        const float2* fb, const dev::CicF& s, float e[3],
                                        float b[3]) {
    const int li = local_index(s.i0, f.orgx, a.nx), lj = local_index(s.j0, f.orgy, a.ny);
    if (dev::in_tile(li, f.W - 2) && dev::in_tile(lj, f.H - 2)) {
        const int n0 = lj * f.W + li, n1 = n0 + 1, n2 = n0 + f.W, n3 = n2 + 1;
        const float4 a0 = fa[n0], a1 = fa[n1], a2 = fa[n2], a3 = fa[n3];
        const float2 b0 = fb[n0], b1 = fb[n1], b2 = fb[n2], b3 = fb[n3];
        e[0] = dev::gather4(s, a0.x, a1.x, a2.x, a3.x);
        e[1] = dev::gather4(s, a0.y, a1.y, a2.y, a3.y);
        e[2] = dev::gather4(s, a0.z, a1.z, a2.z, a3.z);
        b[0] = dev::gather4(s, a0.w, a1.w, a2.w, a3.w);
        b[1] = dev::gather4(s, b0.x, b1.x, b2.x, b3.x);
        b[2] = dev::gather4(s, b0.y, b1.y, b2.y, b3.y);
        return true;
    }
    int i0, i1, j0, j1;
    dev::wrap_pair(s.i0, a.nx, i0, i1);
    dev::wrap_pair(s.j0, a.ny, j0, j1);
    const int c0 = j0 * a.nx + i0, c1 = j0 * a.nx + i1, c2 = j1 * a.nx + i0, c3 = j1 * a.nx + i1;
    const float* F[6] = {a.Ex, a.Ey, a.Ez, a.Bx, a.By, a.Bz};
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const float v = dev::gather4(s, F[q][c0], F[q][c1], F[q][c2], F[q][c3]);
        if (q < 3) e[q] = v;
        else b[q - 3] = v;
    }
    return false;
}

// Esirkepov current of the move (x0, y0) -> (x1, y1) into the J grids
// (q = 1..3) of the moment tile, or into the global accumulators when the 4x4
// union stencil leaves the tile frame.  cj = the J coefficient (fixed-point
// scaled, times the particle weight): Jx = -cj dx/dt sum DSx(..),
// Jy = -cj dy/dt sum DSy(..), Jz = cj uz W_z.  Every contribution is bounded
// by cj |u|, the bound of the CIC current, so the J scale carries over.
__device__ __forceinline__ void esk_deposit(const EmArgs& a, const Frame& f,
                                            unsigned long long* s_acc, float x0, float y0,
                                            float x1, float y1, float uz, double cj) {
    dev::EskShape m;
    dev::esk_shape(x0, y0, x1, y1, a.nx, a.ny, m);
    const double cJx = -cj * a.dxdt, cJy = -cj * a.dydt, cJz = cj * (double)uz;
    const int li = local_index(m.ib - 1, f.orgx, a.nx), lj = local_index(m.jb - 1, f.orgy, a.ny);
    if (dev::in_tile(li, f.W - 4) && dev::in_tile(lj, f.H - 4)) {
        unsigned long long* s = s_acc + f.R + lj * f.W + li;
        dev::esk_emit(m, cJx, cJy, cJz, [&](int q, int k, int b, unsigned long long v) {
            atomicAdd(&s[q * f.R + b * f.W + k], v);
        });
    } else {
        unsigned long long* g = a.acc + (size_t)a.ncell;
        int gx[3], gy[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            gx[k] = dev::wrapfar(m.ib + k, a.nx);
            gy[k] = dev::wrapfar(m.jb + k, a.ny) * a.nx;
        }
        dev::esk_emit(m, cJx, cJy, cJz, [&](int q, int k, int b, unsigned long long v) {
            atomicAdd(&g[(size_t)q * a.ncell + (gy[b - 1] + gx[k - 1])], v);
        });
    }
}

template <bool PER_W>
__global__ void __launch_bounds__(kThreads) em_moments_kernel(EmArgs a) {
    select_run(a);
    extern __shared__ unsigned long long smem[];
    const Frame f = frame(a);
    for (int c = threadIdx.x; c < 8 * f.R; c += kThreads) smem[c] = 0ull;
    __syncthreads();
    unsigned int nstray = 0;
    const float cq[3] = {a.cq[0], a.cq[1], a.cq[2]};
    for (int r = f.r0 + (int)threadIdx.x; r < f.r1; r += kThreads) {
        const int k = a.idx ? a.idx[r] : r;
        const float mw = PER_W ? a.w[k] : 1.0f;
        float v[8];
        moments8(cq, mw, a.ux[k], a.uy[k], a.uz[k], v);
        deposit_q<8>(smem, f.R, f.W, f.H, a.acc, a.ncell, a.nx, a.ny, f.orgx, f.orgy,
                     dev::cic_d(a.x[k], a.y[k]), v, nstray);
    }
    __syncthreads();
    flush_q<8>(smem, f.R, f.W, a.acc, a.ncell, a.nx, a.ny, f.orgx, f.orgy);
    if (nstray && a.strays) atomicAdd(a.strays, stray_word(nstray));
}

template <bool PER_W>
__global__ void __launch_bounds__(kThreads) dcu_kernel(EmArgs a) {
    select_run(a);
    extern __shared__ unsigned long long smem[];
    const Frame f = frame(a);
    unsigned long long* s_acc = smem;
    float4* fa = reinterpret_cast<float4*>(smem + 3 * f.R);
    float2* fb = reinterpret_cast<float2*>(fa + f.R);
    for (int c = threadIdx.x; c < 3 * f.R; c += kThreads) s_acc[c] = 0ull;
    load_fields(a, f, fa, fb);
    __syncthreads();
    const float cd = *a.c_dcu;
    unsigned int nstray = 0;
    // two particles per thread per iteration, both loaded first
    auto one = [&](float x, float y, float vx, float vy, float vz, float mw) {
        const dev::CicF s = dev::cic_f(x, y);
        float e[3], b[3];
        if (!gather6(a, f, fa, fb, s, e, b)) ++nstray;
        const float base = PER_W ? cd * mw : cd;
        float v[3];
        v[0] = base * (e[0] + (vy * b[2] - vz * b[1]));
        v[1] = base * (e[1] + (vz * b[0] - vx * b[2]));
        v[2] = base * (e[2] + (vx * b[1] - vy * b[0]));
        deposit_q<3>(s_acc, f.R, f.W, f.H, a.acc, a.ncell, a.nx, a.ny, f.orgx, f.orgy,
                     dev::cic_d(x, y), v, nstray);
    };
    int r = f.r0 + (int)threadIdx.x;
    for (; r + kThreads < f.r1; r += 2 * kThreads) {
        const int k0 = a.idx ? a.idx[r] : r;
        const int k1 = a.idx ? a.idx[r + kThreads] : r + kThreads;
        const float x0 = a.x[k0], y0 = a.y[k0], ux0 = a.ux[k0], uy0 = a.uy[k0], uz0 = a.uz[k0];
        const float x1 = a.x[k1], y1 = a.y[k1], ux1 = a.ux[k1], uy1 = a.uy[k1], uz1 = a.uz[k1];
        const float w0 = PER_W ? a.w[k0] : 1.0f, w1 = PER_W ? a.w[k1] : 1.0f;
        one(x0, y0, ux0, uy0, uz0, w0);
        one(x1, y1, ux1, uy1, uz1, w1);
    }
    if (r < f.r1) {
        const int k = a.idx ? a.idx[r] : r;
        one(a.x[k], a.y[k], a.ux[k], a.uy[k], a.uz[k], PER_W ? a.w[k] : 1.0f);
    }
    __syncthreads();
    flush_q<3>(s_acc, f.R, f.W, a.acc, a.ncell, a.nx, a.ny, f.orgx, f.orgy);
    if (nstray && a.strays) atomicAdd(a.strays, stray_word(nstray));
}

// Moves that leave their cell wait in LDS (esk_device.hpp): as many slots as
// the 16x16-cell tile leaves of a quarter of a CU's LDS (fewer where a larger
// tile leaves less).
using esk::MoveQueue;
constexpr int kQueueSlots = 20;
// static LDS of the push's kinetic-energy instances, beside the tile and the
// queue: a double a wavefront
constexpr size_t kPushStaticLds = (kThreads / 64) * sizeof(double);

struct EmIn {
    float x, y, ux, uy, uz, w;
};

// E, B gathered at x^n, Boris, move, wrap and the eight moments of the new
// state.  ESK: the current is the Esirkepov current of this step's move
// (staggered Jx, Jy), not the CIC current at x^{n+1}; rho and amu stay CIC at
// x^{n+1}.  A move inside one cell (nearly all of them) has both on the same
// four nodes: 20 + 8 contributions where the general stencil has 20 + 21.
// Particle k of the uniform first particle `base` keeps a lane's offset below
// 32 bits; the next iteration's loads are in flight while this one's particle
// is pushed.  16.8 M particles (512x128, vth 0.019 cells a step), ESK: 325 ->
// 286 us.  It is bound by LDS: a particle's 28 atomics take 14 cycles a
// wavefront at random cells, its eight gather reads 93, 210 us in all
// (HBM: 40 B a particle, 130 us).
template <bool PER_W, bool KE, bool ESK>
__global__ void __launch_bounds__(kThreads) em_push_kernel(EmArgs a) {
    select_run(a);
    extern __shared__ unsigned long long smem[];
    const Frame f = frame(a);
    constexpr int kNq = 8;
    unsigned long long* s_acc = smem;
    float4* fa = reinterpret_cast<float4*>(smem + kNq * f.R);
    float2* fb = reinterpret_cast<float2*>(fa + f.R);
    MoveQueue queue{reinterpret_cast<float*>(fb + f.R) +
                        (threadIdx.x >> 6) * a.qslots * MoveQueue::kFloats,
                    a.qslots};
    auto slot = [&](float* q, int b, int k) -> float& {
        return *reinterpret_cast<float*>(reinterpret_cast<char*>(q + b) + ((unsigned)k << 2));
    };
    auto fetch = [&](int b) {  // lanes past the end load the last particle and drop it
        const int k = min((int)threadIdx.x, f.r1 - 1 - b);
        return EmIn{slot(a.x, b, k),  slot(a.y, b, k),  slot(a.ux, b, k), slot(a.uy, b, k),
                    slot(a.uz, b, k), PER_W ? slot(const_cast<float*>(a.w), b, k) : 1.0f};
    };
    EmIn p{};
    if (f.r0 < f.r1) p = fetch(f.r0);
    for (int c = threadIdx.x; c < kNq * f.R; c += kThreads) s_acc[c] = 0ull;
    load_fields(a, f, fa, fb);
    __syncthreads();
    unsigned int nstray = 0;
    double ke = 0.0;
    const float cq[3] = {a.cq[0], a.cq[1], a.cq[2]};
    // the J coefficient (Jx = -cj dx/dt .., Jy = -cj dy/dt .., Jz = cj uz ..)
    const double cju = (double)cq[1];
    const double cJxu = dev::clamp_fix_f64(-cju * a.dxdt), cJyu = dev::clamp_fix_f64(-cju * a.dydt);
    auto general = [&](float x0, float y0, float x1, float y1, float uz, float w) {
        esk_deposit(a, f, s_acc, x0, y0, x1, y1, uz, (double)cq[1] * (double)w);
    };
    for (int base = f.r0; base < f.r1; base += kThreads) {
        const bool valid = base + (int)threadIdx.x < f.r1;
        const EmIn pn = fetch(min(base + kThreads, f.r1 - 1));
        bool leaves = false;
        float xn = 0.f, yn = 0.f, uz = 0.f;
        if (valid) {
            float ux = p.ux, uy = p.uy;
            uz = p.uz;
            const dev::CicF s = dev::cic_f(p.x, p.y);
            float e[3], b[3];
            if (!gather6(a, f, fa, fb, s, e, b)) ++nstray;
            dev::boris_full(a.qmh, e[0], e[1], e[2], b[0], b[1], b[2], ux, uy, uz);
            xn = dev::wrap_coord(fmaf(ux, a.cx, p.x), (float)a.nx);
            yn = dev::wrap_coord(fmaf(uy, a.cy, p.y), (float)a.ny);
            const int k = (int)threadIdx.x;
            slot(a.x, base, k) = xn;
            slot(a.y, base, k) = yn;
            slot(a.ux, base, k) = ux;
            slot(a.uy, base, k) = uy;
            slot(a.uz, base, k) = uz;
            if constexpr (KE)
                ke += (PER_W ? (double)p.w : 1.0) *
                      ((double)ux * ux + (double)uy * uy + (double)uz * uz);
            float v[8];
            moments8(cq, p.w, ux, uy, uz, v);
            const dev::CicD d = dev::cic_d(xn, yn);
            if constexpr (ESK) {
                // rho and amu of every particle, then J of the moves inside a cell
                deposit_q<8, 0xF1u>(s_acc, f.R, f.W, f.H, a.acc, a.ncell, a.nx, a.ny, f.orgx,
                                    f.orgy, d, v, nstray);
                const int mi = local_index(d.i0, f.orgx, a.nx),
                          mj = local_index(d.j0, f.orgy, a.ny);
                leaves = !(dev::esk_same_cell(p.x, p.y, xn, yn, floorf(p.x), floorf(p.y), a.nx,
                                              a.ny) &&
                           dev::in_tile(mi, f.W - 2) && dev::in_tile(mj, f.H - 2));
                if (!leaves) {
                    const dev::EskCell c = dev::esk_cell(
                        (double)p.x - (double)d.i0, (double)p.y - (double)d.j0,
                        (double)xn - (double)d.i0, (double)yn - (double)d.j0);
                    double cj = cju, cJx = cJxu, cJy = cJyu;
                    if constexpr (PER_W) {
                        cj = (double)cq[1] * (double)p.w;
                        cJx = dev::clamp_fix_f64(-cj * a.dxdt);
                        cJy = dev::clamp_fix_f64(-cj * a.dydt);
                    }
                    const double cz = dev::clamp_fix_f64(cj * (double)uz * (16.0 / 12.0));
                    unsigned long long* sj = s_acc + f.R + mj * f.W + mi;
                    dev::esk_emit_cell(c, cJx, cJy, cz,
                                       [&](int q, int k, int b, unsigned long long t) {
                                           atomicAdd(&sj[q * f.R + (b - 1) * f.W + (k - 1)], t);
                                       });
                }
            } else {
                deposit_q<8>(s_acc, f.R, f.W, f.H, a.acc, a.ncell, a.nx, a.ny, f.orgx, f.orgy, d,
                             v, nstray);
            }
        }
        if constexpr (ESK) queue.push(leaves, p.x, p.y, xn, yn, uz, p.w, general);
        p = pn;
    }
    if constexpr (ESK) queue.drain(general);
    __shared__ double s_ke[kThreads / 64];
    if constexpr (KE) {
        for (int o = 32; o > 0; o >>= 1) ke += __shfl_down(ke, o, 64);
        if ((threadIdx.x & 63) == 0) s_ke[threadIdx.x >> 6] = ke;
    }
    __syncthreads();
    flush_q<8>(s_acc, f.R, f.W, a.acc, a.ncell, a.nx, a.ny, f.orgx, f.orgy);
    if (nstray && a.strays) atomicAdd(a.strays, stray_word(nstray));
    if constexpr (KE) {
        if (threadIdx.x == 0) {
            double t = 0.0;
            for (int w = 0; w < kThreads / 64; ++w) t += s_ke[w];
            a.ke_part[blockIdx.x] = t;
        }
    }
}

// Push, move and wrap only (Pusher::boris_em + migrate), for particles in any
// order.  Cell c's fields are packed first as two float4, (Ex, Ey, Ez, Bx) and
// (By, Bz, -, -), so the nodes of a row are 64 contiguous bytes and a particle
// issues 8 wide loads for its 24 values; they come from L2, the particle
// arrays stream.  At 1.6 M particles in no order: 34 us with the packing,
// against 203 us through tile bins (whose permuted reads and writes are not
// coalesced) and the 110 us of binning first.
__global__ void __launch_bounds__(kThreads)
em_pack_kernel(const float* __restrict__ Ex, const float* __restrict__ Ey,
               const float* __restrict__ Ez, const float* __restrict__ Bx,
               const float* __restrict__ By, const float* __restrict__ Bz, int ncell,
               float4* __restrict__ pk) {
    const int c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= ncell) return;
    pk[2 * (size_t)c] = make_float4(Ex[c], Ey[c], Ez[c], Bx[c]);
    pk[2 * (size_t)c + 1] = make_float4(By[c], Bz[c], 0.f, 0.f);
}

__global__ void __launch_bounds__(kThreads)
em_push_any_kernel(float* __restrict__ X, float* __restrict__ Y, float* __restrict__ UX,
                   float* __restrict__ UY, float* __restrict__ UZ, int n, int nx, int ny,
                   const float4* __restrict__ pk, float qmh, float cx, float cy) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= n) return;
    const float x = X[k], y = Y[k];
    float ux = UX[k], uy = UY[k], uz = UZ[k];
    const dev::CicF s = dev::cic_f(x, y);
    int i0, i1, j0, j1;
    dev::wrap_pair(s.i0, nx, i0, i1);
    dev::wrap_pair(s.j0, ny, j0, j1);
    const size_t c0 = 2 * ((size_t)j0 * nx + i0), c1 = 2 * ((size_t)j0 * nx + i1),
                 c2 = 2 * ((size_t)j1 * nx + i0), c3 = 2 * ((size_t)j1 * nx + i1);
    const float4 a0 = pk[c0], a1 = pk[c1], a2 = pk[c2], a3 = pk[c3];
    const float4 b0 = pk[c0 + 1], b1 = pk[c1 + 1], b2 = pk[c2 + 1], b3 = pk[c3 + 1];
    dev::boris_full(qmh, dev::gather4(s, a0.x, a1.x, a2.x, a3.x),
                    dev::gather4(s, a0.y, a1.y, a2.y, a3.y),
                    dev::gather4(s, a0.z, a1.z, a2.z, a3.z),
                    dev::gather4(s, a0.w, a1.w, a2.w, a3.w),
                    dev::gather4(s, b0.x, b1.x, b2.x, b3.x),
                    dev::gather4(s, b0.y, b1.y, b2.y, b3.y), ux, uy, uz);
    X[k] = dev::wrap_coord(fmaf(ux, cx, x), (float)nx);
    Y[k] = dev::wrap_coord(fmaf(uy, cy, y), (float)ny);
    UX[k] = ux;
    UY[k] = uy;
    UZ[k] = uz;
}

// nq int64 grids -> float grids (assign), acc cleared; inv scale per grid
// from device memory (the dcu scale changes every step).  out2 receives a
// second copy: rocFFT may overwrite the input of an out-of-place R2C, so the
// transform reads the copy and the source grids stay intact.
// Batched (gridDim.y runs): run r uses acc + r*sa, out + r*so, out2 + r*so2,
// inv + r*si.
// base0 (per run, may be NULL): the integer baseline taken off grid 0's copy
// in out2 -- the run's mean charge density, which the E_L solve drops (k = 0),
// so the FP32 transform rounds relative to the fluctuation.
__global__ void convert_multi_kernel(unsigned long long* __restrict__ acc, float* __restrict__ out,
                                     float* __restrict__ out2, int ncell, int nq,
                                     const double* __restrict__ inv, long long sa, long long so,
                                     long long so2, int si, const long long* __restrict__ base0) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    const long long r = blockIdx.y;
    acc += r * sa;
    out += r * so;
    if (out2) out2 += r * so2;
    inv += r * si;
    for (int q = 0; q < nq; ++q) {
        const size_t i = (size_t)q * ncell + c;
        const long long a = (long long)acc[i];
        const float v = (float)((double)a * inv[q]);
        out[i] = v;
        if (out2) {
            const long long b = (q == 0 && base0) ? base0[r] : 0ll;
            out2[i] = b ? (float)((double)(a - b) * inv[q]) : v;
        }
        acc[i] = 0ull;
    }
}

// E = (E_L + s*E_T) + pump(t) (combine_etotal_kernel, solver_darwin.hpp:134-144;
// add_pump_kernel, pump.hpp:34-47); ET[0] may be null (s = 0).
__global__ void form_e_kernel(FormE f, int nx, int ncell, PumpArgs p) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    if (const long long r = blockIdx.y) {  // run r of a batch
        for (int q = 0; q < 3; ++q) {
            f.E[q] += r * f.sE;
            if (f.ET[q]) f.ET[q] += r * f.sT;
        }
        f.EL[0] += r * f.sL;
        f.EL[1] += r * f.sL;
    }
    float ex = f.EL[0][c], ey = f.EL[1][c], ez = 0.0f;
    if (f.ET[0]) {
        ex = ex + 1.0f * f.ET[0][c];
        ey = ey + 1.0f * f.ET[1][c];
        ez = 1.0f * f.ET[2][c];
    }
    if (p.on && p.t < p.toff) {
        float px, py, pz;
        dev::pump_at(p, c % nx, px, py, pz);
        ex += px;
        ey += py;
        ez += pz;
    }
    f.E[0][c] = ex;
    f.E[1][c] = ey;
    f.E[2][c] = ez;
}

struct Field6 {
    const float* f[6];  // Ex, Ey, Ez, Bx, By, Bz
};

// block maxima of |E|, |B| components -> part[blockIdx]
__global__ void __launch_bounds__(kThreads)
field_max_kernel(Field6 F, int ncell, float* __restrict__ part, long long sE, long long sB) {
    __shared__ float sh[2][kThreads];
    if (const long long r = blockIdx.y) {  // run r of a batch
        for (int q = 0; q < 3; ++q) {
            F.f[q] += r * sE;
            F.f[3 + q] += r * sB;
        }
        part += r * 2 * gridDim.x;
    }
    float me = 0.f, mb = 0.f;
    for (int c = blockIdx.x * kThreads + threadIdx.x; c < ncell; c += gridDim.x * kThreads) {
        for (int q = 0; q < 3; ++q) {
            me = fmaxf(me, fabsf(F.f[q][c]));
            mb = fmaxf(mb, fabsf(F.f[3 + q][c]));
        }
    }
    sh[0][threadIdx.x] = me;
    sh[1][threadIdx.x] = mb;
    __syncthreads();
    for (int o = kThreads / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            sh[0][threadIdx.x] = fmaxf(sh[0][threadIdx.x], sh[0][threadIdx.x + o]);
            sh[1][threadIdx.x] = fmaxf(sh[1][threadIdx.x], sh[1][threadIdx.x + o]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sh[0][0];
        part[2 * blockIdx.x + 1] = sh[1][0];
    }
}

// dcu scale: per-contribution bound = |qm^2 w/area| (max|E| + umax max|B|);
// S = 48 - ceil(log2(bound)) maps the bound to 2^48.  Writes the float
// coefficient used by dcu_kernel and the inverse scale used by conversion.
// meas (optional, device): {coef_abs, umax} measured from the particles.
// Batched: a workgroup per run (blockIdx.x), run r reads part + 2*nb*r and
// writes c_dcu[r], inv_dcu + si*r.
constexpr int kScaleWaves = 256;
__global__ void __launch_bounds__(kScaleWaves)
dcu_scale_kernel(const float* __restrict__ part, int nb, double coef_abs, double coef_signed,
                 double umax, const double* __restrict__ meas, float* __restrict__ c_dcu,
                 double* __restrict__ inv_dcu, int si) {
    const int r = blockIdx.x;
    part += (size_t)2 * nb * r;
    c_dcu += r;
    inv_dcu += (size_t)si * r;
    float me = 0.f, mb = 0.f;
    for (int i = threadIdx.x; i < nb; i += kScaleWaves) {
        me = fmaxf(me, part[2 * i]);
        mb = fmaxf(mb, part[2 * i + 1]);
    }
    dev::block_max2(me, mb);
    if (threadIdx.x != 0) return;
    if (meas) {
        coef_abs = meas[0];
        umax = meas[1];
    }
    double bound = coef_abs * ((double)me + umax * (double)mb);
    if (!(bound > 1e-300)) bound = 1e-300;
    int S = 48 - (int)ceil(log2(bound));
    if (S > 120) S = 120;
    if (S < -120) S = -120;
    *c_dcu = (float)ldexp(coef_signed, S);
    const double inv = ldexp(1.0, -S);
    inv_dcu[0] = inv;  // one entry per dcu component (convert_multi reads 3)
    inv_dcu[1] = inv;
    inv_dcu[2] = inv;
}

__device__ __forceinline__ int scale_exp(double bound) {
    if (!(bound > 1e-300)) bound = 1e-300;
    const int S = 48 - (int)ceil(log2(bound));
    return S > 120 ? 120 : (S < -120 ? -120 : S);
}

// per-workgroup max |w| (per-particle weights) and max |u| component into
// part[2 b], part[2 b + 1].  One address for every wave's maximum cost 97 us
// at 1.6 M particles: the atomics follow one another in L2.
__global__ void __launch_bounds__(kThreads)
moment_bound_kernel(const float* __restrict__ ux, const float* __restrict__ uy,
                    const float* __restrict__ uz, const float* __restrict__ w, int n,
                    float* __restrict__ part) {
    float mw = 0.f, mu = 0.f;
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        mu = fmaxf(mu, fmaxf(fabsf(ux[i]), fmaxf(fabsf(uy[i]), fabsf(uz[i]))));
        if (w) mw = fmaxf(mw, fabsf(w[i]));
    }
    dev::block_max2(mw, mu);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = mw;
        part[2 * blockIdx.x + 1] = mu;
    }
}

// Moment scales from the npart measured bounds (the same rule as the
// Simulation's static scales): cq = {rho, J, amu} coefficients, inv[0..7] the
// inverse scales of rho, Jx..Jz, amu0..3, dv = {dcu coef_abs, umax}.
constexpr int kScaleThreads = 1024;
__global__ void __launch_bounds__(kScaleThreads)
moment_scale_kernel(const float* __restrict__ part, int npart, int per_w, double qm, double area,
                    double w_uniform, float* __restrict__ cq, double* __restrict__ inv,
                    double* __restrict__ dv) {
    float mw = 0.f, mu = 0.f;
    for (int b = threadIdx.x; b < npart; b += kScaleThreads) {
        mw = fmaxf(mw, part[2 * b]);
        mu = fmaxf(mu, part[2 * b + 1]);
    }
    dev::block_max2(mw, mu);
    if (threadIdx.x != 0) return;
    const double wmax = per_w ? (double)mw : fabs(w_uniform);
    const double umax = (double)mu;
    const double cabs = fabs(qm) * wmax / area;
    const int S[3] = {scale_exp(cabs), scale_exp(cabs * umax), scale_exp(cabs * umax * umax)};
    const double mult = per_w ? 1.0 : w_uniform;
    for (int q = 0; q < 3; ++q) cq[q] = (float)ldexp(qm * mult / area, S[q]);
    inv[0] = ldexp(1.0, -S[0]);
    for (int q = 1; q < 4; ++q) inv[q] = ldexp(1.0, -S[1]);
    for (int q = 4; q < 8; ++q) inv[q] = ldexp(1.0, -S[2]);
    dv[0] = qm * qm * wmax / area;
    dv[1] = umax;
}

struct Out8 {
    float* o[8];
};

// out_q += acc_q * inv[q] for q < nq (separate output grids)
__global__ void convert_add_kernel(const unsigned long long* __restrict__ acc, Out8 out, int ncell,
                                   int nq, const double* __restrict__ inv) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    for (int q = 0; q < nq; ++q)  // a NULL output skips its quantity
        if (out.o[q]) out.o[q][c] += (float)((double)(long long)acc[(size_t)q * ncell + c] * inv[q]);
}

}  // namespace

// ---- host side ------------------------------------------------------------------------


static EmArgs em_args(aw_ctx& c, const aw_particles& p, const int32_t* off, const int32_t* idx,
                      const float* const* F, unsigned long long* acc, const float* cq,
                      const float* c_dcu, double qm, double dt, int bpt,
                      unsigned long long* strays, double* ke_part) {
    EmArgs a{};
    a.x = p.x;
    a.y = p.y;
    a.ux = p.ux;
    a.uy = p.uy;
    a.uz = p.uz;
    a.w = p.w;
    a.off = off;
    a.idx = idx;
    a.ntx = c.ntx;
    a.tx = c.tx;
    a.ty = c.ty;
    a.apron = c.apron;
    a.W = c.tx + 2 * c.apron + 1;
    a.H = c.ty + 2 * c.apron + 1;
    a.bpt = bpt;
    a.nx = c.g.nx;
    a.ny = c.g.ny;
    a.ncell = (int)ncell(c);
    if (F) {
        a.Ex = F[0];
        a.Ey = F[1];
        a.Ez = F[2];
        a.Bx = F[3];
        a.By = F[4];
        a.Bz = F[5];
    }
    a.acc = acc;
    a.cq = cq;
    a.c_dcu = c_dcu;
    a.qmh = (float)(qm * 0.5 * dt);
    a.cx = (float)(dt / c.g.dx);
    a.cy = (float)(dt / c.g.dy);
    a.dxdt = dt != 0.0 ? c.g.dx / dt : 0.0;
    a.dydt = dt != 0.0 ? c.g.dy / dt : 0.0;
    a.strays = strays;
    a.ke_part = ke_part;
    return a;
}

static size_t tile_nodes(const aw_ctx& c) {
    return (size_t)(c.tx + 2 * c.apron + 1) * (c.ty + 2 * c.apron + 1);
}
// the moments' and the push's accumulators (and fields) per node of the tile
int em_push_bpt(const aw_ctx& c, int64_t n, int runs) {
    return balanced_bpt(c, n, tile_nodes(c) * 88, 4, 3, runs);
}
int em_moments_bpt(const aw_ctx& c, int64_t n, int runs) {
    return balanced_bpt(c, n, tile_nodes(c) * 64, 8, 3, runs);
}

static void set_batch(EmArgs& a, const EmBatch& b) {
    a.bp = b.pstride;
    a.be = b.estride;
    a.bb = b.bstride;
    a.ba = b.astride;
    a.bk = b.kstride;
    a.bo = b.ostride;
}

// Batched forms (b.runs > 1): p describes run 0 (p.n particles per run);
// runs 1.. lie at the strides of b.
void em_moments(aw_ctx& c, const aw_particles& p, const int32_t* off, const int32_t* idx,
                unsigned long long* acc8, const float* cq, int bpt, unsigned long long* strays,
                hipStream_t s, const EmBatch& b) {
    if (p.n == 0) return;
    EmArgs a = em_args(c, p, off, idx, nullptr, acc8, cq, nullptr, 0.0, 0.0, bpt, strays,
                       nullptr);
    set_batch(a, b);
    const size_t sh = (size_t)a.W * a.H * 8 * 8;
    AW_REQUIRE(sh <= c.lds_per_block, "tile too large for the LDS of the moment deposit");
    const dim3 grid(c.ntiles * bpt, b.runs);
    if (p.w) em_moments_kernel<true><<<grid, kThreads, sh, s>>>(a);
    else em_moments_kernel<false><<<grid, kThreads, sh, s>>>(a);
    AW_LAUNCH_CHECK();
}

void em_dcu(aw_ctx& c, const aw_particles& p, const int32_t* off, const int32_t* idx,
            const float* const* F, unsigned long long* acc3, const float* c_dcu, int bpt,
            unsigned long long* strays, hipStream_t s, const EmBatch& b) {
    if (p.n == 0) return;
    EmArgs a = em_args(c, p, off, idx, F, acc3, nullptr, c_dcu, 0.0, 0.0, bpt, strays, nullptr);
    set_batch(a, b);
    const size_t sh = (size_t)a.W * a.H * (3 * 8 + 16 + 8);
    AW_REQUIRE(sh <= c.lds_per_block, "tile too large for the LDS of the dcu deposit");
    const dim3 grid(c.ntiles * bpt, b.runs);
    if (p.w) dcu_kernel<true><<<grid, kThreads, sh, s>>>(a);
    else dcu_kernel<false><<<grid, kThreads, sh, s>>>(a);
    AW_LAUNCH_CHECK();
}

// esk: the J moments of acc8 are the Esirkepov current of the move (staggered
// Jx, Jy).
int em_push(aw_ctx& c, const aw_particles& p, const int32_t* off, const float* const* F,
            unsigned long long* acc8, const float* cq, double qm,
            double dt, int bpt, unsigned long long* strays, double* ke_part, hipStream_t s,
            bool esk, const EmBatch& b) {
    if (p.n == 0) return 0;
    EmArgs a = em_args(c, p, off, nullptr, F, acc8, cq, nullptr, qm, dt, bpt, strays, ke_part);
    set_batch(a, b);
    size_t sh = (size_t)a.W * a.H * (8 * 8 + 16 + 8);
    if (esk) {
        constexpr size_t slot = (kThreads / 64) * MoveQueue::kFloats * sizeof(float);
        const size_t held = sh + kPushStaticLds;
        const size_t left = c.lds_per_block > held ? c.lds_per_block - held : 0;
        a.qslots = (int)std::clamp<size_t>(left / slot, 1, kQueueSlots);
        sh += a.qslots * slot;
    }
    AW_REQUIRE(sh <= c.lds_per_block, "tile too large for the LDS of the EM push");
    const int nblk = c.ntiles * bpt;
    const bool pw = p.w != nullptr, ke = ke_part != nullptr;
    auto launch = [&](auto kernel) {
        kernel<<<dim3(nblk, b.runs), kThreads, sh, s>>>(a);
        AW_LAUNCH_CHECK();
    };
    if (esk) {
        if (pw && ke) launch(em_push_kernel<true, true, true>);
        else if (pw) launch(em_push_kernel<true, false, true>);
        else if (ke) launch(em_push_kernel<false, true, true>);
        else launch(em_push_kernel<false, false, true>);
    } else {
        if (pw && ke) launch(em_push_kernel<true, true, false>);
        else if (pw) launch(em_push_kernel<true, false, false>);
        else if (ke) launch(em_push_kernel<false, true, false>);
        else launch(em_push_kernel<false, false, false>);
    }
    return nblk;
}

// Batched (runs > 1): run r converts acc + r*sa into out + r*so (and
// out2 + r*so2) with the scales at inv + r*si.
void convert_multi(unsigned long long* acc, float* out, float* out2, int64_t ncell, int nq,
                   const double* inv, hipStream_t s, int runs, long long sa, long long so,
                   long long so2, int si, const long long* base0) {
    convert_multi_kernel<<<dim3(blocks_for(ncell), runs), kThreads, 0, s>>>(
        acc, out, out2, (int)ncell, nq, inv, sa, so, so2, si, base0);
    AW_LAUNCH_CHECK();
}

PumpArgs pump_args(const aw_grid& g, const aw_run_params& rp, double t) {
    PumpArgs p{};
    p.on = rp.pump ? 1 : 0;
    p.ex = rp.pump_ex;
    p.ey = rp.pump_ey;
    p.ez = rp.pump_ez;
    p.k0 = rp.pump_k0;
    p.w0 = rp.pump_w0;
    p.trmp = rp.pump_trmp;
    p.toff = rp.pump_toff;
    p.t = t;
    p.dx = g.dx;
    return p;
}

// Batched (runs > 1): f carries run 0's pointers and the per-run strides.
void form_e(const FormE& f, const aw_grid& g, const aw_run_params& rp, double t, hipStream_t s,
            int runs) {
    const PumpArgs p = pump_args(g, rp, t);
    const int64_t nc = (int64_t)g.nx * g.ny;
    form_e_kernel<<<dim3(blocks_for(nc), runs), kThreads, 0, s>>>(f, g.nx, (int)nc, p);
    AW_LAUNCH_CHECK();
}

void dcu_scale_parts(const float* part, int nb, double coef_abs, double coef_signed, double umax,
                     const double* dev, float* c_dcu, double* inv_dcu, hipStream_t s, int runs,
                     int si);

// Batched (runs > 1): F holds run 0's fields, E components at stride sE and
// B at stride sB per run; part holds dcu_part_capacity(ncell) floats per run,
// c_dcu one float and inv_dcu si doubles per run.
void dcu_scale(const float* const* F, int64_t ncell, float* part, double coef_abs,
               double coef_signed, double umax, const double* dev, float* c_dcu, double* inv_dcu,
               hipStream_t s, int runs, long long sE, long long sB, int si) {
    AW_REQUIRE(runs >= 1 && runs <= 64, "dcu scale: 1..64 runs");
    const int nb = (int)std::min<int64_t>(256, std::max<int64_t>(1, (ncell + 4095) / 4096));
    Field6 f6{{F[0], F[1], F[2], F[3], F[4], F[5]}};
    field_max_kernel<<<dim3(nb, runs), kThreads, 0, s>>>(f6, (int)ncell, part, sE, sB);
    AW_LAUNCH_CHECK();
    dcu_scale_parts(part, nb, coef_abs, coef_signed, umax, dev, c_dcu, inv_dcu, s, runs, si);
}

// the same from maxima already taken, nb pairs per run
void dcu_scale_parts(const float* part, int nb, double coef_abs, double coef_signed, double umax,
                     const double* dev, float* c_dcu, double* inv_dcu, hipStream_t s, int runs,
                     int si) {
    dcu_scale_kernel<<<runs, kScaleWaves, 0, s>>>(part, nb, coef_abs, coef_signed, umax, dev, c_dcu,
                                                  inv_dcu, si);
    AW_LAUNCH_CHECK();
}

int dcu_part_capacity() { return 2 * 256; }

// ---- standalone operators (any particle order) ------------------------------------------
//
// aw_deposit_rho_j_amu, aw_deposit_dcu and aw_push_boris_em take particles in
// any order.  The deposits sort a copy of them by tile (or, without room for
// it, bin them into the context's permutation and read them through it); their
// fixed-point scales come from the measured max |w| and max |u|.  The push
// gathers from the packed grid.

// q = p in tile order and no permutation, or p itself and the bins of its tiles
static const int32_t* bin_particles(aw_ctx& c, const aw_particles& p, aw_particles& q,
                                    hipStream_t s) {
    if (tile_sorted_copy(c, p, false, q, s)) return nullptr;
    q = p;
    c.sort.bin_off.reserve((size_t)c.ntiles + 1);
    c.sort.bin_perm.reserve((size_t)std::max<int64_t>(1, p.n));
    bin_tiles(c, p, c.sort.bin_perm.get(), c.sort.bin_off.get(), s);
    return c.sort.bin_perm.get();
}

static void measure_scales(aw_ctx& c, const aw_particles& p, double qm, hipStream_t s) {
    EmScratch& e = c.em;
    e.cq.reserve(3);
    e.inv.reserve(11);
    e.dv.reserve(2);
    const int most = 4 * std::max(1, c.num_cu);
    const int nb = (int)std::clamp<int64_t>((p.n + kThreads - 1) / kThreads, 1, most);
    e.bound.reserve((size_t)2 * most);
    moment_bound_kernel<<<nb, kThreads, 0, s>>>(p.ux, p.uy, p.uz, p.w, (int)p.n, e.bound.get());
    AW_LAUNCH_CHECK();
    moment_scale_kernel<<<1, kScaleThreads, 0, s>>>(e.bound.get(), nb, p.w ? 1 : 0, qm,
                                                    c.g.dx * c.g.dy, p.w_uniform, e.cq.get(),
                                                    e.inv.get(), e.dv.get());
    AW_LAUNCH_CHECK();
}

void deposit_rho_j_amu(aw_ctx& c, const aw_particles& p, double qm, float* const out[8],
                       hipStream_t s) {
    if (p.n == 0) return;
    AW_REQUIRE(p.n < (int64_t)INT32_MAX, "particle count must fit int32");
    const int64_t nc = ncell(c);
    EmScratch& e = c.em;
    e.acc.reserve((size_t)(8 * nc));
    AW_HIP(hipMemsetAsync(e.acc.get(), 0, (size_t)(8 * nc) * sizeof(unsigned long long), s));
    measure_scales(c, p, qm, s);  // its scratch before the copy of the particles
    aw_particles q;
    const int32_t* idx = bin_particles(c, p, q, s);
    em_moments(c, q, c.sort.bin_off.get(), idx, e.acc.get(), e.cq.get(),
               em_moments_bpt(c, p.n, 1), nullptr, s, EmBatch{});
    Out8 o{};
    for (int q = 0; q < 8; ++q) o.o[q] = out[q];
    convert_add_kernel<<<blocks_for(nc), kThreads, 0, s>>>(e.acc.get(), o, (int)nc, 8, e.inv.get());
    AW_LAUNCH_CHECK();
}

void deposit_dcu(aw_ctx& c, const aw_particles& p, double qm, const float* const* F,
                 float* const out[3], hipStream_t s) {
    if (p.n == 0) return;
    AW_REQUIRE(p.n < (int64_t)INT32_MAX, "particle count must fit int32");
    const int64_t nc = ncell(c);
    EmScratch& e = c.em;
    e.acc.reserve((size_t)(8 * nc));
    e.cdcu.reserve(1);
    e.fpart.reserve(512);
    AW_HIP(hipMemsetAsync(e.acc.get(), 0, (size_t)(3 * nc) * sizeof(unsigned long long), s));
    measure_scales(c, p, qm, s);  // its scratch before the copy of the particles
    aw_particles q;
    const int32_t* idx = bin_particles(c, p, q, s);
    const double mult = p.w ? 1.0 : p.w_uniform;
    dcu_scale(F, nc, e.fpart.get(), 0.0, qm * qm * mult / (c.g.dx * c.g.dy), 0.0, e.dv.get(),
              e.cdcu.get(), e.inv.get() + 8, s, 1, 0, 0, 0);
    em_dcu(c, q, c.sort.bin_off.get(), idx, F, e.acc.get(), e.cdcu.get(),
           tile_bpt(c, p.n), nullptr, s, EmBatch{});
    Out8 o{};
    for (int q = 0; q < 3; ++q) o.o[q] = out[q];
    convert_add_kernel<<<blocks_for(nc), kThreads, 0, s>>>(e.acc.get(), o, (int)nc, 3,
                                                            e.inv.get() + 8);
    AW_LAUNCH_CHECK();
}

void push_boris_em(aw_ctx& c, const aw_particles& p, double qm, double dt, const float* const* F,
                   hipStream_t s) {
    if (p.n == 0) return;
    AW_REQUIRE(p.n < (int64_t)INT32_MAX, "particle count must fit int32");
    const int64_t nc = ncell(c);
    c.fpack.reserve((size_t)(8 * nc));
    float4* pk = reinterpret_cast<float4*>(c.fpack.get());
    em_pack_kernel<<<blocks_for(nc), kThreads, 0, s>>>(F[0], F[1], F[2], F[3], F[4], F[5],
                                                       (int)nc, pk);
    AW_LAUNCH_CHECK();
    em_push_any_kernel<<<blocks_for(p.n), kThreads, 0, s>>>(
        p.x, p.y, p.ux, p.uy, p.uz, (int)p.n, c.g.nx, c.g.ny, pk, (float)(qm * 0.5 * dt),
        (float)(dt / c.g.dx), (float)(dt / c.g.dy));
    AW_LAUNCH_CHECK();
}

}  // namespace aw
