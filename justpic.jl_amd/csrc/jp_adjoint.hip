// jp_adjoint.hip -- reverse mode of advection! + particle2grid! on a flat
// particle list (no reference counterpart: JustPIC.jl has no adjoint).
//
// Forward model, per particle: nsteps steps of the reference's integrator
// (src/Particles/Advection/advection.jl:66-91 with Euler.jl, RK2.jl, RK4.jl;
// same operations and fma placement as jp_advect.hip), deletion when the new
// position is not strictly inside the domain (src/Particles/move_safe.jl:
// 99-103), then the particle2grid! gather (src/Interpolations/
// particle_to_grid.jl:37-68, 113-151) of the survivors: each node sums
// w = inv(distance^2) and w*T over the particles of its 2^D adjacent cells.
// Brackets are seeded at the uniform-spacing estimate; for a point strictly
// inside one interval every seed gives the same bracket.
//
// Kernels, one thread per particle:
//  - k_adj_fwd: the whole trajectory in registers; the position at the start
//    of every block of `every` steps goes to the checkpoint array; survivors
//    record their final cell and count themselves into it.
//  - particle2grid! of the survivors without float atomics: the per-cell
//    counts are scanned, particle ids are bucketed by cell and each bucket is
//    put in order of id, with its positions and tracers; every node then merges
//    the buckets of its 2^D cells and accumulates w and fma(w, T, .) in
//    increasing particle id, the order of the oracle's restatement, so F and W
//    are reproducible and equal to it bit for bit.
//  - k_adj_bwd: blocks of steps in reverse order; a block is recomputed from
//    its checkpoint into a tape (the position at the start of each step, in
//    global scratch), then reversed step by step.  x0bar and Tpbar are per-thread
//    values.
// In 2D both trajectory kernels read the velocities and axes of a workgroup's
// block of steps from a window in LDS, and the pullback sums its velocity
// cotangents there (LDS atomic adds) before it adds them to Vbar once; see Window.
// The adjoint is the exact derivative of the forward model on the branch the
// forward pass takes (brackets, cells and survivors fixed): the n-linear
// interpolation's weights and slopes, the integrator's stage weights, and for
// the gather dF/dw = (T - F)/W, dw/dx = -2 (x - x_node) w^2 (w taken as
// 1/|x - x_node|^2).  Operation order matches the oracle's restatement, so
// x0bar and Tpbar agree with it bit for bit given the same F, W and Fbar.
#include "jp_ctx.hpp"
#include "jp_splitmath.hpp"

#include <cmath>

using namespace jp;

namespace {

template <int D>
struct AdjArgs {
    Grid<D> G;
    Vel<D> vg;
    const double* V[D];
    double dt;
    double adt;  // (1*alpha)*dt, first RK2 stage
    double w0;   // muladd(-0.5, inv(alpha), 1)
    double w1;   // 0.5*inv(alpha)
    int half;    // alpha == 0.5
    int nsteps;
    int every;
    int64_t np;
    int64_t nn[D];  // nodes per dimension
};

// interval of p by the uniform spacing 1/i0 from x0, any p: the hardware's conversion
// saturates and gives 0 for NaN, where C++ leaves the result open (clamped before a C++
// conversion: pullback of RK4 2 to 3% slower)
__device__ inline int estimate(double p, double x0, double i0) {
    int e;
    asm("v_cvt_i32_f64_e32 %0, %1" : "=v"(e) : "v"((p - x0) * i0));
    return e;
}

// bracket of p, which lies in [x[0], x[n-1]], seeded at the uniform estimate (outside
// the search ends at an end interval, but not early)
__device__ inline int64_t adj_bracket(double p, const Axis& A) {
    const int64_t last = A.n - 2, s = estimate(p, A.x[0], A.idx[0]);
    return find_cell(p, A, s < 0 ? 0 : (s > last ? last : s));
}

// The velocity window of a workgroup and block of steps (2D): component c's nodes
// lo[c] .. lo[c] + ext[c] - 1 per dimension.  In LDS lie the cotangent tile (the
// components one after the other, c's at off[c]; `tiled`), and, where that fits as
// well (`staged`), the velocities in the same order at `vo` and each axis's x and
// idx at ax[c][d] and ax[c][d] + ext[c][d].  Points outside the window, and all
// points of a footprint too large for it, take global loads and global FP64
// atomic adds.
// Particles of a patch disperse over a block (64 lanes from 4 to 28 cache lines of
// velocities in 100 steps), and every one of those lines is a cycle of the CU's
// address unit for each of the 16 loads of a velocity: 1 M particles, 100 RK2
// steps, checkpoints every 10: pullback 7.18 ms and forward 1.64 ms with global
// loads, 3.20 and 1.07 with windows (1200 and 200 cycles per CU, wavefront and
// step, most of them the LDS's: its 48 loads and 16 adds of a reversed step).
// (The array is named, not pointed to: a pointer that may be null makes the adds
// flat ones, 7.61 ms for 7.18.)
extern __shared__ double adj_lds[];

template <int D>
struct Window {
    double* g[D];  // Vbar
    bool staged, tiled;
    int vo;
    int lo[D][D], ext[D][D], off[D], ax[D][D];
    double x0[D][D], i0[D][D];  // x[0] and idx[0] of every axis
};

// lower corner, values, local coordinates and inverse spacings of a point's
// interval in component c
template <int D>
struct Corners {
    int64_t at;  // lower corner: index in the tile (in) or in the component's array
    double v[1 << D];
    double t[D];
    double iv[D];
    bool in;     // the corners lie in the tile
};

template <int D>
__device__ inline void gather_global(const AdjArgs<D>& A, const Window<D>& Wn, int c,
                                     const double (&p)[D], Corners<D>& K) {
    int64_t k[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const Axis& X = A.vg.ax[c][d];
        k[d] = adj_bracket(p[d], X);
        K.iv[d] = X.idx[k[d]];
        K.t[d] = (p[d] - X.x[k[d]]) * K.iv[d];
    }
    const int64_t n0 = A.vg.ax[c][0].n, n1 = A.vg.ax[c][1].n;
    const double* __restrict__ Vc = A.V[c];
    K.at = k[0] + n0 * (k[1] + n1 * (D == 3 ? k[D - 1] : 0));
#pragma unroll
    for (int q = 0; q < (1 << D); ++q)
        K.v[q] = Vc[K.at + (q & 1) + n0 * (((q >> 1) & 1) + n1 * ((q >> 2) & 1))];
    K.in = false;
    if constexpr (D == 2) {
        if (Wn.tiled) {
            const unsigned a = (unsigned)((int)k[0] - Wn.lo[c][0]);
            const unsigned b = (unsigned)((int)k[1] - Wn.lo[c][1]);
            if (a < (unsigned)(Wn.ext[c][0] - 1) && b < (unsigned)(Wn.ext[c][1] - 1)) {
                K.in = true;
                K.at = Wn.off[c] + (int)a + Wn.ext[c][0] * (int)b;
            }
        }
    }
}

// corners of interval s of the window; true when p lies strictly inside it
__device__ inline bool gather_window(const Window<2>& Wn, int c, const double (&p)[2],
                                     const int (&s)[2], Corners<2>& K) {
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        const double* __restrict__ x = adj_lds + Wn.ax[c][d] + s[d];
        const double xa = x[0], xb = x[1];
        K.iv[d] = x[Wn.ext[c][d]];
        K.t[d] = (p[d] - xa) * K.iv[d];
        ok = ok && xa < p[d] && p[d] < xb;
    }
    const int e0 = Wn.ext[c][0], at = Wn.off[c] + s[0] + e0 * s[1];
    const double* __restrict__ v = adj_lds + Wn.vo + at;
    K.v[0] = v[0];
    K.v[1] = v[1];
    K.v[2] = v[e0];
    K.v[3] = v[e0 + 1];
    K.at = at;
    K.in = true;
    return ok;
}

// interval of p among the n nodes x of a window axis (its last one or its first
// where p lies outside)
__device__ inline int window_search(const double* __restrict__ x, int n, double p) {
    int a = 0, b = n - 1;
    while (b - a > 1) {
        const int m = (a + b) >> 1;
        if (x[m] <= p)
            a = m;
        else
            b = m;
    }
    return a;
}

template <int D>
__device__ inline bool in_limits(const AdjArgs<D>& A, const Window<D>& Wn, int c,
                                 const double (&p)[D]) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const Axis& X = A.vg.ax[c][d];
        if (!(Wn.x0[c][d] <= p[d] && p[d] <= X.x[X.n - 1])) return false;
    }
    return true;
}

// corners of p in component c; true for a point known to be inside its grid.  LIMITS:
// K is set for those only, else always.  In the window the interval is the one at the uniform
// spacing's estimate when p lies strictly inside it, as in adj_bracket, else the one a
// bisection finds; a point strictly inside an interval is inside the grid.  Where the
// estimate misses, the limits come before any search, since no search ends early on a
// point outside: 256 x 256 cells, 1 M particles carried out of the grid, 40 steps:
// forward RK2 4.55 ms and RK4 33.0 with the searches first, now XXX.
template <int D, bool LIMITS>
__device__ inline bool gather(const AdjArgs<D>& A, const Window<D>& Wn, int c,
                              const double (&p)[D], Corners<D>& K) {
    if constexpr (D == 2) {
        if (Wn.staged) {
            int s[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const int e = estimate(p[d], Wn.x0[c][d], Wn.i0[c][d]), lo = Wn.lo[c][d];
                s[d] = min(max(e, lo), lo + Wn.ext[c][d] - 2) - lo;
            }
            if (gather_window(Wn, c, p, s, K)) return true;
        }
    }
    if (LIMITS && !in_limits(A, Wn, c, p)) return false;
    if constexpr (D == 2) {
        if (Wn.staged) {
            int s[2];
#pragma unroll
            for (int d = 0; d < 2; ++d)
                s[d] = window_search(adj_lds + Wn.ax[c][d], Wn.ext[c][d], p[d]);
            if (gather_window(Wn, c, p, s, K)) return true;
        }
    }
    gather_global(A, Wn, c, p, K);
    return LIMITS;
}

// lerp(v, t) of src/Interpolations/ndlerp.jl:11-15
template <int D>
__device__ inline double lerp_n(const Corners<D>& K) {
    const double* v = K.v;
    const double* t = K.t;
    if constexpr (D == 2) {
        return lerp1(t[1], lerp1(t[0], v[0], v[1]), lerp1(t[0], v[2], v[3]));
    } else {
        const double a = lerp1(t[1], lerp1(t[0], v[0], v[1]), lerp1(t[0], v[2], v[3]));
        const double b = lerp1(t[1], lerp1(t[0], v[4], v[5]), lerp1(t[0], v[6], v[7]));
        return lerp1(t[2], a, b);
    }
}

// velocity component c at p; +Inf outside its grid (check_local_limits,
// src/Advection/advection.jl:83-91)
// LIVE: p is a point of a survivor, inside but for the pullback's FP64 recompute of a
// split trajectory along a boundary, so the corners' loads need not wait for the limits
// (3D, 16^3 cells carried out: pullback 4.02 ms for 3.66)
template <int D, bool LIVE>
__device__ inline double vel_c(const AdjArgs<D>& A, const Window<D>& Wn, int c,
                               const double (&p)[D], Corners<D>& K) {
    const bool inside = gather<D, !LIVE>(A, Wn, c, p, K) || (LIVE && in_limits(A, Wn, c, p));
    return inside ? lerp_n(K) : __builtin_inf();
}

template <int D, bool LIVE>
__device__ inline void vel(const AdjArgs<D>& A, const Window<D>& Wn, const double (&p)[D],
                           double (&v)[D]) {
#pragma unroll
    for (int c = 0; c < D; ++c) {
        Corners<D> K;
        v[c] = vel_c<D, LIVE>(A, Wn, c, p, K);
    }
}

// adjoint of component c at the point of the corners K for the cotangent vb:
// Vbar[c] += weights*vb, pb += slope*vb.  Only called on points the forward pass
// found inside the component's grid.
template <int D>
__device__ inline void vel_c_bw(const AdjArgs<D>& A, const Window<D>& Wn, int c,
                                const Corners<D>& K, double vb, double (&pb)[D]) {
    if (vb == 0.0) return;
    const double* v = K.v;
    const double* t = K.t;
    double dd[D];
    if constexpr (D == 2) {
        dd[0] = (1.0 - t[1]) * (v[1] - v[0]) + t[1] * (v[3] - v[2]);
        dd[1] = (1.0 - t[0]) * (v[2] - v[0]) + t[0] * (v[3] - v[1]);
    } else {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if ((q >> d) & 1) continue;
                const int q1 = q | (1 << d);
                double w = 1.0;
#pragma unroll
                for (int e = 0; e < 3; ++e) {
                    if (e == d) continue;
                    w *= ((q >> e) & 1) ? t[e] : 1.0 - t[e];
                }
                s += w * (v[q1] - v[q]);
            }
            dd[d] = s;
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) pb[d] += dd[d] * K.iv[d] * vb;
    const int64_t n0 = A.vg.ax[c][0].n, n1 = A.vg.ax[c][1].n;
#pragma unroll
    for (int q = 0; q < (1 << D); ++q) {
        double w = 1.0;
#pragma unroll
        for (int d = 0; d < D; ++d) w *= ((q >> d) & 1) ? t[d] : 1.0 - t[d];
        if (K.in)
            unsafeAtomicAdd(adj_lds + (int)K.at + (q & 1) + ((q >> 1) & 1) * Wn.ext[c][0],
                            w * vb);
        else
            unsafeAtomicAdd(
                Wn.g[c] + K.at + (q & 1) + n0 * (((q >> 1) & 1) + n1 * ((q >> 2) & 1)), w * vb);
    }
}
template <int D>
__device__ inline void vel_c_bw(const AdjArgs<D>& A, const Window<D>& Wn, int c,
                                const double (&p)[D], double vb, double (&pb)[D]) {
    if (vb == 0.0) return;
    Corners<D> K;
    gather<D, false>(A, Wn, c, p, K);
    vel_c_bw(A, Wn, c, K, vb, pb);
}

// one step (Euler.jl, RK2.jl with @muladd, RK4.jl unfused)
template <int D, int M, bool LIVE>
__device__ inline void step(const AdjArgs<D>& A, const Window<D>& Wn, const double (&p0)[D],
                            double (&out)[D]) {
    double v0[D];
    vel<D, LIVE>(A, Wn, p0, v0);
    if constexpr (M == JP_EULER) {
#pragma unroll
        for (int d = 0; d < D; ++d) out[d] = fma(A.dt, v0[d], p0[d]);
    } else if constexpr (M == JP_RK2) {
        double p1[D], v1[D];
#pragma unroll
        for (int d = 0; d < D; ++d) p1[d] = fma(A.adt, v0[d], p0[d]);
        vel<D, LIVE>(A, Wn, p1, v1);
        if (A.half) {
#pragma unroll
            for (int d = 0; d < D; ++d) out[d] = fma(A.dt, v1[d], p0[d]);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) out[d] = fma(A.dt, fma(A.w1, v1[d], A.w0 * v0[d]), p0[d]);
        }
    } else {
        double q[D], k2[D], k3[D], k4[D];
#pragma unroll
        for (int d = 0; d < D; ++d) q[d] = p0[d] + (A.dt * v0[d]) / 2.0;
        vel<D, LIVE>(A, Wn, q, k2);
#pragma unroll
        for (int d = 0; d < D; ++d) q[d] = p0[d] + (A.dt * k2[d]) / 2.0;
        vel<D, LIVE>(A, Wn, q, k3);
#pragma unroll
        for (int d = 0; d < D; ++d) q[d] = p0[d] + A.dt * k3[d];
        vel<D, LIVE>(A, Wn, q, k4);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const double sum = ((v0[d] + 2.0 * k2[d]) + 2.0 * k3[d]) + k4[d];
            out[d] = p0[d] + (A.dt * sum) / 6.0;
        }
    }
}

// reverse of step at p0: pb is the output's cotangent on entry, p0's on exit
template <int D, int M>
__device__ inline void step_bw(const AdjArgs<D>& A, const Window<D>& Wn, const double (&p0)[D],
                               double (&pb)[D]) {
    double ob[D];
#pragma unroll
    for (int d = 0; d < D; ++d) ob[d] = pb[d];
    if constexpr (M == JP_EULER) {
#pragma unroll
        for (int c = 0; c < D; ++c) vel_c_bw(A, Wn, c, p0, A.dt * ob[c], pb);
    } else if constexpr (M == JP_RK2) {
        double v0[D], p1[D], v0b[D], v1b[D], p1b[D];
        // kept for the reverse at p0, in 2D: four gathers for five (in 3D the
        // registers would halve the wavefronts: 186 for 127)
        Corners<D> K0[D];
#pragma unroll
        for (int c = 0; c < D; ++c) v0[c] = vel_c<D, true>(A, Wn, c, p0, K0[c]);
#pragma unroll
        for (int d = 0; d < D; ++d) p1[d] = fma(A.adt, v0[d], p0[d]);
        if (A.half) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                v1b[d] = A.dt * ob[d];
                v0b[d] = 0.0;
            }
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                v1b[d] = A.dt * A.w1 * ob[d];
                v0b[d] = A.dt * A.w0 * ob[d];
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) p1b[d] = 0.0;
#pragma unroll
        for (int c = 0; c < D; ++c) vel_c_bw(A, Wn, c, p1, v1b[c], p1b);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            pb[d] += p1b[d];
            v0b[d] += A.adt * p1b[d];
        }
#pragma unroll
        for (int c = 0; c < D; ++c) {
            if constexpr (D == 2)
                vel_c_bw(A, Wn, c, K0[c], v0b[c], pb);
            else
                vel_c_bw(A, Wn, c, p0, v0b[c], pb);
        }
    } else {
        double k1[D], k2[D], k3[D], q2[D], q3[D], q4[D], kb[4][D], qb[D];
        vel<D, true>(A, Wn, p0, k1);
#pragma unroll
        for (int d = 0; d < D; ++d) q2[d] = p0[d] + (A.dt * k1[d]) / 2.0;
        vel<D, true>(A, Wn, q2, k2);
#pragma unroll
        for (int d = 0; d < D; ++d) q3[d] = p0[d] + (A.dt * k2[d]) / 2.0;
        vel<D, true>(A, Wn, q3, k3);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            q4[d] = p0[d] + A.dt * k3[d];
            kb[0][d] = A.dt / 6.0 * ob[d];
            kb[1][d] = 2.0 * A.dt / 6.0 * ob[d];
            kb[2][d] = 2.0 * A.dt / 6.0 * ob[d];
            kb[3][d] = A.dt / 6.0 * ob[d];
        }
        // k4 = v(q4), q4 = p0 + dt*k3; k3 = v(q3), q3 = p0 + dt*k2/2; k2 = v(q2), q2 = p0 + dt*k1/2
#pragma unroll
        for (int st = 3; st >= 1; --st) {
            const double(&qs)[D] = st == 3 ? q4 : (st == 2 ? q3 : q2);
            const double fac = st == 3 ? A.dt : A.dt / 2.0;
#pragma unroll
            for (int d = 0; d < D; ++d) qb[d] = 0.0;
#pragma unroll
            for (int c = 0; c < D; ++c) vel_c_bw(A, Wn, c, qs, kb[st][c], qb);
#pragma unroll
            for (int d = 0; d < D; ++d) {
                pb[d] += qb[d];
                kb[st - 1][d] += fac * qb[d];
            }
        }
#pragma unroll
        for (int c = 0; c < D; ++c) vel_c_bw(A, Wn, c, p0, kb[0][c], pb);
    }
}

// strictly inside the domain (move_safe.jl:199-206); NaN and Inf fail
template <int D>
__device__ inline bool indomain(const Grid<D>& G, const double (&p)[D]) {
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const Axis& X = G.xv[d];
        in = in && (X.x[0] < p[d] && p[d] < X.x[X.n - 1]);
    }
    return in;
}

// node q (bit d: +1 along d) of cell k: linear index, coordinates, inv(distance^2)
template <int D>
__device__ inline int64_t node_of(const AdjArgs<D>& A, const int64_t (&k)[D], int q,
                                  const double (&p)[D], double (&xn)[D], double& wi) {
    int64_t N[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        N[d] = k[d] + ((q >> d) & 1);
        xn[d] = A.G.xv[d].x[N[d]];
    }
    // distance (src/Interpolations/utils.jl:9-19), node minus particle
    double e = xn[0] - p[0];
    double s = e * e;
#pragma unroll
    for (int d = 1; d < D; ++d) {
        e = xn[d] - p[d];
        s = s + e * e;
    }
    const double dist = sqrt(s);
    wi = 1.0 / (dist * dist);
    return D == 2 ? N[0] + A.nn[0] * N[1] : N[0] + A.nn[0] * (N[1] + A.nn[1] * N[D - 1]);
}

// threads of the largest workgroup with a window: 16 wavefronts
constexpr int kWindowBlock = 1024;

__device__ inline double uniform(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return __longlong_as_double((int64_t)(((uint64_t)hi << 32) | lo));
}

// window index r -> component, column, row (r < 2^15: the product's rounding is
// far below the 0.5/ext that r + 0.5 keeps from a row's edge)
__device__ inline void window_node(const Window<2>& Wn, int r, int& c, int& x, int& y) {
    c = r >= Wn.off[1] ? 1 : 0;
    r -= c ? Wn.off[1] : 0;
    const int e = c ? Wn.ext[1][0] : Wn.ext[0][0];
    y = (int)(((float)r + 0.5f) * (1.0f / (float)e));
    x = r - y * e;
}

template <int D>
__device__ inline void init_window(const AdjArgs<D>& A, Window<D>& Wn) {
#pragma unroll
    for (int c = 0; c < D; ++c) {
        Wn.g[c] = nullptr;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            Wn.x0[c][d] = uniform(A.vg.ax[c][d].x[0]);
            Wn.i0[c][d] = uniform(A.vg.ax[c][d].idx[0]);
        }
    }
    Wn.staged = Wn.tiled = false;
}

// box of the brackets of the positions mn .. mx (the workgroup's, per dimension),
// `margin` intervals wider; what fits of it (with TILE the tile, then the
// velocities and axes) is cleared and loaded.  Called by the whole workgroup;
// returns the tile's nodes (0: no tile).
template <bool TILE>
__device__ inline int open_window(const AdjArgs<2>& A, Window<2>& Wn, const double (&mn)[2],
                                  const double (&mx)[2], int margin, int cap) {
    __shared__ double sred[kWindowBlock / 64][4];
    __shared__ int sbox[2][2][2];
    const int lt = threadIdx.x, B = blockDim.x;
    double m[4] = {mn[0], -mx[0], mn[1], -mx[1]};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m[j] = fmin(m[j], __shfl_xor(m[j], o));
        if ((lt & 63) == 0) sred[lt >> 6][j] = m[j];
    }
    __syncthreads();
    if (lt < 8) {
        const int c = lt >> 2, d = (lt >> 1) & 1, hi = lt & 1;
        double v = sred[0][2 * d + hi];
        for (int w = 1; w < B / 64; ++w) v = fmin(v, sred[w][2 * d + hi]);
        int k = -1;  // no live particle
        if (v < __builtin_inf()) {
            const Axis& X = A.vg.ax[c][d];
            const double p = fmax(X.x[0], fmin(hi ? -v : v, X.x[X.n - 1]));
            const int b = (int)adj_bracket(p, X);
            k = hi ? min(b + 1 + margin, (int)X.n - 1) : max(b - margin, 0);
        }
        sbox[c][d][hi] = k;
    }
    __syncthreads();
    int total = 0, axes = 0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const int lo = __builtin_amdgcn_readfirstlane(sbox[c][d][0]);
            const int hi = __builtin_amdgcn_readfirstlane(sbox[c][d][1]);
            if (lo < 0) return 0;
            Wn.lo[c][d] = lo;
            Wn.ext[c][d] = hi - lo + 1;
        }
        const int64_t sz = (int64_t)Wn.ext[c][0] * Wn.ext[c][1];
        Wn.off[c] = total;
        if (sz > cap) return 0;
        total += (int)sz;
    }
    if (total > cap) return 0;
    Wn.tiled = TILE;
    Wn.vo = TILE ? total : 0;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            Wn.ax[c][d] = Wn.vo + total + axes;
            axes += 2 * Wn.ext[c][d];
        }
    Wn.staged = Wn.vo + total + axes <= cap;
    if (TILE)
        for (int t = lt; t < total; t += B) adj_lds[t] = 0.0;
    if (Wn.staged) {
        for (int t = lt; t < total; t += B) {
            int c, x, y;
            window_node(Wn, t, c, x, y);
            const double* __restrict__ V = c ? A.V[1] : A.V[0];
            const int64_t n = c ? A.vg.ax[1][0].n : A.vg.ax[0][0].n;
            const int lx = c ? Wn.lo[1][0] : Wn.lo[0][0], ly = c ? Wn.lo[1][1] : Wn.lo[0][1];
            adj_lds[Wn.vo + t] = V[lx + x + n * (ly + y)];
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const Axis& X = A.vg.ax[c][d];
                const int lo = Wn.lo[c][d], e = Wn.ext[c][d];
                for (int t = lt; t < e; t += B) {
                    adj_lds[Wn.ax[c][d] + t] = X.x[lo + t];
                    // intervals: one fewer than nodes
                    adj_lds[Wn.ax[c][d] + e + t] = t + 1 < e ? X.idx[lo + t] : 0.0;
                }
            }
    }
    __syncthreads();
    return total;
}

// the tile's nonzero entries go to Vbar; called by the whole workgroup
__device__ inline void close_window(const AdjArgs<2>& A, Window<2>& Wn, int total) {
    __syncthreads();
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        const double v = adj_lds[t];
        if (v == 0.0) continue;
        int c, x, y;
        window_node(Wn, t, c, x, y);
        const int64_t n = c ? A.vg.ax[1][0].n : A.vg.ax[0][0].n;
        const int lx = c ? Wn.lo[1][0] : Wn.lo[0][0], ly = c ? Wn.lo[1][1] : Wn.lo[0][1];
        unsafeAtomicAdd((c ? Wn.g[1] : Wn.g[0]) + lx + x + n * (ly + y), v);
    }
    __syncthreads();  // the tile is reused by the next block
    Wn.staged = Wn.tiled = false;
}

// 2D: the velocities of a block of steps from LDS windows (80 KB: two workgroups
// of 16 wavefronts per CU), sized for a straight line on from the block before
// (before the first: along the velocity at the start).
constexpr int kFwd2 = 512;
constexpr size_t kFwdLds = 80 * 1024 - 1024;  // less the static words
template <int D, int M>
__global__ __launch_bounds__(D == 2 ? kFwd2 : kBlock, D == 2 ? 4 : 1) void k_adj_fwd(
    AdjArgs<D> A, CPtr3 x0, double* __restrict__ ckpt, uint8_t* __restrict__ alive, Ptr3 xN,
    int32_t* __restrict__ cell, int32_t* __restrict__ cnt, int cap) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool own = i < A.np;  // every thread reaches the block-wide barriers
    if (D == 3 && !own) return;
    Window<D> Wn;
    init_window(A, Wn);
    double x[D], go[D];  // position, displacement expected of the block
#pragma unroll
    for (int d = 0; d < D; ++d) {
        x[d] = own ? x0.p[d][i] : 0.0;
        go[d] = 0.0;
    }
    bool a = own && indomain(A.G, x);
    if (D == 2 && a) {
        double v[D];
        vel<D, false>(A, Wn, x, v);
#pragma unroll
        for (int d = 0; d < D; ++d) go[d] = (A.every < A.nsteps ? A.every : A.nsteps) * (A.dt * v[d]);
    }
    for (int s0 = 0;; s0 += A.every) {
        if (own) {
#pragma unroll
            for (int d = 0; d < D; ++d)
                ckpt[((int64_t)(s0 / A.every) * D + d) * A.np + i] = x[d];
        }
        const int n = A.nsteps - s0 < A.every ? A.nsteps - s0 : A.every;
        if (n <= 0) break;
        if constexpr (D == 2) {
            double mn[2], mx[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                mn[d] = a ? fmin(x[d], x[d] + go[d]) : __builtin_inf();
                mx[d] = a ? fmax(x[d], x[d] + go[d]) : -__builtin_inf();
            }
            open_window<false>(A, Wn, mn, mx, 1, cap);
        }
#pragma unroll
        for (int d = 0; d < D; ++d) go[d] = -x[d];
        for (int j = 0; j < n && a; ++j) {
            double y[D];
            step<D, M, false>(A, Wn, x, y);
#pragma unroll
            for (int d = 0; d < D; ++d) x[d] = y[d];
            a = indomain(A.G, x);
        }
#pragma unroll
        for (int d = 0; d < D; ++d) go[d] += x[d];
        if (s0 + A.every >= A.nsteps) break;
        if constexpr (D == 2) {
            __syncthreads();  // the window is reused
            Wn.staged = false;
        }
    }
    if (!own) return;
    alive[i] = a ? 1 : 0;
#pragma unroll
    for (int d = 0; d < D; ++d) xN.p[d][i] = x[d];
    int32_t c = -1;
    if (a) {
        int64_t k[D];
#pragma unroll
        for (int d = 0; d < D; ++d) k[d] = adj_bracket(x[d], A.G.xv[d]);
        c = (int32_t)lin<D>(A.G.ni, k);
        atomicAdd(cnt + c, 1);
    }
    cell[i] = c;
}

// The forward model in the FP32-split form (jp_adjoint_forward_split): each
// particle is a cell index plus a float32 offset in cell units, every step
// the split advection's per-particle arithmetic (jp_splitmath.hpp: velocity
// scaled to cells per step in float32, every corner read from global memory,
// the same values a split advection window holds) followed by the split
// move's renormalisation to the destination cell in FP64; a particle whose
// cell leaves the grid, or whose offset is not finite, is deleted.  The
// checkpoints, xN and the gather use the FP64 position x_I + u*h, so the
// FP64 backward recomputes each block from the split trajectory.
template <int D, int M>
__global__ __launch_bounds__(kBlock) void k_adj_fwd_split(
    AdjArgs<D> A, split::SVelIn<D> SV, const SplitGeom* __restrict__ geo, split::RKf P, CPtr3 x0,
    double* __restrict__ ckpt, uint8_t* __restrict__ alive, Ptr3 xN, int32_t* __restrict__ cell,
    int32_t* __restrict__ cnt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= A.np || geo->bad) return;  // a rejected grid is reported by the call
    split::SMap<D> m;
    double sc[D];
#pragma unroll
    for (int c = 0; c < D; ++c) {
        sc[c] = A.dt / A.G.xv[c].dx[0];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            m.r[c][d] = geo->r[c][d];
            m.o[c][d] = geo->o[c][d];
        }
    }
    double x[D];
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = x0.p[d][i];
    bool a = indomain(A.G, x);
    int I[D];
    float u[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        I[d] = 0;
        u[d] = 0.0f;
        if (a) {
            const Axis& X = A.G.xv[d];
            I[d] = (int)adj_bracket(x[d], X);
            const double ud = (x[d] - X.x[I[d]]) * X.idx[I[d]];
            float uf = (float)ud;
            if (ud < 1.0 && uf >= 1.0f) uf = 0x1.fffffep-1f;  // stays inside its cell
            u[d] = uf;
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) ckpt[(int64_t)d * A.np + i] = x[d];
    int64_t blk = 0;
    int left = A.every;
    for (int s = 0; s < A.nsteps; ++s) {
        if (left == 0) {
            ++blk;
            left = A.every;
#pragma unroll
            for (int d = 0; d < D; ++d) ckpt[(blk * D + d) * A.np + i] = x[d];
        }
        --left;
        if (!a) continue;
        split::CellMap<D> cm;
        split::cell_map<D, false>(m, I, cm);
        float out[D];
        split::advect_split_one<D, M>(split::GlobalVelocity<D>{SV, sc, I, cm}, P, u, out);
        bool gone = false;
        int sd[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const bool fin = fabsf(out[d]) < 1.0e6f;  // false for NaN/Inf
            sd[d] = fin ? (int)floorf(out[d]) : 0;
            const int J = I[d] + sd[d];
            gone = gone || !fin || J < 0 || J >= A.G.ni[d];
        }
        if (gone) {  // deleted: the last position, as the FP64 model keeps it
#pragma unroll
            for (int d = 0; d < D; ++d)
                x[d] = A.G.xv[d].x[I[d]] + (double)out[d] * A.G.xv[d].dx[I[d]];
            a = false;
            continue;
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            I[d] += sd[d];
            u[d] = (float)((double)out[d] - (double)sd[d]);
            x[d] = A.G.xv[d].x[I[d]] + (double)u[d] * A.G.xv[d].dx[I[d]];
        }
    }
    alive[i] = a ? 1 : 0;
#pragma unroll
    for (int d = 0; d < D; ++d) xN.p[d][i] = x[d];
    int32_t c = -1;
    if (a) {
        int64_t k[D];
#pragma unroll
        for (int d = 0; d < D; ++d) k[d] = I[d];
        c = (int32_t)lin<D>(A.G.ni, k);
        atomicAdd(cnt + c, 1);
    }
    cell[i] = c;
}

// exclusive scan of the C cell counts into start[0..C], kScan counts per workgroup:
// the workgroups' sums, then each one's scan from the sum of those before it (one
// workgroup for all, a chunk per thread, took 110 us for 65536 cells; the two 10)
constexpr int kScan = 2048;
__device__ inline int32_t scan_chunk(const int32_t* __restrict__ cnt, int64_t C, int64_t c,
                                     int32_t (&v)[kScan / kBlock]) {
    int32_t s = 0;
#pragma unroll
    for (int j = 0; j < kScan / kBlock; ++j) {
        v[j] = c + j < C ? cnt[c + j] : 0;
        s += v[j];
    }
    return s;
}
__device__ inline int32_t block_sum(int32_t s, int32_t* part) {  // all threads; part: a word per wave
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    int32_t r = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) r += part[w];
    __syncthreads();
    return r;
}
__global__ __launch_bounds__(kBlock) void k_adj_sums(const int32_t* __restrict__ cnt,
                                                     int32_t* __restrict__ sums, int64_t C) {
    __shared__ int32_t part[kBlock / 64];
    int32_t v[kScan / kBlock];
    const int64_t c = blockIdx.x * (int64_t)kScan + threadIdx.x * (kScan / kBlock);
    const int32_t s = block_sum(scan_chunk(cnt, C, c, v), part);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}
__global__ __launch_bounds__(kBlock) void k_adj_starts(const int32_t* __restrict__ cnt,
                                                       const int32_t* __restrict__ sums,
                                                       int32_t* __restrict__ start, int64_t C) {
    __shared__ int32_t part[kBlock / 64];
    int32_t before = 0;
    for (unsigned b = threadIdx.x; b < blockIdx.x; b += kBlock) before += sums[b];
    before = block_sum(before, part);
    int32_t v[kScan / kBlock];
    const int64_t c = blockIdx.x * (int64_t)kScan + threadIdx.x * (kScan / kBlock);
    const int32_t s = scan_chunk(cnt, C, c, v);
    int32_t incl = s;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int32_t u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
    }
    if (lane == 63) part[threadIdx.x >> 6] = incl;
    __syncthreads();
    int32_t run = before + incl - s;
    for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) run += part[w];
#pragma unroll
    for (int j = 0; j < kScan / kBlock; ++j) {
        if (c + j < C) start[c + j] = run;
        run += v[j];
        if (c + j == C - 1) start[C] = run;
    }
}

// bucket the survivors by cell (order inside a bucket fixed by k_adj_order);
// consumes the counts
__global__ __launch_bounds__(kBlock) void k_adj_bucket(const int32_t* __restrict__ cell,
                                                      int32_t* __restrict__ cnt,
                                                      const int32_t* __restrict__ start,
                                                      int32_t* __restrict__ list, int64_t np) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const int32_t c = cell[i];
    if (c < 0) return;
    const int32_t slot = atomicSub(cnt + c, 1) - 1;
    list[start[c] + slot] = (int32_t)i;
}

// every bucket in order of particle id, with the positions and tracers (a thread
// per survivor counts the smaller ids of its bucket, which holds tens): what the
// gather reads then lies together
template <int D>
__global__ __launch_bounds__(kBlock) void k_adj_order(const int32_t* __restrict__ cell,
                                                     const int32_t* __restrict__ start,
                                                     const int32_t* __restrict__ list,
                                                     CPtr3 xN, const double* __restrict__ Tp,
                                                     int64_t C, int32_t* __restrict__ ids,
                                                     Ptr3 xs, double* __restrict__ Ts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= start[C]) return;
    const int32_t id = list[i];
    const int32_t c = cell[id];
    const int32_t lo = start[c], hi = start[c + 1];
    double x[D];
#pragma unroll
    for (int d = 0; d < D; ++d) x[d] = xN.p[d][id];
    const double T = Tp[id];
    int32_t at = lo;
    for (int32_t j = lo; j < hi; ++j) at += list[j] < id ? 1 : 0;
    ids[at] = id;
#pragma unroll
    for (int d = 0; d < D; ++d) xs.p[d][at] = x[d];
    Ts[at] = T;
}

// per node: merge the id-sorted buckets of its 2^D cells; w = inv(distance^2),
// W += w, S = fma(w, T, S) in increasing particle id; F = S / W (2D),
// S * inv(W) (3D); a node without particles gets 0/0 = NaN.  The heads of the
// buckets are in registers, and the one taken is replaced by its successor, one
// load from where its bucket lies (the ids' list and then the particle's own
// arrays: two dependent loads far apart, 165 us for 257 x 257 nodes of 1 M
// particles, with the sort 231; now with the order 144).
template <int D>
__global__ __launch_bounds__(kBlock) void k_adj_gather(AdjArgs<D> A,
                                                      const int32_t* __restrict__ start,
                                                      const int32_t* __restrict__ ids, CPtr3 xs,
                                                      const double* __restrict__ Ts,
                                                      double* __restrict__ F,
                                                      double* __restrict__ W, int64_t nodes) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nodes) return;
    constexpr int NQ = 1 << D;
    constexpr int32_t kNone = 0x7fffffff;
    int64_t N[D];
    int64_t r = n;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        N[d] = r % A.nn[d];
        r /= A.nn[d];
    }
    double xn[D];
#pragma unroll
    for (int d = 0; d < D; ++d) xn[d] = A.G.xv[d].x[N[d]];
    int32_t h[NQ], e[NQ], id[NQ];
    double x[NQ][D], T[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int64_t I[D];
        bool ok = true;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            I[d] = N[d] - ((q >> d) & 1);
            ok = ok && I[d] >= 0 && I[d] < A.G.ni[d];
        }
        h[q] = e[q] = 0;
        if (ok) {
            const int64_t c = lin<D>(A.G.ni, I);
            h[q] = start[c];
            e[q] = start[c + 1];
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        id[q] = kNone;
        T[q] = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) x[q][d] = 0.0;
        if (h[q] < e[q]) {
            id[q] = ids[h[q]];
#pragma unroll
            for (int d = 0; d < D; ++d) x[q][d] = xs.p[d][h[q]];
            T[q] = Ts[h[q]];
        }
    }
    double w = 0.0, s = 0.0;
    for (;;) {
        int32_t first = id[0];
#pragma unroll
        for (int q = 1; q < NQ; ++q) first = id[q] < first ? id[q] : first;
        if (first == kNone) break;
        double p[D], t = T[0];
        int32_t nx = h[0], end = e[0];
#pragma unroll
        for (int d = 0; d < D; ++d) p[d] = x[0][d];
#pragma unroll
        for (int q = 1; q < NQ; ++q) {
            const bool m = id[q] == first;
            t = m ? T[q] : t;
            nx = m ? h[q] : nx;
            end = m ? e[q] : end;
#pragma unroll
            for (int d = 0; d < D; ++d) p[d] = m ? x[q][d] : p[d];
        }
        // its successor (the last one again at the bucket's end: not used)
        nx += 1;
        const bool more = nx < end;
        const int32_t at = more ? nx : nx - 1;
        const int32_t idn = ids[at];
        double pn[D];
#pragma unroll
        for (int d = 0; d < D; ++d) pn[d] = xs.p[d][at];
        const double tn = Ts[at];
        // distance (src/Interpolations/utils.jl:9-19), node minus particle
        double dl = xn[0] - p[0];
        double ss = dl * dl;
#pragma unroll
        for (int d = 1; d < D; ++d) {
            dl = xn[d] - p[d];
            ss = ss + dl * dl;
        }
        const double dist = sqrt(ss);
        const double wi = 1.0 / (dist * dist);
        w += wi;
        s = fma(wi, t, s);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const bool m = id[q] == first;
            h[q] = m ? nx : h[q];
            T[q] = m ? tn : T[q];
#pragma unroll
            for (int d = 0; d < D; ++d) x[q][d] = m ? pn[d] : x[q][d];
            id[q] = m ? (more ? idn : kNone) : id[q];
        }
    }
    W[n] = w;
    F[n] = D == 2 ? s / w : s * (1.0 / w);
}

__global__ __launch_bounds__(kBlock) void k_adj_zero(double* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// Backward workgroups.  2D: the LDS of a CU holds the window of one workgroup, so
// a workgroup has as many particles as spread the list over the CUs, up to 1024
// (16 wavefronts, what 128 registers allow); a list from compact patches touches
// 1.3-8 k nodes of both components in ten steps of CFL 1, patches of 1024 as many
// as of 512 (the cells' rows and the flow set the extent).  3D: no window.
constexpr int kBwd3 = 512;
constexpr size_t kLdsBudget = 160 * 1024 - 1024;  // less the static words

template <int D, int M>
__global__ __launch_bounds__(D == 2 ? kWindowBlock : kBwd3) void k_adj_bwd(
    AdjArgs<D> A, const double* __restrict__ ckpt, const uint8_t* __restrict__ alive,
    const double* __restrict__ Tp, const double* __restrict__ F, const double* __restrict__ W,
    const double* __restrict__ Fbar, Ptr3 Vb, Ptr3 x0b, double* __restrict__ Tpb,
    double* __restrict__ tape, int cap) {
    // tape (global scratch, [every][D][threads of the grid]): step-start positions
    // of the block of steps being reversed; dynamic LDS: the window (cap doubles)
    const int lt = threadIdx.x;
    const int64_t nt = (int64_t)gridDim.x * blockDim.x;
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + lt;
    const int nblk = A.nsteps == 0 ? 1 : (A.nsteps + A.every - 1) / A.every;
    Window<D> Wn;
    init_window(A, Wn);
#pragma unroll
    for (int c = 0; c < D; ++c) Wn.g[c] = Vb.p[c];
    for (int64_t first = (int64_t)blockIdx.x * blockDim.x; first < A.np; first += nt) {
        const int64_t i = first + lt;
        // every thread reaches the block-wide barriers below
        const bool live = i < A.np && alive[i];
        double pb[D];
#pragma unroll
        for (int d = 0; d < D; ++d) pb[d] = 0.0;
        double tb = 0.0;
        for (int b = nblk - 1; b >= 0; --b) {
            const int s0 = b * A.every;
            const int n = A.nsteps - s0 < A.every ? A.nsteps - s0 : A.every;
            double x[D];
            if (live) {
#pragma unroll
                for (int d = 0; d < D; ++d) x[d] = ckpt[((int64_t)b * D + d) * A.np + i];
            }
            int total = 0;
            if constexpr (D == 2) {
                // where the block begins and ends: the next block's start; for the
                // last block a straight line on from the one before.  Points beyond
                // it (a bend of the path) are few and take the global path.
                double mn[2], mx[2];
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    mn[d] = __builtin_inf();
                    mx[d] = -__builtin_inf();
                    if (live && n > 0) {
                        double e = x[d];
                        if (b + 1 < nblk)
                            e = ckpt[((int64_t)(b + 1) * 2 + d) * A.np + i];
                        else if (b > 0)
                            e += (x[d] - ckpt[((int64_t)(b - 1) * 2 + d) * A.np + i]) *
                                 ((double)n / (double)A.every);
                        mn[d] = fmin(x[d], e);
                        mx[d] = fmax(x[d], e);
                    }
                }
                total = open_window<true>(A, Wn, mn, mx, nblk == 1 ? n : 1, cap);
            }
            if (live) {
                for (int j = 0; j < n; ++j) {
#pragma unroll
                    for (int d = 0; d < D; ++d) tape[((int64_t)j * D + d) * nt + tid] = x[d];
                    double y[D];
                    step<D, M, true>(A, Wn, x, y);
#pragma unroll
                    for (int d = 0; d < D; ++d) x[d] = y[d];
                }
                if (b == nblk - 1) {
                    // particle2grid! adjoint at the final position x
                    int64_t k[D];
#pragma unroll
                    for (int d = 0; d < D; ++d) k[d] = adj_bracket(x[d], A.G.xv[d]);
                    const double t = Tp[i];
#pragma unroll
                    for (int q = 0; q < (1 << D); ++q) {
                        double xn[D], wi;
                        const int64_t nd = node_of(A, k, q, x, xn, wi);
                        const double iw = 1.0 / W[nd];
                        const double fb = Fbar[nd];
                        tb += fb * wi * iw;
                        const double gw = fb * (t - F[nd]) * iw;
#pragma unroll
                        for (int d = 0; d < D; ++d)
                            pb[d] += gw * (-2.0 * (x[d] - xn[d]) * wi * wi);
                    }
                }
                for (int j = n - 1; j >= 0; --j) {
                    double p0[D];
#pragma unroll
                    for (int d = 0; d < D; ++d) p0[d] = tape[((int64_t)j * D + d) * nt + tid];
                    step_bw<D, M>(A, Wn, p0, pb);
                }
            }
            if constexpr (D == 2) close_window(A, Wn, total);
        }
        if (i < A.np) {
#pragma unroll
            for (int d = 0; d < D; ++d) x0b.p[d][i] = pb[d];
            Tpb[i] = tb;
        }
    }
}

template <int D>
Vel<D> vel_of(const jp_velgrid* vg) {
    Vel<D> V;
    for (int c = 0; c < D; ++c)
        for (int d = 0; d < D; ++d) {
            const jp_axis& a = vg->ax[c][d];
            V.ax[c][d] = Axis{a.x, a.dx, a.inv_dx, a.n};
        }
    return V;
}

int check_args(jp_ctx* ctx, const jp_cellgrid* g, const jp_velgrid* vg, const double* const* V,
               int method, double alpha, int nsteps, int every, int64_t np) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if (!vg || !V) return fail(ctx, JP_ERR_ARG, "null velocity grid or array%s");
    for (int c = 0; c < g->ndim; ++c) {
        if (!V[c]) return fail(ctx, JP_ERR_ARG, "null velocity component%s %lld", "", c);
        for (int d = 0; d < g->ndim; ++d) {
            const jp_axis& a = vg->ax[c][d];
            if (!a.x || !a.dx || !a.inv_dx || a.n < 2)
                return fail(ctx, JP_ERR_ARG, "bad velocity axis%s (component %lld)", "", c);
        }
    }
    if (method < JP_EULER || method > JP_RK4)
        return fail(ctx, JP_ERR_ARG, "unknown integrator%s %lld", "", method);
    if (method == JP_RK2 && !(0.0 < alpha && alpha < 1.0))
        return fail(ctx, JP_ERR_ARG, "Only 0 < α < 1 is supported%s");
    if (nsteps < 0) return fail(ctx, JP_ERR_ARG, "negative step count%s %lld", "", nsteps);
    if (every < 1 || every > JP_ADJ_MAX_EVERY)
        return fail(ctx, JP_ERR_ARG, "checkpoint interval out of range%s %lld", "", every);
    if (np < 0) return fail(ctx, JP_ERR_ARG, "negative particle count%s %lld", "", np);
    if (np >= ((int64_t)1 << 31))  // 32-bit particle ids and launch size
        return fail(ctx, JP_ERR_ARG, "too many particles%s %lld", "", np);
    int64_t C = 1;
    for (int d = 0; d < g->ndim; ++d) C *= g->ni[d];
    if (C >= ((int64_t)1 << 31))  // 32-bit cell ids
        return fail(ctx, JP_ERR_ARG, "too many cells%s %lld", "", C);
    return JP_OK;
}

template <int D>
AdjArgs<D> make_args(const jp_cellgrid* g, const jp_velgrid* vg, const double* const* V,
                     double alpha, double dt, int nsteps, int every, int64_t np) {
    AdjArgs<D> A;
    A.G = to_grid<D>(g);
    A.vg = vel_of<D>(vg);
    for (int c = 0; c < D; ++c) A.V[c] = V[c];
    A.dt = dt;
    A.adt = (1.0 * alpha) * dt;
    A.half = alpha == 0.5;
    const double ia = 1.0 / alpha;
    A.w0 = std::fma(-0.5, ia, 1.0);
    A.w1 = 0.5 * ia;
    A.nsteps = nsteps;
    A.every = every;
    A.np = np;
    for (int d = 0; d < D; ++d) A.nn[d] = g->ni[d] + 1;
    return A;
}

int zero(jp_ctx* ctx, double* p, int64_t n) {
    if (n <= 0) return JP_OK;
    k_adj_zero<<<(unsigned)blocks_for(n), kBlock, 0, ctx->stream>>>(p, n);
    JP_LAUNCHED(ctx);
    return JP_OK;
}

// threads of a workgroup with a window: as many as spread np particles over the
// workgroups that the CUs hold at once, one wavefront at least
int window_block(int64_t np, int held, int most) {
    int B = 64;
    while (B < most && (int64_t)B * held < np) B *= 2;
    return B;
}

template <int D>
int64_t node_count(const jp_cellgrid* g) {
    int64_t n = 1;
    for (int d = 0; d < D; ++d) n *= g->ni[d] + 1;
    return n;
}

// the trajectories (FP64, or the split form with its velocity description,
// RK parameters and the current geometry verdict), then the gather
template <int D>
struct SplitFwd {
    bool on = false;
    split::SVelIn<D> SV;
    split::RKf P;
    const SplitGeom* geo = nullptr;
};

template <int D, int M>
int forward(jp_ctx* ctx, const AdjArgs<D>& A, const double* const* x0, const double* Tp,
            double* ckpt, uint8_t* alive, double* const* xN, double* F, double* W,
            int64_t nodes, const SplitFwd<D>& sf = SplitFwd<D>()) {
    // scratch: counts (C) | bucket starts (C+1) | the scan's sums | cell of each
    // particle | buckets | their ids, positions and tracers in order
    const int64_t C = A.G.C;
    const int64_t scans = (C + kScan - 1) / kScan;
    size_t end = 0;
    auto part = [&](size_t bytes) {
        const size_t at = end;
        end = (end + bytes + 255) & ~(size_t)255;
        return at;
    };
    const size_t o_cnt = part((size_t)C * 4), o_start = part((size_t)(C + 1) * 4);
    const size_t o_sums = part((size_t)scans * 4), o_cell = part((size_t)A.np * 4);
    const size_t o_list = part((size_t)A.np * 4), o_ids = part((size_t)A.np * 4);
    const size_t o_xs = part((size_t)A.np * 8 * D), o_Ts = part((size_t)A.np * 8);
    int rc = ensure_scratch(ctx, end);
    if (rc) return rc;
    char* base = static_cast<char*>(ctx->scratch);
    int32_t* cnt = reinterpret_cast<int32_t*>(base + o_cnt);
    int32_t* start = reinterpret_cast<int32_t*>(base + o_start);
    int32_t* sums = reinterpret_cast<int32_t*>(base + o_sums);
    int32_t* cell = reinterpret_cast<int32_t*>(base + o_cell);
    int32_t* list = reinterpret_cast<int32_t*>(base + o_list);
    int32_t* ids = reinterpret_cast<int32_t*>(base + o_ids);
    double* Ts = reinterpret_cast<double*>(base + o_Ts);
    CPtr3 cxs{{nullptr, nullptr, nullptr}};
    Ptr3 xs{{nullptr, nullptr, nullptr}};
    for (int d = 0; d < D; ++d) {
        xs.p[d] = reinterpret_cast<double*>(base + o_xs) + (int64_t)d * A.np;
        cxs.p[d] = xs.p[d];
    }
    if ((rc = zero_bytes(ctx, cnt, (size_t)C * 4))) return rc;
    CPtr3 xp{{nullptr, nullptr, nullptr}}, xq{{nullptr, nullptr, nullptr}};
    Ptr3 xo{{nullptr, nullptr, nullptr}};
    for (int d = 0; d < D; ++d) {
        xp.p[d] = x0[d];
        xo.p[d] = xN[d];
        xq.p[d] = xN[d];
    }
    if (A.np > 0) {
        if (sf.on) {
            k_adj_fwd_split<D, M><<<(unsigned)blocks_for(A.np), kBlock, 0, ctx->stream>>>(
                A, sf.SV, sf.geo, sf.P, xp, ckpt, alive, xo, cell, cnt);
        } else {
            const int B = D == 2 ? window_block(A.np, 2 * ctx->num_cu, kFwd2) : kBlock;
            const size_t lds = D == 2 ? kFwdLds : 0;
            k_adj_fwd<D, M><<<(unsigned)blocks_for(A.np, B), B, lds, ctx->stream>>>(
                A, xp, ckpt, alive, xo, cell, cnt, (int)(lds / sizeof(double)));
        }
        JP_LAUNCHED(ctx);
    }
    k_adj_sums<<<(unsigned)scans, kBlock, 0, ctx->stream>>>(cnt, sums, C);
    JP_LAUNCHED(ctx);
    k_adj_starts<<<(unsigned)scans, kBlock, 0, ctx->stream>>>(cnt, sums, start, C);
    JP_LAUNCHED(ctx);
    if (A.np > 0) {
        k_adj_bucket<<<(unsigned)blocks_for(A.np), kBlock, 0, ctx->stream>>>(cell, cnt, start,
                                                                             list, A.np);
        JP_LAUNCHED(ctx);
        k_adj_order<D><<<(unsigned)blocks_for(A.np), kBlock, 0, ctx->stream>>>(
            cell, start, list, xq, Tp, C, ids, xs, Ts);
        JP_LAUNCHED(ctx);
    }
    k_adj_gather<D><<<(unsigned)blocks_for(nodes), kBlock, 0, ctx->stream>>>(A, start, ids, cxs,
                                                                            Ts, F, W, nodes);
    JP_LAUNCHED(ctx);
    return sf.on ? split_finish(ctx) : finish(ctx);
}

template <int D, int M>
int backward(jp_ctx* ctx, const AdjArgs<D>& A, const jp_velgrid* vg, const double* ckpt,
             const uint8_t* alive, const double* Tp, const double* F, const double* W,
             const double* Fbar, double* const* Vbar, double* const* x0bar, double* Tpbar) {
    Ptr3 vb{{nullptr, nullptr, nullptr}}, xb{{nullptr, nullptr, nullptr}};
    for (int c = 0; c < D; ++c) {
        int64_t m = 1;
        for (int d = 0; d < D; ++d) m *= vg->ax[c][d].n;
        int rc = zero(ctx, Vbar[c], m);
        if (rc) return rc;
        vb.p[c] = Vbar[c];
        xb.p[c] = x0bar[c];
    }
    if (A.np > 0) {
        // 2D: one workgroup per CU at a time, each going on to further particles
        int B = kBwd3;
        int64_t grid = blocks_for(A.np, B);
        size_t lds = 0;
        if (D == 2) {
            B = window_block(A.np, ctx->num_cu, kWindowBlock);
            grid = std::min<int64_t>(blocks_for(A.np, B), ctx->num_cu);
            lds = kLdsBudget;
        }
        int rc = ensure_scratch(ctx, (size_t)A.every * D * grid * B * sizeof(double));
        if (rc) return rc;
        double* tape = static_cast<double*>(ctx->scratch);
        k_adj_bwd<D, M><<<(unsigned)grid, B, lds, ctx->stream>>>(
            A, ckpt, alive, Tp, F, W, Fbar, vb, xb, Tpbar, tape, (int)(lds / sizeof(double)));
        JP_LAUNCHED(ctx);
    }
    return finish(ctx);
}

int null_ptrs(jp_ctx* ctx, int D, int64_t np, const void* const* list, int n, const char* what) {
    if (np == 0) return JP_OK;
    if (!list) return fail(ctx, JP_ERR_ARG, "null %s", what);
    for (int d = 0; d < n; ++d)
        if (!list[d]) return fail(ctx, JP_ERR_ARG, "null %s pointer %lld", what, d);
    (void)D;
    return JP_OK;
}

}  // namespace

extern "C" int jp_adjoint_forward(jp_ctx* ctx, const jp_cellgrid* g, const jp_velgrid* vg,
                                  const double* const* V, int method, double alpha, double dt,
                                  int nsteps, int every, int64_t np, const double* const* x0,
                                  const double* Tp, double* ckpt, uint8_t* alive,
                                  double* const* xN, double* F, double* W) {
    int rc = check_args(ctx, g, vg, V, method, alpha, nsteps, every, np);
    if (rc) return rc;
    const int D = g->ndim;
    if (!F || !W) return fail(ctx, JP_ERR_ARG, "null nodal output%s");
    if ((rc = null_ptrs(ctx, D, np, (const void* const*)x0, D, "x0"))) return rc;
    if ((rc = null_ptrs(ctx, D, np, (const void* const*)xN, D, "xN"))) return rc;
    if (np > 0 && (!Tp || !ckpt || !alive))
        return fail(ctx, JP_ERR_ARG, "null particle array (Tp, ckpt or alive)%s");
    if (D == 2) {
        const auto A = make_args<2>(g, vg, V, alpha, dt, nsteps, every, np);
        const int64_t nodes = node_count<2>(g);
        if (method == JP_EULER)
            return forward<2, JP_EULER>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes);
        if (method == JP_RK2)
            return forward<2, JP_RK2>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes);
        return forward<2, JP_RK4>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes);
    }
    const auto A = make_args<3>(g, vg, V, alpha, dt, nsteps, every, np);
    const int64_t nodes = node_count<3>(g);
    if (method == JP_EULER)
        return forward<3, JP_EULER>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes);
    if (method == JP_RK2) return forward<3, JP_RK2>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes);
    return forward<3, JP_RK4>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes);
}

namespace {

template <int D>
int forward_split(jp_ctx* ctx, const jp_cellgrid* g, const jp_velgrid* vg,
                  const double* const* V, int method, double alpha, double dt, int nsteps,
                  int every, int64_t np, const double* const* x0, const double* Tp, double* ckpt,
                  uint8_t* alive, double* const* xN, double* F, double* W) {
    const auto A = make_args<D>(g, vg, V, alpha, dt, nsteps, every, np);
    int rc = split_geometry(ctx, g, vg);
    if (rc) return rc;
    SplitFwd<D> sf;
    sf.on = true;
    sf.geo = geo_ptr(ctx);
    for (int c = 0; c < D; ++c) {
        sf.SV.v[c] = V[c];
        for (int d = 0; d < D; ++d) sf.SV.n[c][d] = (int)vg->ax[c][d].n;
    }
    sf.P.alpha = (float)alpha;
    sf.P.half = alpha == 0.5;
    const double ia = 1.0 / alpha;
    sf.P.w0 = (float)std::fma(-0.5, ia, 1.0);
    sf.P.w1 = (float)(0.5 * ia);
    const int64_t nodes = node_count<D>(g);
    if (method == JP_EULER)
        return forward<D, JP_EULER>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes, sf);
    if (method == JP_RK2)
        return forward<D, JP_RK2>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes, sf);
    return forward<D, JP_RK4>(ctx, A, x0, Tp, ckpt, alive, xN, F, W, nodes, sf);
}

}  // namespace

extern "C" int jp_adjoint_forward_split(jp_ctx* ctx, const jp_cellgrid* g, const jp_velgrid* vg,
                                        const double* const* V, int method, double alpha,
                                        double dt, int nsteps, int every, int64_t np,
                                        const double* const* x0, const double* Tp, double* ckpt,
                                        uint8_t* alive, double* const* xN, double* F, double* W) {
    int rc = check_args(ctx, g, vg, V, method, alpha, nsteps, every, np);
    if (rc) return rc;
    if (!F || !W) return fail(ctx, JP_ERR_ARG, "null nodal output%s");
    if ((rc = null_ptrs(ctx, g->ndim, np, (const void* const*)x0, g->ndim, "x0"))) return rc;
    if ((rc = null_ptrs(ctx, g->ndim, np, (const void* const*)xN, g->ndim, "xN"))) return rc;
    if (np > 0 && (!Tp || !ckpt || !alive))
        return fail(ctx, JP_ERR_ARG, "null particle array (Tp, ckpt or alive)%s");
    return g->ndim == 2 ? forward_split<2>(ctx, g, vg, V, method, alpha, dt, nsteps, every, np,
                                           x0, Tp, ckpt, alive, xN, F, W)
                        : forward_split<3>(ctx, g, vg, V, method, alpha, dt, nsteps, every, np,
                                           x0, Tp, ckpt, alive, xN, F, W);
}

extern "C" int jp_adjoint_backward(jp_ctx* ctx, const jp_cellgrid* g, const jp_velgrid* vg,
                                   const double* const* V, int method, double alpha, double dt,
                                   int nsteps, int every, int64_t np, const double* ckpt,
                                   const uint8_t* alive, const double* Tp, const double* F,
                                   const double* W, const double* Fbar, double* const* Vbar,
                                   double* const* x0bar, double* Tpbar) {
    int rc = check_args(ctx, g, vg, V, method, alpha, nsteps, every, np);
    if (rc) return rc;
    const int D = g->ndim;
    if (!F || !W || !Fbar) return fail(ctx, JP_ERR_ARG, "null nodal input%s");
    if ((rc = null_ptrs(ctx, D, 1, (const void* const*)Vbar, D, "Vbar"))) return rc;
    if ((rc = null_ptrs(ctx, D, np, (const void* const*)x0bar, D, "x0bar"))) return rc;
    if (np > 0 && (!Tp || !ckpt || !alive || !Tpbar))
        return fail(ctx, JP_ERR_ARG, "null particle array (Tp, ckpt, alive or Tpbar)%s");
    if (D == 2) {
        const auto A = make_args<2>(g, vg, V, alpha, dt, nsteps, every, np);
        if (method == JP_EULER)
            return backward<2, JP_EULER>(ctx, A, vg, ckpt, alive, Tp, F, W, Fbar, Vbar, x0bar,
                                         Tpbar);
        if (method == JP_RK2)
            return backward<2, JP_RK2>(ctx, A, vg, ckpt, alive, Tp, F, W, Fbar, Vbar, x0bar,
                                       Tpbar);
        return backward<2, JP_RK4>(ctx, A, vg, ckpt, alive, Tp, F, W, Fbar, Vbar, x0bar, Tpbar);
    }
    const auto A = make_args<3>(g, vg, V, alpha, dt, nsteps, every, np);
    if (method == JP_EULER)
        return backward<3, JP_EULER>(ctx, A, vg, ckpt, alive, Tp, F, W, Fbar, Vbar, x0bar,
                                     Tpbar);
    if (method == JP_RK2)
        return backward<3, JP_RK2>(ctx, A, vg, ckpt, alive, Tp, F, W, Fbar, Vbar, x0bar, Tpbar);
    return backward<3, JP_RK4>(ctx, A, vg, ckpt, alive, Tp, F, W, Fbar, Vbar, x0bar, Tpbar);
}
