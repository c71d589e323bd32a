// jp_advect.hip -- advection! (src/Particles/Advection/advection.jl:35-91),
// advection_MQS! / advection_LinP! (advection_MQS.jl, advection_LinP.jl) and
// semilagrangian_advection! with the same three velocity interpolations
// (backtracking.jl, backtracking_MQS.jl, backtracking_LinP.jl) on gfx950, FP64
// drop-in, 2D and 3D, Euler / RK2 / RK4.
//
// One workgroup per tile of cells with each velocity component's window of
// nodes, and its axis windows, staged in LDS; the wavefronts walk the cells'
// slots in lockstep chunks of planes (k_advect_tile, all three schemes).  A
// particle with a stage point outside a window is advected on the slot path
// after the others.  The slot path: the velocity gathered from global memory
// (also k_advect_slot, one thread per slot, for MQS and LinP on small grids).
// A bracket lookup costs one guess (uniform spacing estimate; in the windows
// of refined axes a short search from the particle's cell) and one strict test
// against the stored axis, with the reference search for everything else (ties).
#include "jp_ctx.hpp"

#include <type_traits>

using namespace jp;

namespace {

template <int D>
struct VPtrs {
    const double* v[D];
};

struct RKParams {
    double dt;
    double adt;  // (s*alpha)*dt
    int half;    // alpha == 0.5
    double w0;   // muladd(-0.5, inv(alpha), 1)
    double w1;   // 0.5*inv(alpha)
};

// interp_velocity2particle (advection.jl:93-148) for component c: +Inf outside
// the component's grid (check_local_limits, src/Advection/advection.jl:83-91),
// t = (p - x_k)*inv(dx_k) (normalize_coordinates, src/Interpolations/utils.jl:54-58),
// n-linear lerp of the corner values (src/Interpolations/ndlerp.jl:11-15) in
// extract_field_corners order (src/Advection/advection.jl:47-71).

// Row mapping: a wavefront holds 64 consecutive cells of one grid row at one
// slot plane (grid.y), so coordinate and mask accesses coalesce.  Brackets:
// the uniform-spacing guess confirmed with the strict test x[k] < p < x[k+1]
// (a strictly interior point has one bracket, the one the reference's
// bisection returns whatever its seed), else the reference search seeded at
// the particle's cell.
template <int D>
struct AxisGuess {
    double lo[D][D], hi[D][D], i0[D][D];  // x[0], x[n-1], inv_dx[0] of axis (c, d)
};

__device__ inline int64_t bracket_slot(double p, const Axis& A, double x0, double i0,
                                       int64_t seed) {
    const int64_t last = A.n - 2;
    int64_t gk = (int64_t)((p - x0) * i0);
    gk = gk < 0 ? 0 : (gk > last ? last : gk);
    if (A.x[gk] < p && p < A.x[gk + 1]) return gk;
    return find_cell(p, A, seed);
}

// velocity interpolation schemes
constexpr int kLinear = 0;  // interp_velocity2particle
constexpr int kMQS = 1;     // interp_velocity2particle_MQS (advection_MQS.jl:102-124)
constexpr int kLinP = 2;    // interp_velocity2particle_LinP (advection_LinP.jl:104-131)

// column-major view of one velocity component (k = 0 in 2D)
template <typename Int>
struct FView {
    using I = Int;
    const double* __restrict__ F;
    Int n0, n1;
    __device__ double at(Int i, Int j, Int k) const { return F[i + n0 * (j + n1 * k)]; }
};

// half * (t - half)^2 * (muladd(-2, v1, v0) + v2) (src/Interpolations/MQS.jl:13)
__device__ inline double mqs_corr(double t, double v0, double v1, double v2) {
    const double e = t - 0.5;
    return (0.5 * (e * e)) * (fma(-2.0, v1, v0) + v2);
}

// MQS along x of the corners (v00, v10, v01, v11) of one plane: each row's
// lerp along x corrected with the second difference through the node left of
// the cell (ta < 1/2) or right of it, then the lerp along the plane's second
// axis (MQS.jl:2-27, 73-98, 126-152).  Rows 0 and 1 take their extra node
// from (i-1 | i+2, jb0, kb0) and (i-1 | i+2, jb1, kb1).
template <class FV, class I = typename FV::I>
__device__ inline double mqs_x4(const FV& F, double v0, double v1, double v2, double v3,
                                double ta, double tb, I i, I jb0, I kb0, I jb1, I kb1) {
    const double lb = lerp1(ta, v0, v1), lt = lerp1(ta, v2, v3);
    const bool left = ta < 0.5;
    const double cb = left ? mqs_corr(ta, F.at(i - 1, jb0, kb0), v0, v1)
                           : mqs_corr(ta, v0, v1, F.at(i + 2, jb0, kb0));
    const double ct = left ? mqs_corr(ta, F.at(i - 1, jb1, kb1), v2, v3)
                           : mqs_corr(ta, v2, v3, F.at(i + 2, jb1, kb1));
    return lerp1(tb, lb + cb, lt + ct);
}

// MQS along y (MQS.jl:29-55, 100-124): columns (v00, v01), (v10, v11) lerped
// along y with the correction through the node below or above, then along x.
template <class FV, class I = typename FV::I>
__device__ inline double mqs_y4(const FV& F, double v0, double v1, double v2, double v3,
                                double t1, double t2, I i, I j, I k) {
    const double ll = lerp1(t2, v0, v2), lr = lerp1(t2, v1, v3);
    const bool below = t2 < 0.5;
    const double cl = below ? mqs_corr(t2, F.at(i, j - 1, k), v0, v2)
                            : mqs_corr(t2, v0, v2, F.at(i, j + 2, k));
    const double cr = below ? mqs_corr(t2, F.at(i + 1, j - 1, k), v1, v3)
                            : mqs_corr(t2, v1, v3, F.at(i + 1, j + 2, k));
    return lerp1(t1, ll + cl, lr + cr);
}

// MQS of component c at corner (i, j[, k]) with corner values q.  3D: x and y
// combine the plane-k and plane-k+1 results along z, both with extra nodes of
// plane k (MQS.jl:58-64 pass the same i, j, k); z combines two MQS-x
// evaluations of the (x, z) planes of rows j and j+1 along y, both with extra
// nodes of row j (MQS.jl:67-71, 126-152).
template <int D, class FV, class I = typename FV::I>
__device__ inline double mqs(const FV& F, int c, const I (&k0)[D], const double* q,
                             const double (&t)[D]) {
    const I i = k0[0], j = k0[1], o = 0;
    if constexpr (D == 2) {
        return c == 0 ? mqs_x4(F, q[0], q[1], q[2], q[3], t[0], t[1], i, j, o, j + 1, o)
                      : mqs_y4(F, q[0], q[1], q[2], q[3], t[0], t[1], i, j, o);
    } else {
        const I k = k0[2];
        if (c == 0) {
            const double bot = mqs_x4(F, q[0], q[1], q[2], q[3], t[0], t[1], i, j, k, j + 1, k);
            const double top = mqs_x4(F, q[4], q[5], q[6], q[7], t[0], t[1], i, j, k, j + 1, k);
            return lerp1(t[2], bot, top);
        }
        if (c == 1) {
            const double bot = mqs_y4(F, q[0], q[1], q[2], q[3], t[0], t[1], i, j, k);
            const double top = mqs_y4(F, q[4], q[5], q[6], q[7], t[0], t[1], i, j, k);
            return lerp1(t[2], bot, top);
        }
        const double front = mqs_x4(F, q[0], q[1], q[4], q[5], t[0], t[2], i, j, k, j, k + 1);
        const double back = mqs_x4(F, q[2], q[3], q[6], q[7], t[0], t[2], i, j, k, j, k + 1);
        return lerp1(t[1], front, back);
    }
}

// LinP's pressure-point value of component c (advection_LinP.jl:208-391):
// the corner index moves by one along c when p is past the cell's middle
// (offset_LinP); each row of three nodes along c around it (the reference
// clamps their indices to the array: no effect for the interior corners this
// is called for) is averaged pairwise as (a + b)/2 onto the two pressure points;
// the rows run over the other axes (augment_offset: x and y components in
// axis order, the z component with y before x); y and z components swap the
// middle pairs (swap_F); t is measured from the corner moved by +-dx_c/2
// (correct_xci_to_pressure_point).
template <int D, class FV, class I = typename FV::I>
__device__ inline double linp(const FV& F, int c, const I (&k0)[D], const double (&xc)[D],
                              const double (&dxi)[D], const double (&idx)[D],
                              const double (&p)[D]) {
    I b[D];
#pragma unroll
    for (int d = 0; d < D; ++d) b[d] = k0[d] + ((d == c && p[d] > xc[d] + dxi[d] / 2.0) ? 1 : 0);
    constexpr int nrow = D == 2 ? 2 : 4;
    double av[2 * nrow];
#pragma unroll
    for (int r = 0; r < nrow; ++r) {
        double val[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            I id[3] = {0, 0, 0};
            int other = 0;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                int o;
                if (d == c) {
                    o = e - 1;
                } else {
                    const int bit = (D == 3 && c == 2) ? 1 - other : other;
                    o = (r >> bit) & 1;
                    ++other;
                }
                id[d] = b[d] + o;
            }
            val[e] = F.at(id[0], id[1], id[2]);
        }
        av[2 * r] = (val[0] + val[1]) / 2.0;
        av[2 * r + 1] = (val[2] + val[1]) / 2.0;
    }
    double w[2 * nrow];
#pragma unroll
    for (int m = 0; m < 2 * nrow; ++m) {
        // swap_F: (1, 3, 2, 4[, 5, 7, 6, 8]) for the y and z components
        const int src = (c == 0) ? m : ((m & ~3) | ((m & 1) << 1) | ((m >> 1) & 1));
        w[m] = av[src];
    }
    double t[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        double xp = xc[d];
        if (d == c) {
            const double off = 1.0 - 2.0 * (double)(p[d] < xc[d] + dxi[d] / 2.0);
            xp = xc[d] + (off * dxi[d]) / 2.0;
        }
        t[d] = (p[d] - xp) * idx[d];
    }
    const double lo = lerp1(t[1], lerp1(t[0], w[0], w[1]), lerp1(t[0], w[2], w[3]));
    if constexpr (D == 2) {
        return lo;
    } else {
        const double hi = lerp1(t[1], lerp1(t[0], w[4], w[5]), lerp1(t[0], w[6], w[7]));
        return lerp1(t[2], lo, hi);
    }
}

// Component c at p with scheme S.  LIM: advection's limit check (+Inf outside
// the component's grid); without it (semi-Lagrangian) a point outside the
// grid gives NaN, which the caller reports -- the reference's bisection does
// not terminate there.  MQS and LinP apply where the corner index is interior
// along every axis (1 < idx < size - 1, 1-based), else the linear value.
template <int D, int S, bool LIM>
__device__ inline double interp_slot(const AxisGuess<D>& Gs, const Vel<D>& vg,
                                     const VPtrs<D>& V, int c, const double (&p)[D],
                                     const int64_t (&I)[D]) {
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; ++d) in = in && (Gs.lo[c][d] <= p[d] && p[d] <= Gs.hi[c][d]);
    if (!in) return LIM ? __builtin_inf() : __builtin_nan("");
    int64_t k[D];
    double t[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const Axis& A = vg.ax[c][d];
        k[d] = bracket_slot(p[d], A, Gs.lo[c][d], Gs.i0[c][d], I[d]);
        t[d] = (p[d] - A.x[k[d]]) * A.idx[k[d]];
    }
    const double* __restrict__ F = V.v[c];
    const int64_t n0 = vg.ax[c][0].n, n1 = vg.ax[c][1].n;
    int64_t b = k[0] + n0 * k[1];
    if constexpr (D == 3) b += n0 * n1 * k[2];
    double q[1 << D];
#pragma unroll
    for (int r = 0; r < (1 << D); ++r) {
        const int64_t o = (r & 1) + ((r >> 1) & 1) * n0 + (D == 3 ? ((r >> 2) & 1) * n0 * n1 : 0);
        q[r] = F[b + o];
    }
    double vl = lerp1(t[1], lerp1(t[0], q[0], q[1]), lerp1(t[0], q[2], q[3]));
    if constexpr (D == 3) {
        const double hi = lerp1(t[1], lerp1(t[0], q[4], q[5]), lerp1(t[0], q[6], q[7]));
        vl = lerp1(t[2], vl, hi);
    }
    if constexpr (S == kLinear) {
        return vl;
    } else {
        bool interior = true;
#pragma unroll
        for (int d = 0; d < D; ++d)
            interior = interior && k[d] >= 1 && k[d] <= vg.ax[c][d].n - 3;
        if (!interior) return vl;
        const FView<int64_t> Fv{F, n0, n1};
        if constexpr (S == kMQS) {
            return mqs<D>(Fv, c, k, q, t);
        } else {
            double xc[D], dxi[D], idx[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const Axis& A = vg.ax[c][d];
                xc[d] = A.x[k[d]];
                dxi[d] = A.dx[k[d]];
                idx[d] = A.idx[k[d]];
            }
            const double vp = linp<D>(Fv, c, k, xc, dxi, idx, p);
            const double A = 2.0 / 3.0;
            return A * vl + (1.0 - A) * vp;
        }
    }
}

template <int D, int S, bool LIM>
__device__ inline void interp_v_slot(const AxisGuess<D>& Gs, const Vel<D>& vg, const VPtrs<D>& V,
                                     const double (&p)[D], const int64_t (&I)[D],
                                     double (&v)[D]) {
#pragma unroll
    for (int c = 0; c < D; ++c) v[c] = interp_slot<D, S, LIM>(Gs, vg, V, c, p, I);
}

// advect_particle (Euler.jl, RK2.jl, RK4.jl) for any velocity interpolation
// interp(p, v); the semi-Lagrangian backtracking (advect_particle_SML,
// RK2.jl:53-107, RK4.jl:44-87) is the same with P.dt = -dt and
// P.adt = (-alpha) dt
template <int D, int M, class Interp>
__device__ inline void advect_rk(const RKParams& P, const double (&p0)[D], double (&out)[D],
                                 Interp&& interp) {
    double v0[D];
    interp(p0, v0);
    if constexpr (M == JP_EULER) {
#pragma unroll
        for (int d = 0; d < D; ++d) out[d] = fma(P.dt, v0[d], p0[d]);
    } else if constexpr (M == JP_RK2) {
        double p1[D], v1[D];
#pragma unroll
        for (int d = 0; d < D; ++d) p1[d] = fma(P.adt, v0[d], p0[d]);
        interp(p1, v1);  // same seed I (RK2.jl:14,20)
        if (P.half) {
#pragma unroll
            for (int d = 0; d < D; ++d) out[d] = fma(P.dt, v1[d], p0[d]);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) out[d] = fma(P.dt, fma(P.w1, v1[d], P.w0 * v0[d]), p0[d]);
        }
    } else {
        double q[D], k[D], sum[D];
#pragma unroll
        for (int d = 0; d < D; ++d) q[d] = p0[d] + (P.dt * v0[d]) / 2.0;
        interp(q, k);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            sum[d] = v0[d] + 2.0 * k[d];
            q[d] = p0[d] + (P.dt * k[d]) / 2.0;
        }
        interp(q, k);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            sum[d] = sum[d] + 2.0 * k[d];
            q[d] = p0[d] + P.dt * k[d];
        }
        interp(q, k);
#pragma unroll
        for (int d = 0; d < D; ++d) out[d] = p0[d] + (P.dt * (sum[d] + k[d])) / 6.0;
    }
}

// with the slot-kernel interpolation (velocity gathered from global memory)
template <int D, int M, int S = kLinear, bool LIM = true>
__device__ inline void advect_slot(const AxisGuess<D>& Gs, const Vel<D>& vg, const VPtrs<D>& V,
                                   const RKParams& P, const double (&p0)[D],
                                   const int64_t (&I)[D], double (&out)[D]) {
    advect_rk<D, M>(P, p0, out, [&](const double (&p)[D], double (&v)[D]) {
        interp_v_slot<D, S, LIM>(Gs, vg, V, p, I, v);
    });
}

template <int D>
__device__ inline void axis_guess(const Vel<D>& vg, AxisGuess<D>& Gs) {
#pragma unroll
    for (int cc = 0; cc < D; ++cc)
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const Axis& A = vg.ax[cc][d];
            Gs.lo[cc][d] = A.x[0];
            Gs.hi[cc][d] = A.x[A.n - 1];
            Gs.i0[cc][d] = A.idx[0];
        }
}

template <int D, int M, int S>
__global__ void __launch_bounds__(kBlock) k_advect_slot(Grid<D> g, Vel<D> vg, VPtrs<D> V,
                                                        Ptr3 coords,
                                                        const uint8_t* __restrict__ index,
                                                        RKParams P) {
    int64_t c, I[D];
    if (!row_cell<D>(g, c, I)) return;
    const int64_t e = c + g.C * (int64_t)blockIdx.y;
    if (!index[e]) return;  // doskip (src/Utils.jl:32-33)
    AxisGuess<D> Gs;
    axis_guess<D>(vg, Gs);
    double p0[D], out[D];
#pragma unroll
    for (int d = 0; d < D; ++d) p0[d] = coords.p[d][e];
    advect_slot<D, M, S>(Gs, vg, V, P, p0, I, out);
#pragma unroll
    for (int d = 0; d < D; ++d) coords.p[d][e] = out[d];
}

// The velocity staged in LDS: one workgroup per tile of cells (2D 64x4, 3D
// 16x4x4), one thread per cell walking the cell's slot planes in lockstep
// chunks (a wavefront covers whole 128-byte runs of a plane).  Each
// component's window holds the nodes from two below the tile's first bracket
// to kWinPad - 2 beyond its end, which covers the RK stage points of a step of
// up to one cell and the extra nodes of MQS and LinP around them; its axis
// coordinates and inverse spacings are staged too.  A bracket, and the nodal
// values, come from the window when they lie in it and from global memory
// otherwise, with the same tests and the same values as the slot kernel, so
// the results are identical.  Bound by latency, of LDS reads and dependent FP64
// operations: the VALUs are busy 43% of the time at 512^2 (RK2, 98 us, 2.9
// wavefronts per SIMD) and 41% at 61 x 47 x 74 (RK4, 594 us, 1.7: 173 registers
// and 60 KB of LDS).  MQS RK2 85 us at 300 x 431 (the slot kernel, which gathers
// its stencils from global memory: 191).
template <int D>
struct F64Tile;
template <>
struct F64Tile<2> {
    static constexpr int n[3] = {64, 4, 1};
};
template <>
struct F64Tile<3> {
    static constexpr int n[3] = {16, 4, 4};
};
constexpr int kWinPad = 6;

template <int D>
struct F64Win {
    static constexpr int w(int d) { return d < D ? F64Tile<D>::n[d] + kWinPad : 1; }
    static constexpr int size() { return w(0) * w(1) * w(2); }
    static constexpr int axis() { return w(0) > w(1) ? (w(0) > w(2) ? w(0) : w(2)) : (w(1) > w(2) ? w(1) : w(2)); }
};

// window entries past the end of an axis hold NaN (no bracket test passes)
template <int D, int S>
struct TileLds {
    double v[D][F64Win<D>::size()];
    double x[D][D][F64Win<D>::axis()];
    double idx[D][D][F64Win<D>::axis()];
    double dx[S == kLinP ? D : 1][D][S == kLinP ? F64Win<D>::axis() : 1];
};
// where the windows sit: first node of component c along d, and the window
// position of the bracket that the tile's first cell guesses
template <int D>
struct TileWin {
    int64_t lo[D][D];
    int seed[D][D];
};

// The bracket k of p in a window of W axis nodes x (inverse spacings idx) and
// its node xl; false if it does not hold p strictly: the uniform-spacing
// guess, or (REF: a refined axis) up to two steps from `seed`, the particle's
// cell's own position.
template <bool REF>
__device__ inline bool window_bracket(double p, const double* x, const double* idx, int W,
                                      int seed, int& k, double& xl) {
    if constexpr (!REF) {
        const double g = (p - x[0]) * idx[0];
        k = g >= 0.0 ? (g < (double)(W - 2) ? (int)g : W - 2) : 0;
    } else {
        k = seed < W - 2 ? seed : W - 2;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            k += (p > x[k + 1] ? 1 : 0) - (p < x[k] ? 1 : 0);
            k = k < 0 ? 0 : (k > W - 2 ? W - 2 : k);
        }
    }
    xl = x[k];
    const double xr = x[k + 1];
    return xl < p && p < xr;
}

// Component c at p from the window, if every axis brackets p strictly inside
// it (that bracket is the axis's only one, the one the slot kernel finds, and
// it lies inside the component's grid) and the window holds the scheme's
// nodes around it; false otherwise.  cell: the particle's cell in the tile.
template <int D, int S, bool REF>
__device__ inline bool interp_tile_f64(const TileLds<D, S>& L, const TileWin<D>& wn,
                                       const Vel<D>& vg, int c, const int (&cell)[D],
                                       const double (&p)[D], double& v) {
    using WN = F64Win<D>;
    int w[D];
    double t[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        int k;
        double xl;
        if (!window_bracket<REF>(p[d], L.x[c][d], L.idx[c][d], WN::w(d),
                                 REF ? wn.seed[c][d] + cell[d] : 0, k, xl))
            return false;
        w[d] = k;
        t[d] = (p[d] - xl) * L.idx[c][d][k];
    }
    const int b = w[0] + WN::w(0) * (w[1] + (D == 3 ? WN::w(1) * w[D - 1] : 0));
    double q[1 << D];
#pragma unroll
    for (int r = 0; r < (1 << D); ++r) {
        const int o = (r & 1) + ((r >> 1) & 1) * WN::w(0) +
                      (D == 3 ? ((r >> 2) & 1) * WN::w(0) * WN::w(1) : 0);
        q[r] = L.v[c][b + o];
    }
    double vl = lerp1(t[1], lerp1(t[0], q[0], q[1]), lerp1(t[0], q[2], q[3]));
    if constexpr (D == 3) {
        const double hi = lerp1(t[1], lerp1(t[0], q[4], q[5]), lerp1(t[0], q[6], q[7]));
        vl = lerp1(t[2], vl, hi);
    }
    if constexpr (S != kLinear) {
        bool interior = true, held = true;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int64_t k = wn.lo[c][d] + w[d];
            interior = interior && k >= 1 && k <= vg.ax[c][d].n - 3;
            held = held && w[d] >= 1 && w[d] <= WN::w(d) - 3;
        }
        if (interior) {
            if (!held) return false;
            const FView<int> Fv{L.v[c], WN::w(0), WN::w(1)};
            if constexpr (S == kMQS) {
                vl = mqs<D>(Fv, c, w, q, t);
            } else {
                double xc[D], dxi[D], idx[D];
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    xc[d] = L.x[c][d][w[d]];
                    dxi[d] = L.dx[c][d][w[d]];
                    idx[d] = L.idx[c][d][w[d]];
                }
                const double vp = linp<D>(Fv, c, w, xc, dxi, idx, p);
                const double A = 2.0 / 3.0;
                vl = A * vl + (1.0 - A) * vp;
            }
        }
    }
    v = vl;
    return true;
}

// B: slot planes per chunk.  A particle whose step leaves the windows (or
// sits on a node) is marked in its cell's word and advected as k_advect_slot
// does after the wavefront's other particles, dealt to the lanes in the same
// way: inside the chunk loop that path costs the loop's occupancy (2D RK2 169
// registers, two wavefronts per SIMD instead of four: 165 us against 98 at
// 512^2), and a flag per slot with a pass of its own costs a launch.  When most
// of a chunk's first 64 particles miss, the steps are longer than the windows'
// margin and the wavefront's other slots are marked untried.  Steps of 6 cells at
// 256^2: MQS RK4 149 us, linear RK4 on refined axes 313 (each cell's particles one
// after the other by its own lane, the windows tried for all: 261 and 641).
template <int D, int M, int S, int B>
__global__ void __launch_bounds__(kBlock, D == 2 ? 4 : 2) k_advect_tile(Grid<D> g, Vel<D> vg, VPtrs<D> V,
                                                        Ptr3 coords,
                                                        const uint8_t* __restrict__ index,
                                                        RKParams P, int span) {
    using TL = F64Tile<D>;
    using WN = F64Win<D>;
    __shared__ TileLds<D, S> L;
    __shared__ unsigned long long s_miss[kBlock];  // per cell: slots to do on the slot path
    int64_t t0[D];
    {
        int64_t b = blockIdx.x;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int64_t nt = (g.ni[d] + TL::n[d] - 1) / TL::n[d];
            t0[d] = (b % nt) * TL::n[d];
            b /= nt;
        }
    }
    const int kb = blockIdx.y * span;
    const int ke = kb + span < g.K ? kb + span : g.K;
    const int tid = threadIdx.x;
    // window origins: two nodes below the bracket of the tile's first vertex
    // (only where the window sits depends on it, not a result).  On the
    // staggered grids that is the cell's own number, refined or not; other
    // axes search.
    TileWin<D> wn;
    {
        // (all loads before the first test: one round trip, not one per axis)
        double xt[D], xa[D][D], xb[D][D];
        bool ok = true;
#pragma unroll
        for (int d = 0; d < D; ++d) xt[d] = g.xv[d].x[t0[d]];
#pragma unroll
        for (int c = 0; c < D; ++c)
#pragma unroll
            for (int d = 0; d < D; ++d) {  // (an axis has more nodes than the grid cells)
                xa[c][d] = vg.ax[c][d].x[t0[d]];
                xb[c][d] = vg.ax[c][d].x[t0[d] + 1];
            }
#pragma unroll
        for (int c = 0; c < D; ++c)
#pragma unroll
            for (int d = 0; d < D; ++d) {
                ok = ok && xa[c][d] <= xt[d] && xt[d] <= xb[c][d];
                wn.lo[c][d] = t0[d];
            }
        if (!ok) {
#pragma unroll 1
            for (int c = 0; c < D; ++c)
#pragma unroll 1
                for (int d = 0; d < D; ++d) {
                    const Axis A = vg.ax[c][d];
                    const double x0 = A.x[0], xn = A.x[A.n - 1], x = g.xv[d].x[t0[d]];
                    const int64_t k = find_cell(x < x0 ? x0 : (x > xn ? xn : x), A, t0[d]);
#pragma unroll
                    for (int q = 0; q < D * D; ++q)
                        if (q == c * D + d) wn.lo[q / D][q % D] = k;
                }
        }
#pragma unroll
        for (int c = 0; c < D; ++c)
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int64_t k = wn.lo[c][d];
                wn.lo[c][d] = k - 2 < 0 ? 0 : k - 2;
                wn.seed[c][d] = (int)(k - wn.lo[c][d]);
            }
    }
    const double qnan = __builtin_nan("");
    bool off = false;  // an axis of the windows is not uniform
#pragma unroll
    for (int c = 0; c < D; ++c) {
        const double* __restrict__ F = V.v[c];
        for (int i = tid; i < WN::size(); i += kBlock) {
            int r = i;
            int64_t node = 0, stride = 1;
            bool ok = true;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int64_t kk = wn.lo[c][d] + r % WN::w(d);
                r /= WN::w(d);
                ok = ok && kk < vg.ax[c][d].n;
                node += kk * stride;
                stride *= vg.ax[c][d].n;
            }
            L.v[c][i] = ok ? F[node] : qnan;
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            for (int w = tid; w < WN::w(d); w += kBlock) {
                const Axis& A = vg.ax[c][d];
                const int64_t kk = wn.lo[c][d] + w;
                const double x = kk < A.n ? A.x[kk] : qnan;
                L.x[c][d][w] = x;
                L.idx[c][d][w] = kk < A.n - 1 ? A.idx[kk] : qnan;
                // (false for NaN)
                off = off || fabs((x - A.x[wn.lo[c][d]]) * A.idx[wn.lo[c][d]] - (double)w) > 1e-4;
                if constexpr (S == kLinP) L.dx[c][d][w] = kk < A.n - 1 ? A.dx[kk] : qnan;
            }
    }
    // one refined axis in the windows: brackets start from the particle's cell
    // (the uniform-spacing guess of a window of ~70 refined nodes misses, and
    // every miss is a step on the slot path: 284 us at 389 x 211 with RK4, 85
    // with the search; for uniform axes the guess is the shorter way, and a
    // spacing off by 1e-4 misses too rarely to matter)
    s_miss[tid] = 0;
    const bool refined = __builtin_amdgcn_readfirstlane(__syncthreads_or(off ? 1 : 0)) != 0;
    // the cell of thread t of the tile and whether it is in the grid
    auto cell_of = [&](int t, int64_t (&J)[D]) {
        bool in = true;
        int r = t;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            J[d] = t0[d] + r % TL::n[d];
            r /= TL::n[d];
            in = in && J[d] < g.ni[d];
        }
        return in;
    };
    int64_t I[D];
    const bool inside = cell_of(tid, I);
    const int64_t c = inside ? lin<D>(g.ni, I) : 0;
    const int64_t C = g.C;
    // the step from the windows
    bool win = true;
    int cell[D];  // of the particle, in the tile

    // a thread outside the grid owns no particle but still takes work
    const uint64_t act = !inside ? 0ull
                                 : ((kb == 0 && ke == g.K) ? active_slots(index, c, C, g.K)
                                                           : active_slots_in(index, c, C, kb, ke));
    // Chunks of B slot planes.  The wavefront's active particles of a chunk
    // are listed (plane-major, then lane) and dealt to its lanes in turn, so
    // that every lane advects about the same number of particles; consecutive
    // entries are neighbouring cells of one plane, so the loads and stores
    // stay coalesced.  The list is written and read by the same wavefront
    // (its LDS operations complete in order).
    __shared__ uint16_t s_items[kBlock / 64][B * 64];
    uint16_t* items = s_items[tid >> 6];
    const int lane = tid & 63, wbase = tid & ~63;
    // the entries (slot in the chunk << 6 | lane) of the set bits of slots k0 ..
    auto list = [&](uint64_t bits, int k0) {
        int n = 0;
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const bool a = k0 + j < 64 && ((bits >> (k0 + j)) & 1);
            const uint64_t bal = __ballot(a);
            const int below = (int)__builtin_amdgcn_mbcnt_hi(
                (uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
            if (a) items[n + below] = (uint16_t)((j << 6) | lane);
            n += __popcll(bal);
        }
        return n;
    };
    auto chunks = [&](auto ref) {
        auto interp = [&](const double (&p)[D], double (&v)[D]) {
#pragma unroll
            for (int cc = 0; cc < D; ++cc)
                win = interp_tile_f64<D, S, decltype(ref)::value>(L, wn, vg, cc, cell, p, v[cc]) &&
                      win;
        };
        for (int k0 = kb; k0 < ke; k0 += B) {
            const int n = list(act, k0);
            if (!n) continue;
            // this lane's entries lane, lane + 64, ...: positions loaded first
            double pq[B][D];
            int dq[B];
#pragma unroll
            for (int q = 0; q < B; ++q) {
                const int item = lane + 64 * q;
                dq[q] = item < n ? items[item] : -1;
                int64_t J[D];
                cell_of(wbase + (dq[q] & 63), J);
                const int64_t e = lin<D>(g.ni, J) + C * (k0 + (dq[q] >> 6));
#pragma unroll
                for (int d = 0; d < D; ++d) pq[q][d] = dq[q] >= 0 ? coords.p[d][e] : 0.0;
            }
            bool missed = false;  // the lane's first entry
#pragma unroll
            for (int q = 0; q < B; ++q) {
                if (dq[q] < 0) break;
                int64_t J[D];
                cell_of(wbase + (dq[q] & 63), J);
                const int64_t e = lin<D>(g.ni, J) + C * (k0 + (dq[q] >> 6));
                double out[D];
                win = true;
#pragma unroll
                for (int d = 0; d < D; ++d) cell[d] = (int)(J[d] - t0[d]);
                advect_rk<D, M>(P, pq[q], out, interp);
                if (!win) {
                    if (q == 0) missed = true;
                    atomicOr(&s_miss[wbase + (dq[q] & 63)], 1ull << (k0 + (dq[q] >> 6)));
                    continue;
                }
#pragma unroll
                for (int d = 0; d < D; ++d) coords.p[d][e] = out[d];
            }
            // most first entries missed: the other slots would too
            if (2 * __popcll(__ballot(missed)) > (n < 64 ? n : 64)) {
                if (k0 + B < 64) s_miss[tid] |= act & ~((1ull << (k0 + B)) - 1);
                break;
            }
        }
    };
    if (refined) chunks(std::true_type{});
    else chunks(std::false_type{});
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (the words are the wavefront's own)
    const uint64_t miss = s_miss[tid];
    if (!__any(miss != 0)) return;
    AxisGuess<D> Gs;
    axis_guess<D>(vg, Gs);
    for (int k0 = kb; k0 < ke; k0 += B) {
        const int n = list(miss, k0);
        for (int i = lane; i < n; i += 64) {
            const int item = items[i];
            int64_t J[D];
            cell_of(wbase + (item & 63), J);
            const int64_t e = lin<D>(g.ni, J) + C * (k0 + (item >> 6));
            double p0[D], out[D];
#pragma unroll
            for (int d = 0; d < D; ++d) p0[d] = coords.p[d][e];
            advect_slot<D, M, S>(Gs, vg, V, P, p0, J, out);
#pragma unroll
            for (int d = 0; d < D; ++d) coords.p[d][e] = out[d];
        }
    }
}

// semilagrangian_advection! (backtracking.jl:15-101 and the MQS / LinP forms):
// one thread per interior node I of the nodal grid (x fastest).  The node is
// traced back (velocity brackets seeded at I), the point bracketed on the
// vertex axes seeded at I, and every field F[f][I] = lerp of F0[f]'s corners
// there, t = (p - x[Ib]) * inv(dx[Ib]) -- dx[I] with `at_node` (the linear
// NTuple method, backtracking.jl:79).  A point that left a velocity or vertex
// axis sets range[0] and range[1] and leaves the node unchanged.
template <int D>
struct NodeGrid {
    int64_t n[D];
    int64_t N;  // interior nodes
    Axis x[D];
};
struct SmlFields {
    double* F[JP_MAX_ARGS];
    const double* F0[JP_MAX_ARGS];
    int n;
};

template <int D, int M, int S>
__global__ void __launch_bounds__(kBlock) k_sml(NodeGrid<D> G, Vel<D> vg, VPtrs<D> V,
                                                SmlFields Fs, RKParams P, int at_node,
                                                int* __restrict__ range) {
    const int64_t tid = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (tid >= G.N) return;
    int64_t I[D], r = tid;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const int64_t m = G.n[d] - 2;
        I[d] = r % m + 1;
        r /= m;
    }
    AxisGuess<D> Gs;
    axis_guess<D>(vg, Gs);
    double p[D], pb[D];
#pragma unroll
    for (int d = 0; d < D; ++d) p[d] = G.x[d].x[I[d]];
    advect_slot<D, M, S, false>(Gs, vg, V, P, p, I, pb);
    int64_t Ib[D];
    double t[D];
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; ++d) in = in && (G.x[d].x[0] <= pb[d] && pb[d] <= G.x[d].x[G.n[d] - 1]);
    if (!in) {
        range[0] = 1;
        range[1] = 1;
        return;
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const Axis& A = G.x[d];
        Ib[d] = bracket_slot(pb[d], A, A.x[0], A.idx[0], I[d]);
        t[d] = (pb[d] - A.x[Ib[d]]) * A.idx[at_node ? I[d] : Ib[d]];
    }
    const int64_t n0 = G.n[0], n1 = G.n[1];
    int64_t b = Ib[0] + n0 * Ib[1], node = I[0] + n0 * I[1];
    if constexpr (D == 3) {
        b += n0 * n1 * Ib[2];
        node += n0 * n1 * I[2];
    }
    for (int f = 0; f < Fs.n; ++f) {
        const double* __restrict__ F0 = Fs.F0[f];
        double q[1 << D];
#pragma unroll
        for (int m = 0; m < (1 << D); ++m) {
            const int64_t o =
                (m & 1) + ((m >> 1) & 1) * n0 + (D == 3 ? ((m >> 2) & 1) * n0 * n1 : 0);
            q[m] = F0[b + o];
        }
        double v = lerp1(t[1], lerp1(t[0], q[0], q[1]), lerp1(t[0], q[2], q[3]));
        if constexpr (D == 3) {
            const double hi = lerp1(t[1], lerp1(t[0], q[4], q[5]), lerp1(t[0], q[6], q[7]));
            v = lerp1(t[2], v, hi);
        }
        Fs.F[f][node] = v;
    }
}

template <int D>
Vel<D> to_vel(const jp_velgrid* vg) {
    Vel<D> V;
    for (int c = 0; c < D; ++c)
        for (int d = 0; d < D; ++d) {
            const jp_axis& a = vg->ax[c][d];
            V.ax[c][d] = Axis{a.x, a.dx, a.inv_dx, a.n};
        }
    return V;
}

template <int D, int M, int S>
int launch(jp_ctx* ctx, const Grid<D>& G, const Vel<D>& vg, const VPtrs<D>& V, Ptr3 cp,
           const uint8_t* index, const RKParams& P) {
    // MQS and LinP: a thread per slot where the slots are few (a wavefront per row of 64
    // cells and slot plane, up to 40 per CU, more than it holds at once); a tile's chain
    // of windows and chunks is then longer than the gathers from global memory.  Tiles
    // and slots, MQS RK2 in us: 64^2 cells of 48 slots (3072 wavefronts) 22 and 7, 96^2
    // (9216) 26 and 22, 128^2 (12288) 30 and 29, 160^2 (23040) 35 and 52; 3D 20^3 of 24
    // (9600) 53 and 40, 12^3 of 54 (7776) 44 and 49, 20^3 of 54 (21600) 60 and 104.
    const bool few = S != kLinear && row_count<D>(G) * G.K <= (int64_t)40 * ctx->num_cu;
    if (!ctx->opt_advect_slots && !few) {
        int64_t tiles = 1;
        for (int d = 0; d < D; ++d)
            tiles *= (G.ni[d] + F64Tile<D>::n[d] - 1) / F64Tile<D>::n[d];
        // slot groups when the tiles alone leave the chip under-filled
        const int span = slot_span(ctx, tiles, G.K, 2048);
        const dim3 grid((unsigned)tiles, (unsigned)((G.K + span - 1) / span));
        k_advect_tile<D, M, S, D == 2 ? 8 : 4><<<grid, kBlock, 0, ctx->stream>>>(G, vg, V, cp,
                                                                                index, P, span);
        JP_LAUNCHED(ctx);
        return JP_OK;
    }
    dim3 grid((unsigned)row_blocks<D>(G), (unsigned)G.K);
    k_advect_slot<D, M, S><<<grid, kBlock, 0, ctx->stream>>>(G, vg, V, cp, index, P);
    JP_LAUNCHED(ctx);
    return JP_OK;
}

template <int D, int S>
int launch_method(jp_ctx* ctx, const Grid<D>& G, const Vel<D>& vg, const VPtrs<D>& V, Ptr3 cp,
                  const uint8_t* index, int method, const RKParams& P) {
    if (method == JP_EULER) return launch<D, JP_EULER, S>(ctx, G, vg, V, cp, index, P);
    if (method == JP_RK2) return launch<D, JP_RK2, S>(ctx, G, vg, V, cp, index, P);
    return launch<D, JP_RK4, S>(ctx, G, vg, V, cp, index, P);
}

template <int D>
int run(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords, const uint8_t* index,
        const double* const* Vp, const jp_velgrid* vgp, int method, int scheme,
        const RKParams& P) {
    Grid<D> G = to_grid<D>(g);
    Vel<D> vg = to_vel<D>(vgp);
    VPtrs<D> V;
    for (int c = 0; c < D; ++c) V.v[c] = Vp[c];
    Ptr3 cp{{nullptr, nullptr, nullptr}};
    for (int d = 0; d < D; ++d) cp.p[d] = coords[d];
    int rc;
    if (scheme == kMQS)
        rc = launch_method<D, kMQS>(ctx, G, vg, V, cp, index, method, P);
    else if (scheme == kLinP)
        rc = launch_method<D, kLinP>(ctx, G, vg, V, cp, index, method, P);
    else
        rc = launch_method<D, kLinear>(ctx, G, vg, V, cp, index, method, P);
    if (rc) return rc;
    return finish(ctx);
}

template <int D, int M>
int launch_sml(jp_ctx* ctx, const NodeGrid<D>& G, const Vel<D>& vg, const VPtrs<D>& V,
               const SmlFields& Fs, const RKParams& P, int scheme, int at_node) {
    const unsigned blocks = (unsigned)blocks_for(G.N);
    int* range = drange(ctx);
    if (scheme == kMQS)
        k_sml<D, M, kMQS><<<blocks, kBlock, 0, ctx->stream>>>(G, vg, V, Fs, P, at_node, range);
    else if (scheme == kLinP)
        k_sml<D, M, kLinP><<<blocks, kBlock, 0, ctx->stream>>>(G, vg, V, Fs, P, at_node, range);
    else
        k_sml<D, M, kLinear><<<blocks, kBlock, 0, ctx->stream>>>(G, vg, V, Fs, P, at_node, range);
    JP_LAUNCHED(ctx);
    return JP_OK;
}

template <int D>
int run_sml(jp_ctx* ctx, const jp_axis* grid, const jp_velgrid* vgp, const double* const* Vp,
            const SmlFields& Fs, int method, int scheme, int at_node, const RKParams& P) {
    NodeGrid<D> G;
    G.N = 1;
    for (int d = 0; d < D; ++d) {
        G.n[d] = grid[d].n;
        G.N *= grid[d].n - 2;
        G.x[d] = Axis{grid[d].x, grid[d].dx, grid[d].inv_dx, grid[d].n};
    }
    Vel<D> vg = to_vel<D>(vgp);
    VPtrs<D> V;
    for (int c = 0; c < D; ++c) V.v[c] = Vp[c];
    // this call's flag starts clear (a kernel, so the call can be captured)
    int rc = zero_bytes(ctx, drange(ctx), sizeof(int));
    if (rc) return rc;
    rc = method == JP_RK2 ? launch_sml<D, JP_RK2>(ctx, G, vg, V, Fs, P, scheme, at_node)
                          : launch_sml<D, JP_RK4>(ctx, G, vg, V, Fs, P, scheme, at_node);
    if (rc) return rc;
    if (!ctx->sync || ctx->capturing) return JP_OK;
    int bad = 0;
    JP_HIP(ctx, hipMemcpyAsync(&bad, drange(ctx), sizeof bad, hipMemcpyDeviceToHost, ctx->stream));
    JP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return bad ? range_report(ctx) : JP_OK;
}

int check_velgrid(jp_ctx* ctx, const jp_cellgrid* g, const jp_velgrid* vg,
                  const double* const* V) {
    if (!vg) return fail(ctx, JP_ERR_ARG, "null velocity grid%s");
    if (!V) return fail(ctx, JP_ERR_ARG, "null velocity array%s");
    for (int c = 0; c < g->ndim; ++c) {
        if (!V[c]) return fail(ctx, JP_ERR_ARG, "null velocity component%s %lld", "", c);
        for (int d = 0; d < g->ndim; ++d) {
            const jp_axis& a = vg->ax[c][d];
            if (!a.x || !a.dx || !a.inv_dx)
                return fail(ctx, JP_ERR_ARG, "null velocity axis pointer%s (component %lld)", "", c);
            // the bisection is seeded with the particle's cell index, which
            // must address a bracket [x[s], x[s+1]] of the velocity axis
            if (a.n < g->ni[d] + 1)
                return fail(ctx, JP_ERR_ARG,
                            "velocity axis shorter than the cell grid%s (component %lld)", "", c);
        }
    }
    return JP_OK;
}

RKParams rk_params(double alpha, double dt, double sign) {
    RKParams P;
    P.dt = sign * dt;
    P.adt = (sign * alpha) * dt;
    P.half = alpha == 0.5;
    const double ia = 1.0 / alpha;
    P.w0 = std::fma(-0.5, ia, 1.0);
    P.w1 = 0.5 * ia;
    return P;
}

int advect_entry(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords, const uint8_t* index,
                 const double* const* V, const jp_velgrid* vg, int method, double alpha,
                 double dt, int scheme) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if (!coords) return fail(ctx, JP_ERR_ARG, "null coords%s");
    for (int d = 0; d < g->ndim; ++d)
        if (!coords[d]) return fail(ctx, JP_ERR_ARG, "null coords pointer%s %lld", "", d);
    if (!index) return fail(ctx, JP_ERR_ARG, "null index%s");
    if ((rc = check_velgrid(ctx, g, vg, V))) return rc;
    if (method < JP_EULER || method > JP_RK4)
        return fail(ctx, JP_ERR_ARG, "unknown integrator%s %lld", "", method);
    if (method == JP_RK2 && !(0.0 < alpha && alpha < 1.0))
        return fail(ctx, JP_ERR_ARG, "Only 0 < α < 1 is supported%s");
    if (scheme < kLinear || scheme > kLinP)
        return fail(ctx, JP_ERR_ARG, "unknown velocity interpolation scheme%s %lld", "", scheme);
    const RKParams P = rk_params(alpha, dt, 1.0);
    return g->ndim == 2 ? run<2>(ctx, g, coords, index, V, vg, method, scheme, P)
                        : run<3>(ctx, g, coords, index, V, vg, method, scheme, P);
}

}  // namespace

namespace jp {
int range_report(jp_ctx* ctx) {
    // reported now: clear the call and sticky words
    int rc = zero_bytes(ctx, drange(ctx), 2 * sizeof(int));
    if (rc) return rc;
    JP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return fail(ctx, JP_ERR_ARG,
                "semilagrangian_advection: a backtracked point left the velocity or vertex "
                "grid%s (its node was left unchanged; reduce dt)");
}

int range_sticky(jp_ctx* ctx) {
    int st = 0;
    JP_HIP(ctx, hipMemcpyAsync(&st, drange(ctx) + 1, sizeof st, hipMemcpyDeviceToHost,
                               ctx->stream));
    JP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return st ? range_report(ctx) : JP_OK;
}
}  // namespace jp

extern "C" int jp_advection(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords,
                            const uint8_t* index, const double* const* V, const jp_velgrid* vg,
                            int method, double alpha, double dt) {
    return advect_entry(ctx, g, coords, index, V, vg, method, alpha, dt, kLinear);
}

extern "C" int jp_advection_scheme(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords,
                                   const uint8_t* index, const double* const* V,
                                   const jp_velgrid* vg, int method, double alpha, double dt,
                                   int scheme) {
    return advect_entry(ctx, g, coords, index, V, vg, method, alpha, dt, scheme);
}

extern "C" int jp_semilagrangian(jp_ctx* ctx, int ndim, const jp_axis* grid,
                                 const jp_velgrid* vg, const double* const* V, int nfields,
                                 double* const* F, const double* const* F0, int method,
                                 double alpha, double dt, int scheme, int di_at_node) {
    if (!ctx) return JP_ERR_STATE;
    if (ndim != 2 && ndim != 3) return fail(ctx, JP_ERR_ARG, "ndim must be 2 or 3%s");
    if (!grid) return fail(ctx, JP_ERR_ARG, "null grid%s");
    for (int d = 0; d < ndim; ++d) {
        if (!grid[d].x || !grid[d].dx || !grid[d].inv_dx)
            return fail(ctx, JP_ERR_ARG, "null grid axis pointer%s %lld", "", d);
        if (grid[d].n < 3) return fail(ctx, JP_ERR_ARG, "grid axis%s %lld has fewer than 3 nodes", "", d);
    }
    if (!vg) return fail(ctx, JP_ERR_ARG, "null velocity grid%s");
    if (!V) return fail(ctx, JP_ERR_ARG, "null velocity array%s");
    for (int c = 0; c < ndim; ++c) {
        if (!V[c]) return fail(ctx, JP_ERR_ARG, "null velocity component%s %lld", "", c);
        for (int d = 0; d < ndim; ++d) {
            const jp_axis& a = vg->ax[c][d];
            if (!a.x || !a.dx || !a.inv_dx)
                return fail(ctx, JP_ERR_ARG, "null velocity axis pointer%s (component %lld)", "", c);
            // the velocity brackets are seeded with the node index
            if (a.n < grid[d].n)
                return fail(ctx, JP_ERR_ARG,
                            "velocity axis shorter than the nodal grid%s (component %lld)", "", c);
        }
    }
    if (method != JP_RK2 && method != JP_RK4)
        return fail(ctx, JP_ERR_ARG, "semilagrangian_advection takes RungeKutta2 or RungeKutta4%s");
    if (method == JP_RK2 && !(0.0 < alpha && alpha < 1.0))
        return fail(ctx, JP_ERR_ARG, "Only 0 < α < 1 is supported%s");
    if (scheme < kLinear || scheme > kLinP)
        return fail(ctx, JP_ERR_ARG, "unknown velocity interpolation scheme%s %lld", "", scheme);
    if (nfields < 1 || nfields > JP_MAX_ARGS || !F || !F0)
        return fail(ctx, JP_ERR_ARG, "nfields must be 1..JP_MAX_ARGS%s");
    SmlFields Fs;
    Fs.n = nfields;
    for (int f = 0; f < nfields; ++f) {
        if (!F[f] || !F0[f]) return fail(ctx, JP_ERR_ARG, "null field%s %lld", "", f);
        for (int h = 0; h < nfields; ++h)
            if ((const double*)F[f] == F0[h])
                return fail(ctx, JP_ERR_ARG,
                            "F and F0 must be different arrays%s (F[%lld] is an F0)", "", f);
        Fs.F[f] = F[f];
        Fs.F0[f] = F0[f];
    }
    const RKParams P = rk_params(alpha, dt, -1.0);
    return ndim == 2 ? run_sml<2>(ctx, grid, vg, V, Fs, method, scheme, di_at_node != 0, P)
                     : run_sml<3>(ctx, grid, vg, V, Fs, method, scheme, di_at_node != 0, P);
}
