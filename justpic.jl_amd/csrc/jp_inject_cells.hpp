// jp_inject_cells.hpp -- injection in 3D, with several fields, and with phases
// (inject_particles!, inject_particles_phase!: src/Particles/injection.jl:
// 68-131, 233-325; index_min_distance :330-393), FP64 and FP32-split
// positions.  One launch per colour.
//
// One wavefront per listed cell, lanes = slots (K <= 64), planned like the 2D
// kernel (jp_inject2.hpp): which slots are filled, in which quadrant, follows
// from the quadrant counts; every new position depends on (cell, slot) only;
// the candidates of injection j are the particles present before the call and
// the injections before j.  So the cell is planned with ballots and the new
// positions are drawn in their own lanes.  Every search first looks at the
// cell's own particles, in registers; a neighbour cell is read only if some
// search's bound reaches it (in the slot-plane layout every particle read is a
// cache line, and reading all 26 neighbours bound the launch by those
// requests): the distance to the neighbour's box, which holds all of its
// particles unless the scan found one outside, or an earlier colour put one there
// (a cell's spacing may exceed the distance of its vertices: a range axis has its
// first spacing for every cell).  The neighbours that are needed
// are read once for all searches, four at a time, each search's per-lane
// minimum kept in LDS.  The wavefront minima, the copies of the sources'
// values (an earlier injection's copy when the source is one) and the stores
// follow.  With one search after another, each reading the neighbourhood again
// with a square root per candidate, the eight launches took 1471 us at 61 x 47
// x 74 (K = 54, two fields), now 194 (780 reading all neighbours once); four
// launches with three fields at 389 x 211 76 us, now 42; with phases at 384
// x 257 118 us, now 54.
//
// Distances are compared squared: the square root is monotonic, so the first
// element (neighbour cell, then slot) of minimal rounded distance is found
// from the squares and, where two squares are so close that their roots may
// round to the same value, from the roots themselves.
#pragma once

#include "jp_ctx.hpp"
#include "jp_inject2.hpp"

namespace jp {

struct PhaseInj {
    double* phases;
    const double* fields[JP_MAX_ARGS];
    uint32_t centred;  // bit a: fields[a] is cell-centred (dims ni), else nodal (ni + 1)
    Axis xc[3];        // centre axes (particles.xci with di.center)
};

template <int D>
struct InjectCells {
    Grid<D> g;
    double* x[3];  // FP64 form: coordinates
    float* u[3];   // split form: offsets in cell units
    uint8_t* index;
    uint64_t* occw;       // occupancy word of every cell (updated here)
    uint32_t* out;        // per cell: a particle lies outside the cell's box (the scan, updated here)
    int nargs;
    ArgPtrs args;
    int min_q;  // particles wanted per quadrant
    uint64_t seed, counter;
    const int32_t* list;   // listed cells of the colour
    const int32_t* count;  // their number
    jp_stats* st;
    PhaseInj pi;
};

// Julia's min / max on Float64 (NaN-propagating, -0.0 below 0.0) and clamp
__device__ inline double jl_min(double x, double y) {
    if (x != x || y != y) return x != x ? x : y;
    return (x < y || (x == y && signbit(x) && !signbit(y))) ? x : y;
}
__device__ inline double jl_max(double x, double y) {
    if (x != x || y != y) return x != x ? x : y;
    return (x > y || (x == y && !signbit(x) && signbit(y))) ? x : y;
}

// _grid2particle at corner cell idx of F (dims nn), t = (p - x0) * inv(di),
// clamped to the extrema of the 2^D corner values (src/Particles/
// injection.jl:299-314, cell_field :395-409)
template <int D>
__device__ double g2p_clamped(const double* __restrict__ F, const int64_t (&nn)[D],
                              const int64_t (&idx)[D], const double (&p)[D],
                              const double (&x0)[D], const double (&inv)[D]) {
    double v[1 << D], t[D];
#pragma unroll
    for (int q = 0; q < (1 << D); ++q) {
        int64_t o = 0, stride = 1;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            o += (idx[d] + ((q >> d) & 1)) * stride;
            stride *= nn[d];
        }
        v[q] = F[o];
    }
#pragma unroll
    for (int d = 0; d < D; ++d) t[d] = (p[d] - x0[d]) * inv[d];
    double r = lerp1(t[1], lerp1(t[0], v[0], v[1]), lerp1(t[0], v[2], v[3]));
    if constexpr (D == 3)
        r = lerp1(t[2], r, lerp1(t[1], lerp1(t[0], v[4], v[5]), lerp1(t[0], v[6], v[7])));
    double lo = v[0], hi = v[0];
#pragma unroll
    for (int q = 1; q < (1 << D); ++q) {
        lo = jl_min(lo, v[q]);
        hi = jl_max(hi, v[q]);
    }
    return r > hi ? hi : (r < lo ? lo : r);
}

constexpr int kInjRound = 16;  // searches per pass over the neighbours
// a box whose squared distance exceeds a search's bound by this factor holds no
// element within the tie range (the margin covers the roundings)
constexpr double kPrune = 1.0 + 0x1p-40;

// PHASE (inject_particles_phase!): every short quadrant is topped up (the
// reference continues past a full one, :278, where inject_particles! breaks),
// the new particle takes its nearest neighbour's phase, and each arg is
// interpolated from its field (cell-centred or nodal), clamped to the corner
// extrema.
template <int D, bool SPLIT, bool PHASE>
__global__ void __launch_bounds__(kBlock) k_inject_cells(InjectCells<D> a) {
    using P = typename std::conditional<SPLIT, float, double>::type;
    constexpr int NQ = D == 2 ? 4 : 8, NB = D == 2 ? 9 : 27, CENTER = (NB - 1) / 2, B = 4;
    __shared__ double s_best[kBlock / 64][kInjRound][64];
    __shared__ uint8_t s_nb[kBlock / 64][kInjRound][64];  // neighbour cell of the minimum
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const Grid<D>& g = a.g;
    const int64_t C = g.C;
    const int K = g.K;
    const uint64_t full = K == 64 ? ~0ull : ((1ull << K) - 1);
    const bool slot = lane < K;
    const int64_t nwv = (int64_t)gridDim.x * (kBlock / 64);
    const int64_t total = *a.count;
    int64_t n_inj = 0, n_orph = 0;
    double h[D];  // split form: the uniform vertex spacing
#pragma unroll
    for (int d = 0; d < D; ++d) h[d] = SPLIT ? g.xv[d].dx[0] : 1.0;
    auto pos = [&](int64_t e, P (&v)[D]) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if constexpr (SPLIT) v[d] = a.u[d][e];
            else v[d] = a.x[d][e];
        }
    };
    for (int64_t w = blockIdx.x * (int64_t)(kBlock / 64) + wv; w < total; w += nwv) {
        const int64_t c = __builtin_amdgcn_readfirstlane(a.list[w]);
        int64_t I[D];
        unlin<D>(g.ni, c, I);
        const int64_t e = c + C * (slot ? lane : 0);
        P q[D];  // this cell's slot; the new position once planned
        pos(e, q);
        // lane n: neighbour n's occupancy word and whether its box is known
        auto neighbour = [&](int n, bool& in) {
            int64_t J[D];
            in = true;
            int rr = n;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                J[d] = I[d] + rr % 3 - 1;
                rr /= 3;
                in = in && J[d] >= 0 && J[d] < g.ni[d];
            }
            return lin<D>(g.ni, J);
        };
        bool inside_grid;
        const int64_t cl = neighbour(lane < NB ? lane : CENTER, inside_grid);
        const uint64_t occ_n = inside_grid ? a.occw[cl] : 0ull;
        const uint32_t out_n = inside_grid ? a.out[cl] : 0u;
        const uint64_t occ = (uint64_t)__double_as_longlong(
            readlane_d(__longlong_as_double((long long)occ_n), CENTER));
        double xv[D], xw[D], dq[D], r[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            xv[d] = g.xv[d].x[I[d]];
            xw[d] = g.xv[d].x[I[d] + 1];
            dq[d] = g.xv[d].dx[I[d]] / 2.0;
        }
        const bool act0 = (occ >> lane) & 1;
#pragma unroll
        for (int d = 0; d < D; ++d)
            r[d] = slot && !act0 ? uniform53(a.seed, (uint64_t)c, lane, d, 2, a.counter) : 0.0;
        // plan: the quadrants in order, each topped up from the lowest free
        // slots until it holds min_q particles (injection.jl:87-126)
        uint64_t injm = 0;
        bool act = act0;
        for (int qd = 0; qd < NQ; ++qd) {
            bool inside = act;
            double v[D];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int bit = (qd >> d) & 1;
                if constexpr (SPLIT) {
                    const float q0 = 0.5f * (float)bit;
                    inside = inside && (q0 < q[d] && q[d] < q0 + 0.5f);
                } else {
                    v[d] = xv[d] + dq[d] * (double)bit;
                    inside = inside && (v[d] < q[d] && q[d] < v[d] + dq[d]);
                }
            }
            const int num = __popcll(__ballot(inside));
            if (num >= a.min_q) {
                if constexpr (PHASE) continue;
                break;
            }
            const uint64_t t = lowest_bits(~__ballot(act) & full, a.min_q - num);
            injm |= t;
            if ((t >> lane) & 1) {
                // new_particle: vertex + dq * muladd(0.95, rand, 0.05)
                act = true;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const double f = fma(0.95, r[d], 0.05);
                    if constexpr (SPLIT)
                        q[d] = (float)(0.5 * (double)((qd >> d) & 1) + 0.5 * f);
                    else
                        q[d] = v[d] + dq[d] * f;
                }
            }
        }
        if (!injm) continue;
        // the searches, in injection (= ascending slot) order; lane j of `src`
        // records injection j's nearest particle (order nb*64 + slot)
        int src = 0x7fffffff;
        const int ninj = __popcll(injm);
        uint64_t todo = injm;
        for (int j0 = 0; j0 < ninj; j0 += kInjRound) {
            const int nj = ninj - j0 < kInjRound ? ninj - j0 : kInjRound;
            auto new_pos = [&](int ip, P (&pn)[D]) {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    if constexpr (SPLIT) pn[d] = readlane_f(q[d], ip);
                    else pn[d] = readlane_d(q[d], ip);
                }
            };
            // the cell's own candidates (its particles before the call and the
            // injections before each search's), and the neighbours whose box
            // the best of them does not rule out
            uint32_t need = 0, mine = 0;  // of the round; lane j: of search j
            uint64_t bits = todo;
            for (int j = 0; j < nj; ++j, bits &= bits - 1) {
                const int ip = __builtin_ctzll(bits);
                P pn[D];
                new_pos(ip, pn);
                const bool cand = (act0 || (((injm >> lane) & 1) && lane < ip)) && lane != ip;
                double s = 0.0;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    double t;
                    if constexpr (SPLIT)
                        t = ((double)q[d] - (double)pn[d]) * h[d];
                    else
                        t = q[d] - pn[d];
                    s = d == 0 ? t * t : s + t * t;
                }
                const bool some = cand && s < __builtin_inf();  // (not NaN)
                s = some ? s : __builtin_inf();
                s_best[wv][j][lane] = s;
                s_nb[wv][j][lane] = (uint8_t)(some ? CENTER : 0xFF);
                // an upper bound of the minimum: its high word, rounded up
                const uint32_t hi = wave_min((uint32_t)((uint64_t)__double_as_longlong(s) >> 32));
                const double bound = hi >= 0x7ff00000u
                                         ? __builtin_inf()
                                         : __longlong_as_double((long long)(
                                               ((uint64_t)hi << 32) | 0xFFFFFFFFull));
                double lb = 0.0;  // lane n: to neighbour n's box
                int rr = lane;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    const int o = rr % 3 - 1;
                    rr /= 3;
                    double t;
                    if constexpr (SPLIT)
                        t = (o < 0 ? (double)pn[d] : 1.0 - (double)pn[d]) * h[d];
                    else
                        t = o < 0 ? pn[d] - xv[d] : xw[d] - pn[d];
                    t = o == 0 || !(t > 0.0) ? 0.0 : t;
                    lb = lb + t * t;
                }
                const uint32_t nd = (uint32_t)__ballot(
                    lane < NB && lane != CENTER && occ_n != 0 &&
                    (out_n != 0 || !(lb > bound * kPrune)));
                need |= nd;
                if (lane == j) mine = nd;
            }
            while (need) {
                int nb[B];
                P p[B][D];
                bool on[B];
                uint32_t group = 0;
#pragma unroll
                for (int n = 0; n < B; ++n) {
                    nb[n] = need ? __builtin_ctz(need) : 0;
                    on[n] = false;
                    if (!need) continue;
                    group |= 1u << nb[n];
                    need &= need - 1;
                    bool in;
                    const int64_t e2 = neighbour(nb[n], in) + C * lane;
                    const uint64_t o = (uint64_t)__double_as_longlong(
                        readlane_d(__longlong_as_double((long long)occ_n), nb[n]));
                    on[n] = (o >> lane) & 1;
                    if (on[n]) pos(e2, p[n]);
                }
                bits = todo;
                for (int j = 0; j < nj; ++j, bits &= bits - 1) {
                    if (!((uint32_t)__builtin_amdgcn_readlane((int)mine, j) & group)) continue;
                    P pn[D];
                    new_pos(__builtin_ctzll(bits), pn);
                    double best = s_best[wv][j][lane];
                    int at = s_nb[wv][j][lane];
#pragma unroll
                    for (int n = 0; n < B; ++n) {
                        double s = 0.0;
                        int rr = nb[n];
#pragma unroll
                        for (int d = 0; d < D; ++d) {
                            double t;
                            if constexpr (SPLIT)
                                t = ((double)(rr % 3 - 1) + (double)p[n][d] - (double)pn[d]) * h[d];
                            else
                                t = p[n][d] - pn[d];
                            rr /= 3;
                            s = d == 0 ? t * t : s + t * t;
                        }
                        // (a NaN coordinate compares neither less nor near)
                        if (!on[n] || !(s <= best * (1.0 + 0x1p-50)) || s == __builtin_inf())
                            continue;
                        // roots that round alike: the lower cell stays
                        const bool same = best <= s * (1.0 + 0x1p-50) && sqrt(s) == sqrt(best);
                        if (same ? nb[n] < at : s < best) {
                            best = s;
                            at = nb[n];
                        }
                    }
                    s_best[wv][j][lane] = best;
                    s_nb[wv][j][lane] = (uint8_t)at;
                }
            }
            for (int j = 0; j < nj; ++j, todo &= todo - 1) {
                const double s = s_best[wv][j][lane];
                const int at = s_nb[wv][j][lane];
                double best = s;
                int border = at == 0xFF ? 0x7fffffff : at * 64 + lane;
                const int own = border;
                wave_argmin(best, border);
                resolve_ties_at(s, own, best, border);
                if (lane == j0 + j) src = border;
            }
        }
        const bool inj = (injm >> lane) & 1;
        if (inj) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if constexpr (SPLIT) a.u[d][e] = q[d];
                else a.x[d][e] = q[d];
            }
            a.index[e] = 1;
        }
        if (lane == 0) a.occw[c] = occ | injm;  // for the later colours
        if constexpr (!SPLIT) {  // (a split offset drawn lies in [0, 1])
            bool out = false;
#pragma unroll
            for (int d = 0; d < D; ++d) out = out || !(xv[d] <= q[d] && q[d] <= xw[d]);
            if (__any(inj && out) && lane == 0) a.out[c] = 1;
        }
        // values copied from the sources: one load per injection, all in
        // flight together; then the copies in injection order, a source in
        // this cell read from the current values
        int64_t es = e;
        const bool found = lane < ninj && src != 0x7fffffff;
        if (found) {
            int64_t J[D];
            int rr = src >> 6;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                J[d] = I[d] + rr % 3 - 1;
                rr /= 3;
            }
            es = lin<D>(g.ni, J) + C * (src & 63);
        }
        auto copy = [&](double* const* F, int n) {
            double fc[2], nv[2];  // two fields at a time
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                fc[f] = f < n ? F[f][e] : 0.0;
                nv[f] = f < n && found ? F[f][es] : 0.0;
            }
            uint64_t bits = injm;
            for (int j = 0; j < ninj; ++j, bits &= bits - 1) {
                const int ip = __builtin_ctzll(bits);
                const int sj = __builtin_amdgcn_readlane(src, j);
                if (sj == 0x7fffffff) continue;  // orphan: the slot keeps its value
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    const double v = (sj >> 6) == CENTER ? readlane_d(fc[f], sj & 63)
                                                         : readlane_d(nv[f], j);
                    if (lane == ip) fc[f] = v;
                }
            }
            if (inj) {
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    if (f < n) F[f][e] = fc[f];
            }
        };
        if constexpr (PHASE) {
            double* const ph[2] = {a.pi.phases, a.pi.phases};
            copy(ph, 1);
            if (inj) {
                // args from fields: nodal at this cell's corners, cell-centred
                // at the shifted index clamped to 1..ni-1 (1-based; a grid of one
                // cell in a dimension has none, and no cell-centred field)
                int64_t nnv[D], nnc[D], ic[D], Iv[D];
                double xc0[D], ivc[D], xv0[D], ivv[D], pn[D];
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    pn[d] = q[d];
                    nnv[d] = g.ni[d] + 1;
                    nnc[d] = g.ni[d];
                    Iv[d] = I[d];
                    xv0[d] = xv[d];
                    ivv[d] = g.xv[d].idx[I[d]];
                    if (a.pi.centred) {
                        const int64_t k = pn[d] < xv[d] + dq[d] ? I[d] - 1 : I[d];
                        ic[d] = k > g.ni[d] - 2 ? g.ni[d] - 2 : (k < 0 ? 0 : k);
                        xc0[d] = a.pi.xc[d].x[ic[d]];
                        ivc[d] = a.pi.xc[d].idx[ic[d]];
                    }
                }
                for (int f = 0; f < a.nargs; ++f)
                    a.args.p[f][e] = ((a.pi.centred >> f) & 1)
                                         ? g2p_clamped<D>(a.pi.fields[f], nnc, ic, pn, xc0, ivc)
                                         : g2p_clamped<D>(a.pi.fields[f], nnv, Iv, pn, xv0, ivv);
            }
        } else {
            for (int f = 0; f < a.nargs; f += 2) copy(a.args.p + f, a.nargs - f < 2 ? 1 : 2);
        }
        n_orph += __popcll(__ballot(lane < ninj && src == 0x7fffffff));
        n_inj += ninj;
    }  // work list
    if (lane == 0) {
        stat_add(a.st, ST_INJECTED, n_inj);
        stat_add(a.st, ST_ORPHAN, n_orph);
    }
}

// the colour launches: offsets (o_1 outer ... o_D inner), persistent
// wavefronts, one listed cell at a time each
template <int D, bool SPLIT, bool PHASE>
int launch_inject_cells(jp_ctx* ctx, InjectCells<D> a, const InjectLists& L, int64_t cap) {
    for (int ph = 0; ph < (D == 2 ? 4 : 8); ++ph) {
        a.list = L.list + (int64_t)ph * cap;
        a.count = L.total + ph;
        a.occw = L.occ;
        a.out = L.out;
        k_inject_cells<D, SPLIT, PHASE>
            <<<(unsigned)inject_blocks(ctx, cap), kBlock, 0, ctx->stream>>>(a);
        JP_LAUNCHED(ctx);
    }
    return JP_OK;
}

}  // namespace jp
