// jp_hotpath.hip -- FP64 drop-in kernels for JustPIC's particle hot path on
// gfx950: init, particle2grid, grid2particle and injection, 2D and 3D, on the
// B = 0 cell-plane layout data[c + C*k] (advection: jp_advect.hip, move:
// jp_move.hip).
#include "jp_ctx.hpp"
#include "jp_inject2.hpp"
#include "jp_inject_cells.hpp"

#include <cmath>
#include <type_traits>

using namespace jp;

namespace {

__device__ inline double dnan() { return __builtin_nan(""); }

// ============================================================ init
// fill_coords_index! (src/Particles/particles_utils.jl:168-194), one thread
// per cell writing its K slots (coalesced across the cell planes).
template <int D>
__global__ void __launch_bounds__(kBlock) k_init(Grid<D> g, Ptr3 coords, uint8_t* __restrict__ index,
                                                 int npq, uint64_t seed) {
    int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c >= g.C) return;
    int64_t I[D];
    unlin<D>(g.ni, c, I);
    double x0[D], dx[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        x0[d] = g.xv[d].x[I[d]];
        dx[d] = g.xv[d].dx[I[d]];
    }
    constexpr int nq = D == 2 ? 4 : 8;
    int l = 0;
    for (int iq = 0; iq < nq; ++iq) {
        double xc[D];
#pragma unroll
        for (int d = 0; d < D; ++d) xc[d] = x0[d] + (dx[d] * (double)((iq >> d) & 1)) / 2.0;
        for (int n = 0; n < npq; ++n, ++l) {
            int64_t e = c + g.C * l;
#pragma unroll
            for (int d = 0; d < D; ++d)
                coords.p[d][e] = xc[d] + (dx[d] / 2.0) * uniform53(seed, (uint64_t)c, l, d, 1, 0);
            index[e] = 1;
        }
    }
    for (; l < g.K; ++l) {
        int64_t e = c + g.C * l;
#pragma unroll
        for (int d = 0; d < D; ++d) coords.p[d][e] = dnan();
        index[e] = 0;
    }
}

// ============================================================ particle2grid
// The reference's weight of a particle at distance d = sqrt(s) from a node is
// 1 / (d d), with the square root, the product and the quotient each correctly
// rounded.  weights() gives the same bits as sqrt(s), d * d and
// 1.0 / (d d) for kSafeLo <= s < kSafeHi, where nothing overflows, underflows
// or is denormal, without the scaling and special-case selects of the general
// operations: the square root by Goldschmidt's iteration from the hardware
// estimate and two residual corrections, the quotient from the square of the
// refined reciprocal root by one Newton step and a residual correction (each
// last step rounds a result already within an ulp: P. Markstein, IBM J. Res.
// Dev. 34, 1990).  23 instructions, one of them a slow one, instead of 36 with
// two.
constexpr uint32_t kSafeLo = (1023u - 480u) << 20;  // high words of 2^-480, 2^480
constexpr uint32_t kSafeHi = (1023u + 480u) << 20;
// B of them side by side, step by step: each is one chain of dependent
// operations.
template <int B>
__device__ inline void weights(const double (&s)[B], double (&wi)[B]) {
    double g[B], h[B], e[B];
#pragma unroll
    for (int j = 0; j < B; ++j) h[j] = __builtin_amdgcn_rsq(s[j]);
#pragma unroll
    for (int j = 0; j < B; ++j) g[j] = s[j] * h[j];
#pragma unroll
    for (int j = 0; j < B; ++j) h[j] = 0.5 * h[j];
#pragma unroll
    for (int j = 0; j < B; ++j) e[j] = fma(-h[j], g[j], 0.5);
#pragma unroll
    for (int j = 0; j < B; ++j) g[j] = fma(g[j], e[j], g[j]);
#pragma unroll
    for (int j = 0; j < B; ++j) h[j] = fma(h[j], e[j], h[j]);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int j = 0; j < B; ++j) e[j] = fma(-g[j], g[j], s[j]);
#pragma unroll
        for (int j = 0; j < B; ++j) g[j] = fma(e[j], h[j], g[j]);  // the second: sqrt(s)
    }
#pragma unroll
    for (int j = 0; j < B; ++j) {
        g[j] = g[j] * g[j];
        h[j] = (4.0 * h[j]) * h[j];
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int j = 0; j < B; ++j) e[j] = fma(-g[j], h[j], 1.0);
#pragma unroll
        for (int j = 0; j < B; ++j) h[j] = fma(e[j], h[j], h[j]);
    }
#pragma unroll
    for (int j = 0; j < B; ++j) wi[j] = h[j];
}
__device__ inline double weight_any(double s) {
    const double dist = sqrt(s);
    return 1.0 / (dist * dist);
}

// _particle2grid! (src/Interpolations/particle_to_grid.jl:37-199), exact
// reference accumulation order (cells with the last dim outermost, slots
// ascending).  mode 0: wF/w (2D scalar), 1: wF*inv(w).
//
// A thread walks R + 1 layers of cells along the last dimension for a column
// of R nodes (3D: for PY = 2 columns next to each other in y), two nodes of a
// column at a time: a layer adds to the node below it, which is then done, and
// to the node above it.  A particle is loaded once for all of the column's
// nodes that it touches.  A thread per node reads every particle 2^D times, all
// of it past the L2 (a plane sweep of the resident wavefronts is far larger),
// which bounds it at 5 TB/s; columns read it 2 (R + 1) / R times in 2D and
// 3 (R + 1) / R in 3D.
//
// A chunk of B slot planes is straight-line code: every lane computes the
// weights of B slots side by side (garbage for empty slots), then adds those
// of its active slots in order; a chunk that no lane of the wavefront needs
// is skipped.  One range check for the chunk: if any active slot's s lies
// outside weights()'s range, the chunk's weights come from the general
// operations.  The next chunk's loads are in flight meanwhile, unguarded (all
// lanes are on the same slot plane: coalesced across neighbouring cells).
// NF fields per launch, accumulators in registers.  A thread per node with a
// branch per slot and the general operations took 190 us at 512^2 (now 157),
// 49 at 32^2 (31), 192 at 389 x 211 with three fields (77) and 1470 at 61 x 47
// x 74 with two (383).
template <int NF>
struct P2gFields {
    double* F[NF];
    const double* Fp[NF];
};
template <int D, int NF, int PY>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2, 2))) k_p2g(Grid<D> g, P2gFields<NF> fields, CPtr3 coords,
                                                const uint64_t* __restrict__ occw, int mode,
                                                int R, int64_t threads) {
    static_assert(D == 3 || PY == 1, "patches along y in 3D only");
    int64_t t = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if (t >= threads) return;
    constexpr int L = D - 1;  // the dimension walked along
    constexpr int NY = D == 3 ? PY : 1;
    const int64_t n0 = g.ni[0] + 1, n1 = g.ni[1] + 1;
    // node column: x index i, first y index (3D), first index z along L
    const int64_t i = t % n0;
    t /= n0;
    const int64_t ny = (n1 + PY - 1) / PY;
    const int64_t y0 = D == 3 ? (t % ny) * PY : 0;
    const int64_t z0 = (D == 3 ? t / ny : t) * R;
    const double xn = g.xv[0].x[i];
    double yn[NY];
#pragma unroll
    for (int m = 0; m < NY; ++m)
        yn[m] = D == 3 ? g.xv[1].x[y0 + m < n1 ? y0 + m : n1 - 1] : 0.0;
    const int64_t C = g.C;
    constexpr int NU = 2 * (D == 3 ? PY + 1 : 1);  // cells of a layer, in order
    constexpr int B = 4, V = D + NF;
    struct Chunk {
        double v[B][V];
        uint32_t on;  // active slots of the chunk
        int u;        // cell of the layer
    };
    // accumulators of the nodes below ([m][0]) and above ([m][1]) the layer
    double w[NY][2], wF[NY][2][NF];
#pragma unroll
    for (int m = 0; m < NY; ++m)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w[m][h] = 0.0;
#pragma unroll
            for (int f = 0; f < NF; ++f) wF[m][h][f] = 0.0;
        }
    int64_t cell[NU];
    uint64_t bits[NU];
    auto layer = [&](int64_t z, int64_t (&c)[NU], uint64_t (&b)[NU]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int64_t x = i - 1 + (u & 1), y = y0 - 1 + (u >> 1);
            bool ok = x >= 0 && x < g.ni[0] && z >= 0 && z < g.ni[L];
            if (D == 3) ok = ok && y >= 0 && y < g.ni[1];
            c[u] = !ok ? 0 : x + g.ni[0] * (D == 3 ? y + g.ni[1] * z : z);
            b[u] = ok ? occw[c[u]] : 0ull;
        }
    };
    int64_t cell1[NU];
    uint64_t bits1[NU];
    layer(z0 - 1, cell1, bits1);
#pragma unroll 1
    for (int r = 0; r <= R; ++r) {
        const int64_t z = z0 - 1 + r;  // the layer's cells; nodes z (below) and z + 1 (above)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            cell[u] = cell1[u];
            bits[u] = bits1[u];
        }
        double zn[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t zi = z + h;
            zn[h] = g.xv[L].x[zi < 0 ? 0 : (zi > g.ni[L] ? g.ni[L] : zi)];
        }
        // wait for the layer's words and nodes here: a wait inside the chunk
        // loop would be one for all loads in flight
#pragma unroll
        for (int u = 0; u < NU; ++u) asm volatile("" : "+v"(bits[u]));
        asm volatile("" : "+v"(zn[0]), "+v"(zn[1]));
        if (r < R) layer(z + 1, cell1, bits1);
        // chunk by chunk through the layer's cells: cell u, slot plane k up to
        // the wavefront's last occupied one (all uniform over the wavefront),
        // the lane's cell and remaining occupancy bits
        int last[NU], chunks = 0;
#pragma unroll
        for (int v = 0; v < NU; ++v) {
            int top = 0;
            for (uint64_t any = bits[v]; __any(any != 0); any >>= B) top += B;
            last[v] = top > 0 ? top : B;
            chunks += last[v] / B;
        }
        int u = 0, k = 0, end = last[0];
        int64_t c = cell[0];
        uint64_t left = bits[0];
        auto advance = [&]() __attribute__((always_inline)) {
            k += B;
            left >>= B;
            if (k < end || u == NU - 1) return;
            ++u;
            k = 0;
#pragma unroll
            for (int v = 1; v < NU; ++v) {
                c = u == v ? cell[v] : c;
                left = u == v ? bits[v] : left;
                end = u == v ? last[v] : end;
            }
        };
        // (always the same number of loads, also past the last chunk, so that
        // the wait for one buffer leaves the other's loads in flight)
        auto read = [&](Chunk& ch) __attribute__((always_inline)) {
            ch.on = (uint32_t)left & ((1u << B) - 1);
            ch.u = u;
#pragma unroll
            for (int j = 0; j < B; ++j) {
                const int64_t plane = C * (k + j < g.K ? k + j : g.K - 1);
#pragma unroll
                for (int d = 0; d < D; ++d) ch.v[j][d] = coords.p[d][plane + c];
#pragma unroll
                for (int f = 0; f < NF; ++f) ch.v[j][D + f] = fields.Fp[f][plane + c];
            }
        };
        auto add = [&](const Chunk& ch) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < NY; ++m) {
                if (D == 3 && (ch.u >> 1) != m && (ch.u >> 1) != m + 1) continue;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (h == 0 ? r == 0 : r == R) continue;  // another thread's node
                    double s[B], wi[B];
                    uint32_t far = 0;
#pragma unroll
                    for (int j = 0; j < B; ++j) {
                        const double a = xn - ch.v[j][0];
                        s[j] = a * a;
                        if (D == 3) {
                            const double b = yn[m] - ch.v[j][1];
                            s[j] = s[j] + b * b;
                        }
                        const double e = zn[h] - ch.v[j][L];
                        s[j] = s[j] + e * e;
                        const uint32_t off = (uint32_t)__double2hiint(s[j]) - kSafeLo;
                        far = ((ch.on >> j) & 1) && off > far ? off : far;
                    }
                    weights<B>(s, wi);
                    if (__any(far >= kSafeHi - kSafeLo)) {
#pragma unroll
                        for (int j = 0; j < B; ++j) wi[j] = weight_any(s[j]);
                    }
#pragma unroll
                    for (int j = 0; j < B; ++j) {
                        if (!((ch.on >> j) & 1)) continue;
                        w[m][h] += wi[j];
#pragma unroll
                        for (int f = 0; f < NF; ++f)
                            wF[m][h][f] = fma(wi[j], ch.v[j][D + f], wF[m][h][f]);
                    }
                }
            }
        };
        Chunk a, b;
        read(a);
#pragma unroll 1
        for (int n = 0; n < chunks; n += 2) {
            advance();
            read(b);
            add(a);
            advance();
            read(a);
            add(b);
        }
        // the nodes below are done; those above are below the next layer
#pragma unroll
        for (int m = 0; m < NY; ++m) {
            if (r > 0 && z <= g.ni[L] && (D == 2 || y0 + m < n1)) {
                const int64_t node = i + n0 * (D == 3 ? y0 + m + n1 * z : z);
                if (mode == 0) {
                    fields.F[0][node] = wF[m][0][0] / w[m][0];
                } else {
                    const double iw = 1.0 / w[m][0];
#pragma unroll
                    for (int f = 0; f < NF; ++f) fields.F[f][node] = wF[m][0][f] * iw;
                }
            }
            w[m][0] = w[m][1];
            w[m][1] = 0.0;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                wF[m][0][f] = wF[m][1][f];
                wF[m][1][f] = 0.0;
            }
        }
    }
}

// ============================================================ grid2particle
// grid2particle_classic! (src/Interpolations/grid_to_particle.jl:38-82).  A thread
// takes 8 slots of its cell (blockIdx.y): the cell's corners and vertices are read
// once, and the slots' loads are in flight together (bound by the slots' bytes:
// 512 x 384 cells of 48 slots 52 us with a thread per slot, now 40).
template <int D, int NS>
__global__ void __launch_bounds__(kBlock) k_g2p(Grid<D> g, double* __restrict__ Fp,
                                                const double* __restrict__ F, CPtr3 coords,
                                                const uint8_t* __restrict__ index) {
    int64_t c, I[D];
    if (!row_cell<D>(g, c, I)) return;
    const int kb = (int)blockIdx.y * NS;
    double v[1 << D], x[D], ix[D];
    cell_corners<D>(g, F, I, v);
#pragma unroll
    for (int d = 0; d < D; ++d) {
        x[d] = g.xv[d].x[I[d]];
        ix[d] = g.xv[d].idx[I[d]];
    }
    const uint32_t on = slots_on<NS>(index, c, g.C, kb, g.K);
    double p[NS][D];
    load_slots<D, NS>(coords, c, g.C, kb, on, p);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        if (!((on >> j) & 1)) continue;
        double t[D];
#pragma unroll
        for (int d = 0; d < D; ++d) t[d] = (p[j][d] - x[d]) * ix[d];
        Fp[c + g.C * (kb + j)] = lerp_cell<D>(v, t);
    }
}

// ============================================================ injection
// The first quadrant decides whether a cell injects at all: the reference
// breaks out of the quadrant loop as soon as one quadrant holds min_q
// particles (src/Particles/injection.jl:100), and injection into a cell never
// changes the particles of other cells.  One coalesced pass over all cells
// therefore lists the only cells that can inject, per colour; the colour
// phases then run the reference loop on those cells only.  ANYQ (the phase
// variant, which moves on to the next quadrant instead of breaking,
// src/Particles/injection.jl:278): a cell is listed when any quadrant is short.
// BOX: also whether a particle lies outside the cell's box, for k_inject_cells (in
// the scan of k_inject2 it took 16.1 us for 12.8 at 32^2).
template <int D, bool ANYQ, bool BOX>
__global__ void __launch_bounds__(kBlock) k_inject_scan(Grid<D> g, CPtr3 coords,
                                                        const uint8_t* __restrict__ index,
                                                        int min_q, InjectLists L) {
    const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const bool valid = c < g.C;  // all lanes stay for the wavefront append
    int64_t I[D];
    unlin<D>(g.ni, valid ? c : 0, I);
    int num = 0;
    bool out = false;  // a particle outside the cell's box (or NaN)
    int cnt_q[1 << D] = {};  // ANYQ: particles strictly inside quadrants 1..2^D-1
    if (valid) {
        double lo[D], hi[D], hq[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            lo[d] = g.xv[d].x[I[d]];
            hi[d] = BOX ? g.xv[d].x[I[d] + 1] : 0.0;
            hq[d] = g.xv[d].dx[I[d]] / 2.0;
        }
        // quadrant c11: vertex + dq*0 (src/Particles/injection.jl:442-448)
        double q0[D], q1[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            q0[d] = lo[d] + hq[d] * 0.0;
            q1[d] = q0[d] + hq[d];
        }
        const uint64_t act = active_slots(index, c, g.C, g.K);
        constexpr int B = 16;  // slots per chunk; lanes share the slot plane (coalesced)
        for (int k0 = 0; k0 < g.K; k0 += B) {
            double pb[B][D];
#pragma unroll
            for (int j = 0; j < B; ++j) {
                const bool on = (act >> (k0 + j)) & 1;
#pragma unroll
                for (int d = 0; d < D; ++d) pb[j][d] = on ? coords.p[d][c + g.C * (k0 + j)] : 0.0;
            }
#pragma unroll
            for (int j = 0; j < B; ++j) {
                const bool on = (act >> (k0 + j)) & 1;
                bool inside = on;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    inside = inside & (q0[d] < pb[j][d] && pb[j][d] < q1[d]);
                    if constexpr (BOX) out = out | (on & !(lo[d] <= pb[j][d] & pb[j][d] <= hi[d]));
                }
                num += inside ? 1 : 0;
                if constexpr (ANYQ) {
                    // the other quadrants (vertex + dq*bit, the wave kernel's bounds)
#pragma unroll
                    for (int q = 1; q < (1 << D); ++q) {
                        bool in_q = on;
#pragma unroll
                        for (int d = 0; d < D; ++d) {
                            const double v = lo[d] + hq[d] * (double)((q >> d) & 1);
                            in_q = in_q & (v < pb[j][d] && pb[j][d] < v + hq[d]);
                        }
                        cnt_q[q] += in_q ? 1 : 0;
                    }
                }
            }
        }
        L.occ[c] = act;
        if (BOX) L.out[c] = out ? 1u : 0u;
    }
    bool want = valid && num < min_q;
    if constexpr (ANYQ) {
#pragma unroll
        for (int q = 1; q < (1 << D); ++q) want = want || (valid && cnt_q[q] < min_q);
    }
    if (valid && L.state) L.state[c] = want ? 1u : 0u;
    int col = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) col = col * 2 + (int)(I[d] & 1);
    wave_segment<D == 2 ? 4 : 8>(want, col, (int32_t)c, c >> 6, L.nwave, L.seg, L.cnt);
}

// ============================================================ host side
int check_ptrs(jp_ctx* ctx, int n, const void* const* p, const char* what) {
    if (!p) return fail(ctx, JP_ERR_ARG, "null %s array", what);
    for (int i = 0; i < n; ++i)
        if (!p[i]) return fail(ctx, JP_ERR_ARG, "null %s pointer %lld", what, i);
    return JP_OK;
}

Ptr3 ptr3(double* const* c, int D) {
    Ptr3 p{{nullptr, nullptr, nullptr}};
    for (int d = 0; d < D; ++d) p.p[d] = c[d];
    return p;
}
CPtr3 cptr3(const double* const* c, int D) {
    CPtr3 p{{nullptr, nullptr, nullptr}};
    for (int d = 0; d < D; ++d) p.p[d] = c[d];
    return p;
}
ArgPtrs argptrs(double* const* a, int n) {
    ArgPtrs p;
    for (int i = 0; i < JP_MAX_ARGS; ++i) p.p[i] = i < n ? a[i] : nullptr;
    return p;
}

Off3 phase_offsets(int D, int ph, int base) {
    // for o1 in 1:base, o2 in 1:base [, o3 in 1:base] -- last offset fastest; 0-based result
    Off3 o{{0, 0, 0}};
    if (D == 2) {
        o.o[0] = ph / base;
        o.o[1] = ph % base;
    } else {
        o.o[0] = ph / (base * base);
        o.o[1] = (ph / base) % base;
        o.o[2] = ph % base;
    }
    return o;
}

template <int D>
int run_init(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords, uint8_t* index, int npq,
             uint64_t seed) {
    Grid<D> G = to_grid<D>(g);
    k_init<D><<<blocks_for(G.C), kBlock, 0, ctx->stream>>>(G, ptr3(coords, D), index, npq, seed);
    JP_LAUNCHED(ctx);
    return finish(ctx);
}

// occ_fixed: caller-provided occupancy-word scratch of at least C words (the
// allocation-free entry point); null: the context's growable scratch
template <int D>
int run_p2g(jp_ctx* ctx, const jp_cellgrid* g, int nf, double* const* F, const double* const* Fp,
            const double* const* coords, const uint8_t* index, int mode,
            uint64_t* occ_fixed = nullptr) {
    Grid<D> G = to_grid<D>(g);
    int rc;
    uint64_t* occ = occ_fixed;
    if (!occ) {
        if ((rc = ensure_scratch(ctx, (size_t)G.C * 8))) return rc;
        occ = static_cast<uint64_t*>(ctx->scratch);
    }
    if ((rc = occ_words(ctx, index, G.C, G.K, occ))) return rc;
    constexpr int PY = D == 3 ? 2 : 1;
    int64_t cols = G.ni[0] + 1;  // node columns
    if (D == 3) cols *= (G.ni[1] + 1 + PY - 1) / PY;
    // nodes per thread: as many (a power of two, up to 16) as leave about 9
    // wavefronts for every 16 SIMDs.  Longer columns read less, fewer
    // wavefronts leave SIMDs idle; R = 1, 2, 4, 8 at 512^2 (4116 wavefronts
    // with R = 1): 187, 180, 157, 190 us; 389 x 211, three fields (1292): 104,
    // 77, 118, 216; 61 x 47 x 74, two fields (1744): 509, 383, 542, 965; 32^2
    // (18): 31, 51, 91, 172.
    const int64_t want = (int64_t)ctx->num_cu * 4 * 9 / 16 * 64;  // threads
    int R = 1;
    while (R < 16 && cols * ((G.ni[D - 1] + 2 * R) / (2 * R)) >= want) R *= 2;
    const int64_t threads = cols * ((G.ni[D - 1] + R) / R);
    // up to three fields per launch (their sums are independent: every launch
    // computes the same weights); four would spill
    for (int f = 0; f < nf;) {
        const int m = nf - f < 3 ? nf - f : 3;
        auto launch = [&](auto n) {
            constexpr int NF = decltype(n)::value;
            P2gFields<NF> a;
            for (int i = 0; i < NF; ++i) {
                a.F[i] = F[f + i];
                a.Fp[i] = Fp[f + i];
            }
            k_p2g<D, NF, PY><<<blocks_for(threads), kBlock, 0, ctx->stream>>>(
                G, a, cptr3(coords, D), occ, mode, R, threads);
        };
        if (m == 1) launch(std::integral_constant<int, 1>{});
        else if (m == 2) launch(std::integral_constant<int, 2>{});
        else launch(std::integral_constant<int, 3>{});
        JP_LAUNCHED(ctx);
        f += m;
    }
    return finish(ctx);
}

template <int D>
int run_g2p(jp_ctx* ctx, const jp_cellgrid* g, double* Fp, const double* F,
            const double* const* coords, const uint8_t* index) {
    Grid<D> G = to_grid<D>(g);
    const int ns = slots_per_thread(ctx, G);
    const dim3 grid((unsigned)row_blocks<D>(G), (unsigned)((G.K + ns - 1) / ns));
    if (ns == 2)
        k_g2p<D, 2><<<grid, kBlock, 0, ctx->stream>>>(G, Fp, F, cptr3(coords, D), index);
    else
        k_g2p<D, kSlots8><<<grid, kBlock, 0, ctx->stream>>>(G, Fp, F, cptr3(coords, D), index);
    JP_LAUNCHED(ctx);
    return finish(ctx);
}

template <int D>
InjectCells<D> inject_cells(const Grid<D>& G, double* const* coords, uint8_t* index, int nargs,
                            double* const* args, int min_q, uint64_t seed, uint64_t counter,
                            jp_stats* st) {
    InjectCells<D> a{};
    a.g = G;
    for (int d = 0; d < D; ++d) a.x[d] = coords[d];
    a.index = index;
    a.nargs = nargs;
    a.args = argptrs(args, nargs);
    a.min_q = min_q;
    a.seed = seed;
    a.counter = counter;
    a.st = st;
    return a;
}

template <int D>
int run_inject(jp_ctx* ctx, const jp_cellgrid* gc, double* const* coords, uint8_t* index,
               int nargs, double* const* args, int min_xcell, uint64_t seed, uint64_t counter,
               jp_stats* stats) {
    Grid<D> G = to_grid<D>(gc);
    int rc;
    if ((rc = stats_begin(ctx, stats))) return rc;
    constexpr int NQ = D == 2 ? 4 : 8;
    const int min_q = (min_xcell + NQ - 1) / NQ;
    // cells per colour: at most prod(ceil(ni/2))
    int64_t cap = 1;
    for (int d = 0; d < D; ++d) cap *= (G.ni[d] + 1) / 2;
    InjectLists L;
    const bool two = D == 2 && nargs <= 1;  // the 2D kernel (k_inject2)
    const bool ordered = two && inject2_ordered(ctx);
    if ((rc = inject_lists(ctx, G.C, NQ, cap, ordered, L))) return rc;
    if (two)
        k_inject_scan<D, false, D == 3><<<blocks_for(G.C), kBlock, 0, ctx->stream>>>(
            G, cptr3(coords, D), index, min_q, L);
    else
        k_inject_scan<D, false, true><<<blocks_for(G.C), kBlock, 0, ctx->stream>>>(
            G, cptr3(coords, D), index, min_q, L);
    JP_LAUNCHED(ctx);
    if ((rc = join_segments(ctx, NQ, L))) return rc;
    jp_stats* st = stats ? dstats(ctx) : nullptr;
    if constexpr (D == 2) {
        if (two) {
            Inject2 a{};
            a.g = G;
            a.x[0] = coords[0];
            a.x[1] = coords[1];
            a.index = index;
            a.arg = nargs ? args[0] : nullptr;
            a.min_q = min_q;
            a.seed = seed;
            a.counter = counter;
            a.occw = L.occ;
            a.st = st;
            if ((rc = launch_inject2<false>(ctx, a, L, cap))) return rc;
        }
    }
    if (!two) {
        InjectCells<D> a = inject_cells<D>(G, coords, index, nargs, args, min_q, seed, counter, st);
        if ((rc = launch_inject_cells<D, false, false>(ctx, a, L, cap))) return rc;
    }
    if ((rc = stats_end(ctx, stats))) return rc;
    if (ordered && stats && (rc = inject_wait_report(ctx))) return rc;
    return finish(ctx);
}

// inject_particles_phase! (src/Particles/injection.jl:146-325): the same
// scan / colour structure, cells listed when any quadrant is short
template <int D>
int run_inject_phase(jp_ctx* ctx, const jp_cellgrid* gc, const jp_axis* xc,
                     double* const* coords, uint8_t* index, double* phases, int nargs,
                     double* const* args, const double* const* fields, uint32_t centred,
                     int min_xcell, uint64_t seed, uint64_t counter, jp_stats* stats) {
    Grid<D> G = to_grid<D>(gc);
    int rc;
    if ((rc = stats_begin(ctx, stats))) return rc;
    constexpr int NQ = D == 2 ? 4 : 8;
    const int min_q = (min_xcell + NQ - 1) / NQ;
    int64_t cap = 1;
    for (int d = 0; d < D; ++d) cap *= (G.ni[d] + 1) / 2;
    InjectLists L;
    if ((rc = inject_lists(ctx, G.C, NQ, cap, false, L))) return rc;
    k_inject_scan<D, true, true><<<blocks_for(G.C), kBlock, 0, ctx->stream>>>(
        G, cptr3(coords, D), index, min_q, L);
    JP_LAUNCHED(ctx);
    if ((rc = join_segments(ctx, NQ, L))) return rc;
    InjectCells<D> a = inject_cells<D>(G, coords, index, nargs, args, min_q, seed, counter,
                                       stats ? dstats(ctx) : nullptr);
    a.pi.phases = phases;
    a.pi.centred = centred;
    for (int f = 0; f < nargs; ++f) a.pi.fields[f] = fields[f];
    for (int d = 0; d < D; ++d) a.pi.xc[d] = Axis{xc[d].x, xc[d].dx, xc[d].inv_dx, xc[d].n};
    if ((rc = launch_inject_cells<D, false, true>(ctx, a, L, cap))) return rc;
    if ((rc = stats_end(ctx, stats))) return rc;
    return finish(ctx);
}

// cell_index (src/particles.jl:205-217) for n points per dimension:
// abs(trunc((x - x0) / dx)) + 1 with dx = |xv[2] - xv[1]| and x0 = first(xv)
// (subtracted only when nonzero: x - 0.0 would turn -0.0 into 0.0, which the
// result does not see either way).  1-based, as the reference returns it.
struct CellIndexArgs {
    const double* x[3];
    int64_t* out[3];
    const double* xv[3];  // vertex axes (only their first two points are read)
};

__global__ void __launch_bounds__(kBlock) k_cell_index(CellIndexArgs a, int ndim, int64_t n) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int d = 0; d < ndim; ++d) {
        const double x0 = a.xv[d][0];
        const double dx = fabs(a.xv[d][1] - x0);
        const double x = a.x[d][i];
        const double q = x0 == 0.0 ? x / dx : (x - x0) / dx;
        // unsafe_trunc(Int, trunc(q)): finite in-grid quotients only
        const int64_t t = (int64_t)trunc(q);
        a.out[d][i] = (t < 0 ? -t : t) + 1;
    }
}

}  // namespace

extern "C" {

int jp_cell_index(jp_ctx* ctx, int ndim, const jp_axis* xv, int64_t n, const double* const* x,
                  int64_t* const* out) {
    if (!ctx) return JP_ERR_STATE;
    if (ndim < 1 || ndim > 3) return fail(ctx, JP_ERR_ARG, "ndim must be 1, 2 or 3%s");
    if (n < 0) return fail(ctx, JP_ERR_ARG, "negative point count%s");
    if (!xv || !x || !out) return fail(ctx, JP_ERR_ARG, "null argument%s");
    CellIndexArgs a{};
    for (int d = 0; d < ndim; ++d) {
        if (!x[d] || !out[d] || !xv[d].x || xv[d].n < 2)
            return fail(ctx, JP_ERR_ARG, "bad axis or array%s (dim %lld)", "", d);
        a.x[d] = x[d];
        a.out[d] = out[d];
        a.xv[d] = xv[d].x;
    }
    if (n == 0) return JP_OK;
    k_cell_index<<<(unsigned)blocks_for(n), kBlock, 0, ctx->stream>>>(a, ndim, n);
    JP_LAUNCHED(ctx);
    return finish(ctx);
}

int jp_init_particles(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords, uint8_t* index,
                      int np_quadrant, uint64_t seed) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index) return fail(ctx, JP_ERR_ARG, "null index%s");
    int nq = g->ndim == 2 ? 4 : 8;
    if (np_quadrant < 0 || np_quadrant * nq > g->max_xcell)
        return fail(ctx, JP_ERR_ARG, "np_quadrant*2^D exceeds max_xcell%s");
    return g->ndim == 2 ? run_init<2>(ctx, g, coords, index, np_quadrant, seed)
                        : run_init<3>(ctx, g, coords, index, np_quadrant, seed);
}

int jp_particle2grid(jp_ctx* ctx, const jp_cellgrid* g, double* F, const double* Fp,
                     const double* const* coords, const uint8_t* index) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index || !F || !Fp) return fail(ctx, JP_ERR_ARG, "null field or index%s");
    double* Fa[1] = {F};
    const double* Fpa[1] = {Fp};
    int mode = g->ndim == 2 ? 0 : 1;
    return g->ndim == 2 ? run_p2g<2>(ctx, g, 1, Fa, Fpa, coords, index, mode)
                        : run_p2g<3>(ctx, g, 1, Fa, Fpa, coords, index, mode);
}

int jp_particle2grid_noalloc(jp_ctx* ctx, const jp_cellgrid* g, double* F, const double* Fp,
                             const double* const* coords, const uint8_t* index) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index || !F || !Fp) return fail(ctx, JP_ERR_ARG, "null field or index%s");
    int64_t C = 1;
    for (int d = 0; d < g->ndim; ++d) C *= g->ni[d];
    if (C > JP_NOALLOC_MAX_CELLS)
        return fail(ctx, JP_ERR_ARG,
                    "particle2grid without allocation supports at most JP_NOALLOC_MAX_CELLS%s "
                    "= 2097152 cells (got %lld)",
                    "", (long long)C);
    if (!ctx->noalloc) return fail(ctx, JP_ERR_STATE, "fixed scratch address unknown%s");
    double* Fa[1] = {F};
    const double* Fpa[1] = {Fp};
    const int mode = g->ndim == 2 ? 0 : 1;
    return g->ndim == 2 ? run_p2g<2>(ctx, g, 1, Fa, Fpa, coords, index, mode, ctx->noalloc)
                        : run_p2g<3>(ctx, g, 1, Fa, Fpa, coords, index, mode, ctx->noalloc);
}

int jp_particle2grid_multi(jp_ctx* ctx, const jp_cellgrid* g, int nfields, double* const* F,
                           const double* const* Fp, const double* const* coords,
                           const uint8_t* index) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index) return fail(ctx, JP_ERR_ARG, "null index%s");
    if (nfields < 1 || nfields > JP_MAX_ARGS)
        return fail(ctx, JP_ERR_ARG, "nfields out of range%s");
    if ((rc = check_ptrs(ctx, nfields, (const void* const*)F, "F"))) return rc;
    if ((rc = check_ptrs(ctx, nfields, (const void* const*)Fp, "Fp"))) return rc;
    return g->ndim == 2 ? run_p2g<2>(ctx, g, nfields, F, Fp, coords, index, 1)
                        : run_p2g<3>(ctx, g, nfields, F, Fp, coords, index, 1);
}

int jp_grid2particle(jp_ctx* ctx, const jp_cellgrid* g, double* Fp, const double* F,
                     const double* const* coords, const uint8_t* index) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index || !F || !Fp) return fail(ctx, JP_ERR_ARG, "null field or index%s");
    return g->ndim == 2 ? run_g2p<2>(ctx, g, Fp, F, coords, index)
                        : run_g2p<3>(ctx, g, Fp, F, coords, index);
}

int jp_inject_particles(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords, uint8_t* index,
                        int nargs, double* const* args, int min_xcell, uint64_t seed,
                        uint64_t call_counter, jp_stats* stats) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index) return fail(ctx, JP_ERR_ARG, "null index%s");
    if (nargs < 0 || nargs > JP_MAX_ARGS) return fail(ctx, JP_ERR_ARG, "nargs out of range%s");
    if (nargs && (rc = check_ptrs(ctx, nargs, (const void* const*)args, "args"))) return rc;
    if (min_xcell < 0) return fail(ctx, JP_ERR_ARG, "min_xcell must be non-negative%s");
    return g->ndim == 2
               ? run_inject<2>(ctx, g, coords, index, nargs, args, min_xcell, seed, call_counter, stats)
               : run_inject<3>(ctx, g, coords, index, nargs, args, min_xcell, seed, call_counter, stats);
}

int jp_inject_particles_phase(jp_ctx* ctx, const jp_cellgrid* g, const jp_axis* xc,
                              double* const* coords, uint8_t* index, double* phases, int nargs,
                              double* const* args, const double* const* fields,
                              const int* centred, int min_xcell, uint64_t seed,
                              uint64_t call_counter, jp_stats* stats) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index || !phases || !xc) return fail(ctx, JP_ERR_ARG, "null index, phases or xc%s");
    if (nargs < 0 || nargs > JP_MAX_ARGS) return fail(ctx, JP_ERR_ARG, "nargs out of range%s");
    if (nargs && (rc = check_ptrs(ctx, nargs, (const void* const*)args, "args"))) return rc;
    if (nargs && (rc = check_ptrs(ctx, nargs, (const void* const*)fields, "fields"))) return rc;
    if (nargs && !centred) return fail(ctx, JP_ERR_ARG, "null centred flags%s");
    if (min_xcell < 0) return fail(ctx, JP_ERR_ARG, "min_xcell must be non-negative%s");
    uint32_t cmask = 0;
    bool any_centred = false;
    for (int a = 0; a < nargs; ++a)
        if (centred[a]) {
            cmask |= 1u << a;
            any_centred = true;
        }
    for (int d = 0; d < g->ndim; ++d) {
        if (any_centred && g->ni[d] < 2)
            return fail(ctx, JP_ERR_ARG, "a cell-centred field needs two cells per dimension%s");
        if (!xc[d].x || !xc[d].inv_dx || xc[d].n != g->ni[d])
            return fail(ctx, JP_ERR_ARG, "centre axis%s %lld must have ni points", "", d);
    }
    return g->ndim == 2
               ? run_inject_phase<2>(ctx, g, xc, coords, index, phases, nargs, args, fields, cmask,
                                     min_xcell, seed, call_counter, stats)
               : run_inject_phase<3>(ctx, g, xc, coords, index, phases, nargs, args, fields, cmask,
                                     min_xcell, seed, call_counter, stats);
}

}  // extern "C"
