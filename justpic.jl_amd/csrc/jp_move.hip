// jp_move.hip -- move_particles! (src/Particles/move_safe.jl:23-125) on gfx950.
//
// The reference visits cells in 3^D colour phases; inside a cell it walks the
// slots in order, and a particle that left its cell goes to the first free
// slot >= starting_point of its destination (starting_point shared by all
// destinations of one source cell).  The outcome depends only on which slots
// are occupied, so it is computed on 64-bit occupancy words and the particle
// data are moved afterwards in one parallel pass:
//
//   1. classify (one thread per cell, or per cell and chunk of 8 slots;
//      coalesced over the cell planes): in-cell test, domain test,
//      destination (bisection seeded at the cell) as a neighbour code,
//      occupancy/mover words, and a copy of every mover's coordinates and
//      fields into a staging area, packed per cell like the codes;
//   2. 3^D colour phases (one thread per source cell of the colour): the
//      reference's slot loop replayed on the free-slot words of the 3^D
//      neighbourhood (kept in LDS), recording for every slot that received a
//      particle where that particle came from;
//   3. scatter (threads as in classify): arrivals copy their staged data
//      into their final slot, vacated slots get NaN and mask false.
//
// A particle that jumps more than one cell breaks the colour independence;
// classify raises a flag (and records the largest jump), the regular phases
// return immediately, and a one-workgroup kernel runs the same slot loops on
// the same words, cell by cell in levels that keep the reference's order
// wherever two cells interact, finding the far destinations from the staged
// positions, and clears the flag; the scatter then moves the data as usual.
// The split classify raises another bit of the same flag when the grid's
// geometry was rejected: then nothing moves.
#include "jp_ctx.hpp"

#include <type_traits>

using namespace jp;

namespace {

// A mover's code is its destination cell in the 3^D neighbourhood: in 3D n =
// (dx+1) + 3 (dy+1) + 9 (dz+1), in 2D the same with the row pitch of the tiled
// phases' region (dx+1) + 42 (dy+1), so that a destination's word there is one
// addition away.  Codes without a bit of 0x80 below: the phases' fast loop
// takes them.  The centre's code fills the rows up to a multiple of 8.
constexpr uint8_t kRare = 0x80;  // re-slotted in its own cell (the centre's code), or an
                                 // arrival that fails the strict test of its destination
// a mover whose destination is found from its staged position when its cell
// is processed (far-jump path only: movers that jump more than one cell, and
// arrivals there that fail the strict test of their new cell)
constexpr uint8_t kFar = 0xFF;
constexpr int kFlagFar = 1;       // a mover jumps more than one cell
constexpr int kFlagRejected = 2;  // split geometry rejected
// s_waitcnt immediate of gfx9 for vmcnt(0) with expcnt and lgkmcnt left free
constexpr int kVmcnt0 = 0x0F70;

__device__ inline double dnan() { return __builtin_nan(""); }

struct MoveScratch {
    uint64_t* occ0;  // occupancy before the call
    uint64_t* occ;   // running occupancy
    uint64_t* mov;   // slots whose particle leaves or is re-slotted (classify)
    uint64_t* rar;   // 2D: rare movers (kRare), read by the tiled phases
    uint64_t* gap;   // rare movers, then also the slots whose arrival the cell re-slots (at
                     // the end: slots that an arrival was removed from, and some of occ0)
    uint8_t* code;   // the codes of the staged movers in slot order, 8 per word (word j*C + c)
    uint16_t* org;   // per slot: where an arrival came from (org_code; layout: org_at)
    uint32_t* orgf;  // far-jump path: the arrival's record (org: kOrgFar)
    char* stg;       // staged movers (layout: stg_coord; index: stage_index)
    uint64_t* stm;   // each cell's staged movers (bit k), written by classify
    int64_t S;       // slots
    int64_t stride;  // record bytes (multiple of 8)
    int64_t foff;    // byte offset of the fields in a record
};

// Slots of a cell that hold an arrival of this call.  A slot that was occupied
// before the call keeps its particle unless that particle is a mover, which
// leaves its slot when its own cell is processed: every other occupied slot
// holds an arrival, so no words are kept for arrivals.  (Before its cell is
// processed no mover has left: there the arrivals are occ & ~occ0.)
__device__ inline uint64_t arrivals(uint64_t occ, uint64_t occ0, uint64_t mov) {
    return occ & ~(occ0 & ~mov);
}

// Position of (cell, slot) in the origin array.  2D: plane-major like the
// particle data (c + C k).  3D: cell-major (c K + k): each mover of a colour
// phase stores one origin into a neighbour cell, and cell-major keeps a
// wavefront's stores inside the few lines of its cells' neighbourhoods
// (plane-major scatters them over an array as large as the last-level cache).
template <int D>
__device__ inline uint32_t org_at(uint32_t c, uint32_t k, uint32_t C, uint32_t K) {
    return D == 2 ? c + C * k : c * K + k;
}
// An arrival's origin is a neighbour of its cell: the code of its move and its
// rank among the source's staged movers fit 13 bits (half the bytes of a
// record number for the phases' scattered stores and the scatter's reads).
__device__ inline uint32_t org_code(uint32_t code, uint32_t rank) { return (code << 6) + rank; }
constexpr uint32_t kOrgFar = 0xFFFFu;  // the record is in orgf

template <int D>
constexpr int kNB = D == 2 ? 9 : 27;
template <int D>
constexpr int kCenter = (kNB<D> - 1) / 2;

constexpr int kPitch2 = 42;  // row length of the tiled 2D phases' region
// neighbour n (0..3^D-1) <-> code
template <int D>
__device__ inline uint32_t code_of(int n) {
    return D == 2 ? (uint32_t)(n + (kPitch2 - 3) * (n / 3)) : (uint32_t)n;
}
template <int D>
__device__ inline int neighbour_of(uint32_t cd) {
    return D == 2 ? (int)(cd - (kPitch2 - 3) * (cd / kPitch2)) : (int)cd;
}
// offset of a move's destination from its source, in cells (str: the strides
// of dimensions 1.. in cells)
template <int D>
__device__ inline int move_offset(uint32_t cd, int str1, int str2) {
    if (D == 2) {
        const int q = (int)(cd / kPitch2);
        return (int)cd - kPitch2 * q - 1 + str1 * (q - 1);
    }
    const int z = (int)(cd / 9), y = (int)(cd / 3) - 3 * z;
    return (int)cd - 3 * (int)(cd / 3) - 1 + str1 * (y - 1) + str2 * (z - 1);
}
template <int D>
constexpr uint32_t kHere = D == 2 ? kPitch2 + 1 : kCenter<3>;  // code of the cell itself

// colour phase of a cell: offsets (o_1 outer ... o_D inner), 0-based
template <int D>
__device__ inline int phase_of(const int64_t* I) {
    int ph = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) ph = ph * 3 + (int)(I[d] % 3);
    return ph;
}

// Staged coordinate d and field a of the mover from original slot o.  The
// scatter gathers movers by origin, one cache line per array touched, so the
// arrays are few.  2D: the D coordinates interleaved in one array, fields in
// planes (classify's stores stay contiguous across a wavefront's cells).  3D:
// one record per slot, the D coordinates then the fields (3D move -7% split,
// -20% FP64 against planes; full records were 3% slower in 2D).
// Staged movers: one record per mover (coordinates, then the fields at
// byte offset foff), the r-th staged mover of cell c (slot order) at record
// c K + r.  Packed per cell, a destination's arrivals from one origin cell
// share cache lines in the scatter's gathers, and classify writes only the
// movers' bytes (indexed by slot, every record was a cache line of its own
// and the staging writes touched every line of a slot-sized array).
// `below` is the cell's staged movers under the mover's slot.
template <int D>
__device__ inline int64_t stage_index(int64_t c, int K, uint64_t below) {
    return c * K + __popcll(below);
}
template <int D, typename T>
__device__ inline T& stg_coord(const MoveScratch& ms, int64_t o, int d) {
    return reinterpret_cast<T*>(ms.stg + o * ms.stride)[d];
}
template <int D>
__device__ inline double& stg_field(const MoveScratch& ms, int64_t o, int a) {
    return reinterpret_cast<double*>(ms.stg + o * ms.stride + ms.foff)[a];
}
// The 2D split record with one field is 16 bytes (two float offsets, the
// field): written and read with one 16-byte access each.
__device__ inline void stg_put16(const MoveScratch& ms, int64_t o, float u0, float u1, double f) {
    const uint64_t b = (uint64_t)__double_as_longlong(f);
    uint4 v;
    v.x = __float_as_uint(u0);
    v.y = __float_as_uint(u1);
    v.z = (uint32_t)b;
    v.w = (uint32_t)(b >> 32);
    *reinterpret_cast<uint4*>(ms.stg + o * 16) = v;
}
__device__ inline void stg_get16(const MoveScratch& ms, int64_t o, float& u0, float& u1,
                                 double& f) {
    const uint4 v = *reinterpret_cast<const uint4*>(ms.stg + o * 16);
    u0 = __uint_as_float(v.x);
    u1 = __uint_as_float(v.y);
    f = __longlong_as_double((long long)(((uint64_t)v.w << 32) | v.z));
}

// ------------------------------------------------------------ 1. classify
// Fields a0.. of the movers of one chunk of 8 slots, copied to the staging
// area in one batch of independent loads (stg: chunk-local mover bits).
// (o0: the record of the chunk's first staged mover)
template <int D>
__device__ inline void stage_args(int64_t c, int64_t C, int k0, uint32_t stg, int64_t o0,
                                  int nargs, const ArgPtrs& args, const MoveScratch& ms,
                                  int a0 = 0) {
    if (!stg) return;
    for (int a = a0; a < nargs; ++a) {
        const double* __restrict__ src = args.p[a];
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = ((stg >> j) & 1) ? src[c + C * (k0 + j)] : 0.0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if ((stg >> j) & 1) stg_field<D>(ms, o0 + __popc(stg & ((1u << j) - 1)), a) = v[j];
    }
}

// Classify's mapping.  CHUNKS (2D, and the 3D split form): a workgroup per
// 64 cells and one wavefront per 8-slot chunk (enough wavefronts to fill the
// chip at 512^2, loads coalesced along the slot planes, no chunk's loads
// behind an earlier chunk's stores); the chunk-threads of a cell add up
// their staged counts in LDS for the packed record index.  Otherwise (the
// 3D FP64 form, whose 200 registers per lane do not fit such workgroups
// well): one thread per cell, whole cells (chunks of 8 slot planes in
// lockstep across the wavefront).
constexpr int kClassifyMax = 512;  // 2D: 64 x up to 8 chunks
template <int D>
struct ClassifySlots {
    int64_t c;
    int kb, ke;
    bool live;
};
template <int D, bool CHUNKS>
__device__ inline ClassifySlots<D> classify_slots(const Grid<D>& g) {
    ClassifySlots<D> r;
    if constexpr (CHUNKS) {
        r.c = blockIdx.x * (int64_t)64 + (threadIdx.x & 63);
        r.kb = (int)(threadIdx.x >> 6) * 8;
        r.ke = r.kb + 8 < g.K ? r.kb + 8 : g.K;
        r.live = r.c < g.C;
    } else {
        r.c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
        r.kb = 0;
        r.ke = g.K;
        r.live = r.c < g.C;
    }
    return r;
}
// The per-cell words of classify.  CHUNKS: each chunk-thread puts its byte of
// every word into LDS; after the block's barrier the words are whole, give
// the chunk's record index (the cell's staged movers below it), and each
// wavefront stores some of them (8 bytes per lane, contiguous; stored byte by
// byte from the chunks the split classify took 84 us at 512^2, so 78).  Bytes
// above the last chunk are masked on reading.
enum { W_OCC = 0, W_MOV, W_STG, W_GAP, W_COUNT };
struct CellWords {
    uint64_t w[W_COUNT][64];
    __device__ inline void put(int t, uint32_t v) {
        reinterpret_cast<uint8_t*>(&w[t][threadIdx.x & 63])[threadIdx.x >> 6] = (uint8_t)v;
    }
    __device__ inline uint64_t get(int t) const {
        const int n = (int)(blockDim.x >> 6);
        return w[t][threadIdx.x & 63] & (n == 8 ? ~0ull : ((1ull << (8 * n)) - 1));
    }
};
// The codes of the staged movers, packed in slot order: a row of 68 bytes per
// cell in LDS (17 dwords: the lanes' rows start on different banks), filled
// with the centre's code first.
constexpr int kRow = 68;
template <int D>
__device__ inline void fill_codes(uint32_t* row, int from, int to) {  // bytes from..to-1
    for (int b = from >> 2; b < (to >> 2); ++b) row[b] = 0x01010101u * kHere<D>;
}
__device__ inline uint64_t code_word(const uint32_t* row, int j) {
    return (uint64_t)row[2 * j] | ((uint64_t)row[2 * j + 1] << 32);
}
template <int D>
__device__ inline void store_word(const MoveScratch& ms, int64_t c, int t, uint64_t v) {
    if (t == W_OCC) {
        ms.occ0[c] = v;
        ms.occ[c] = v;
    } else if (t == W_MOV) {
        ms.mov[c] = v;
    } else if (t == W_STG) {
        ms.stm[c] = v;
    } else {
        ms.gap[c] = v;
        if (D == 2) ms.rar[c] = v;
    }
}

// Destination codes are packed 8 per 64-bit word, word j of cell c at word
// index j*C + c (coalesced stores here), so the colour phases load a cell's
// codes in one round of word loads.
template <int D>
__global__ void __launch_bounds__(kClassifyMax) k_mv_classify(Grid<D> g, CPtr3 coords,
                                                              const uint8_t* __restrict__ index,
                                                              int nargs, ArgPtrs args,
                                                              MoveScratch ms, int* flag) {
    constexpr bool CH = D == 2;
    __shared__ CellWords s_w;
    __shared__ uint32_t s_code[(CH ? 64 : kBlock) * kRow / 4];
    const ClassifySlots<D> cs = classify_slots<D, CH>(g);
    if (!CH && !cs.live) return;  // (CH: every thread reaches the block's barrier)
    const int64_t c = cs.live ? cs.c : 0;
    const int kb = cs.kb, ke = cs.ke;  // slot chunk(s) kb..ke-1
    const int64_t C = g.C;
    int64_t I[D];
    unlin<D>(g.ni, c, I);
    // vertices x[I-1..I+2] and spacings dx[I-1..I+1] per dimension, loaded once:
    // the strict brackets of the three candidate cells are register compares
    // (a strictly interior point has a unique bracket, so this equals the
    // bisection seeded at the cell; ties and longer jumps take find_cell)
    double xa[D][4], hx[D][3], dlo[D], dhi[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const Axis& A = g.xv[d];
        const int64_t i = I[d], n = A.n;
        xa[d][0] = i > 0 ? A.x[i - 1] : -__builtin_inf();
        xa[d][1] = A.x[i];
        xa[d][2] = A.x[i + 1];
        xa[d][3] = i + 2 < n ? A.x[i + 2] : __builtin_inf();
        hx[d][0] = i > 0 ? A.dx[i - 1] : 0.0;
        hx[d][1] = A.dx[i];
        hx[d][2] = i + 1 < n - 1 ? A.dx[i + 1] : 0.0;
        dlo[d] = A.x[0];
        dhi[d] = A.x[n - 1];
    }
    const uint64_t occ = !cs.live ? 0ull
                         : (kb == 0 && ke == g.K) ? active_slots(index, c, C, g.K)
                                                  : active_slots_in(index, c, C, kb, ke);
    uint64_t mov = 0, staged = 0, rare = 0;
    uint64_t* __restrict__ cw = reinterpret_cast<uint64_t*>(ms.code) + c;
    uint32_t* row = s_code + (CH ? threadIdx.x & 63 : threadIdx.x) * (kRow / 4);
    uint8_t* const crow = reinterpret_cast<uint8_t*>(row);
    fill_codes<D>(row, kb, CH ? kb + 8 : 64);
    // chunks of slot planes walked in lockstep by the wavefront (coalesced
    // loads and stores across neighbouring cells)
    constexpr int B = 8;
    for (int k0 = kb; k0 < ke; k0 += B) {
        double pb[B][D];
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const bool on = (occ >> (k0 + j)) & 1;
#pragma unroll
            for (int d = 0; d < D; ++d) pb[j][d] = on ? coords.p[d][c + C * (k0 + j)] : 0.0;
        }
        uint32_t cd8[2] = {0, 0};  // the chunk's codes, by slot
        uint32_t mv8 = 0, stg = 0, rr8 = 0;
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const int k = k0 + j;
            if (!((occ >> k) & 1)) continue;
            double p[D];
#pragma unroll
            for (int d = 0; d < D; ++d) p[d] = pb[j][d];
            bool inc = true, indom = true;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                inc = inc & (xa[d][1] < p[d] && p[d] < xa[d][1] + hx[d][1]);  // isincell
                indom = indom & (dlo[d] < p[d] && p[d] < dhi[d]);  // indomain
            }
            if (inc) continue;
            mv8 |= 1u << j;
            if (indom) {  // (else deleted: empty_particle! only)
                uint32_t cd;
                int n = 0, mult = 1;
                bool far = false, inJ = true;
                int64_t jump = 0;  // cells jumped (largest over the dimensions)
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    int r;
                    if (xa[d][0] < p[d] && p[d] < xa[d][1]) r = -1;
                    else if (xa[d][1] < p[d] && p[d] < xa[d][2]) r = 0;
                    else if (xa[d][2] < p[d] && p[d] < xa[d][3]) r = 1;
                    else {
                        const int64_t t = find_cell(p[d], g.xv[d], I[d]) - I[d];
                        r = t < -1 ? -2 : (t > 1 ? 2 : (int)t);
                        jump = t < -jump ? -t : (t > jump ? t : jump);
                    }
                    far = far || r < -1 || r > 1;
                    n += (r + 1) * mult;
                    mult *= 3;
                    const double lo = r < 0 ? xa[d][0] : (r == 0 ? xa[d][1] : xa[d][2]);
                    const double h = r < 0 ? hx[d][0] : (r == 0 ? hx[d][1] : hx[d][2]);
                    inJ = inJ & (lo < p[d] && p[d] < lo + h);
                }
                if (far) {  // the far-jump path finds the destination again
                    atomicOr(flag, kFlagFar);
                    atomicMax(flag + 1, (int)(jump < (1 << 30) ? jump : (1 << 30)));
                    cd = kFar;
                } else {
                    const bool rr = n == kCenter<D> || !inJ;
                    cd = code_of<D>(n) | (rr ? kRare : 0u);
                    rr8 |= (uint32_t)rr << j;
                }
                stg |= 1u << j;
                cd8[j >> 2] |= cd << (8 * (j & 3));
            }
        }
        mov |= (uint64_t)mv8 << k0;
        rare |= (uint64_t)rr8 << k0;
        // the chunk's staged movers, packed after the cell's earlier ones
        if constexpr (CH) {  // (one chunk per thread)
            s_w.put(W_OCC, (uint32_t)(occ >> k0));
            s_w.put(W_MOV, mv8);
            s_w.put(W_STG, stg);
            s_w.put(W_GAP, rr8);
            __syncthreads();
            staged = s_w.get(W_STG) & ((1ull << k0) - 1);
        }
        const int r0 = __popcll(staged);
#pragma unroll
        for (int j = 0; j < B; ++j)
            if ((stg >> j) & 1)
                crow[r0 + __popc(stg & ((1u << j) - 1))] = (uint8_t)(cd8[j >> 2] >> (8 * (j & 3)));
        const int64_t o0 = c * g.K + r0;
        if constexpr (CH) {
            __syncthreads();
            if (cs.live) {
                // (one code word per chunk-thread)
                if (__popcll(s_w.get(W_STG)) > kb) cw[(kb >> 3) * C] = code_word(row, kb >> 3);
                for (int t = (int)(threadIdx.x >> 6); t < W_COUNT; t += (int)(blockDim.x >> 6))
                    store_word<D>(ms, c, t, s_w.get(t));
            }
        }
        if (cs.live) {
#pragma unroll
            for (int j = 0; j < B; ++j)
                if ((stg >> j) & 1) {
                    const int64_t o = o0 + __popc(stg & ((1u << j) - 1));
#pragma unroll
                    for (int d = 0; d < D; ++d) stg_coord<D, double>(ms, o, d) = pb[j][d];
                }
            stage_args<D>(c, C, k0, stg, o0, nargs, args, ms);
        }
        staged |= (uint64_t)stg << k0;
    }
    if constexpr (!CH) {
        store_word<D>(ms, c, W_OCC, occ);
        store_word<D>(ms, c, W_MOV, mov);
        store_word<D>(ms, c, W_STG, staged);
        store_word<D>(ms, c, W_GAP, rare);
        for (int j = 0; 8 * j < __popcll(staged); ++j) cw[j * C] = code_word(row, j);
    }
}

// ------------------------------------------------------------ 2. colour phases
template <int D>
__device__ inline int64_t nb_cell(const Grid<D>& g, const int64_t* I, int n, bool& ok) {
    int64_t J[D];
    ok = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        J[d] = I[d] + (n % 3) - 1;
        n /= 3;
        ok = ok && J[d] >= 0 && J[d] < g.ni[d];
    }
    return ok ? lin<D>(g.ni, J) : -1;
}

// A cell of the 3^D neighbourhood in LDS: its free slots (0 outside the grid
// and, while a cell's movers are dealt out, for the cell itself) and its number.
constexpr uint32_t kNoCell = 0xFFFFFFFFu;
struct alignas(16) NbEntry {
    uint64_t free;
    uint32_t cell;  // kNoCell: arrivals there are not recorded (outside the grid; another tile's)
    uint32_t pad;
};

// The reference slot loop of a cell without rare movers: the n staged movers in
// slot order, each to the first free slot >= starting_point of its
// destination, which becomes starting_point.
//
// The loop is one serial chain per thread, on one or two wavefronts per SIMD,
// and a phase lasts as long as its longest chain, so what counts is the
// instructions per mover.  The codes come packed (no search for the next
// mover), a dword of four at a time; a destination's entry is one LDS read,
// issued a mover ahead (the previous mover's result is forwarded when both go
// to the same cell); the chain itself is a few operations on masks (mask with
// the slots >= starting_point, isolate the lowest bit, negate it for the next
// mask).  Rows end with codes of the cell itself, whose entry has no free slot
// meanwhile: no test for the last mover, and none for a full destination but
// the one that guards the store.  Nothing else is kept per mover (arrivals
// follow from the occupancy words at the end): ~32 instructions a mover.  A
// loop over the mover bits with two dependent LDS reads, arrival words updated
// per mover and an origin stored for every processing took 105 us for the
// tiled 2D phases at 512^2 (32^2: 87, 3D 128^3: 30.9 per phase), this one 51
// (38; 3D 22.6, 4 of it by loading the neighbours' words in one round).  Of
// that, origins stored for the tile's own cells only: 74 -> 58, in 16 bits:
// 58 -> 51 (scattered stores, each a cache line).
//
// at(code): the entry of a code's destination.
template <int D, bool STATS, typename At>
__device__ inline void run_movers(int n, const uint32_t* row, const At& at,
                                  uint16_t* __restrict__ org, uint32_t C32, uint32_t K,
                                  int& n_moved) {
    uint64_t ge = ~0ull;  // slots >= starting_point
    uint32_t cw = row[0], cd = cw & 0xFFu;
    NbEntry* to = &at(cd);
    NbEntry* last = to;
    uint64_t word = to->free, put = word;
    uint32_t cell = to->cell;
    for (int i = 0; i < n; i += 4) {
        const uint32_t cnext = i + 4 < n ? row[(i >> 2) + 1] : 0x01010101u * kHere<D>;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t cd1 = j < 3 ? (cw >> (8 * (j + 1))) & 0xFFu : cnext & 0xFFu;
            NbEntry* const to1 = &at(cd1);
            const uint64_t word1 = to1->free;
            const uint32_t cell1 = to1->cell;
            const uint64_t fw = to == last ? put : word;
            const uint64_t fr = fw & ge;
            const uint64_t fb = fr & (0 - fr);
            put = fw ^ fb;
            last = to;
            to->free = put;
            const bool got = fr != 0;  // else find_free_memory found nothing: dropped
            ge = got ? 0 - fb : ge;    // starting_point = free_idx
            if (got & (cell != kNoCell))
                org[org_at<D>(cell, (uint32_t)__builtin_ctzll(fb), C32, K)] =
                    (uint16_t)org_code(cd, (uint32_t)(i + j));
            if (STATS) n_moved += got;
            to = to1;
            word = word1;
            cell = cell1;
            cd = cd1;
        }
        cw = cnext;
    }
}

// The same for a cell with rare movers (one re-slotted in its own cell, one
// that its destination will re-slot, an arrival of this call that failed the
// strict test of this cell), every case handled.  `pend`: slots to visit, on
// return the visited ones (re-slotted particles met again included); returns
// the cell's free slots.  later(code, entry, bit): the destination re-slots the
// arrival when its phase comes later.
template <int D, bool STATS, typename At, typename Later>
__device__ inline uint64_t run_rare(uint64_t& pend, uint64_t mov, uint64_t stm,
                                          uint64_t free, const uint8_t* codes, const At& at,
                                          const Later& later, uint16_t* org, uint32_t S32,
                                          uint32_t C32, uint32_t K, int& n_moved, int& n_drop) {
    uint64_t ge = ~0ull, left = pend, again = 0;
    while (left) {
        const int ip = __builtin_ctzll(left);
        const uint64_t bit = 1ull << ip;
        left &= left - 1;
        free |= bit;  // empty_particle! on the source slot
        uint32_t cd = kHere<D>, origin;
        if (!(mov & bit)) {  // an arrival (of another cell, or re-slotted here): stays here
            origin = org[org_at<D>(S32, (uint32_t)ip, C32, K)];
        } else if (stm & bit) {
            const int r = __popcll(stm & (bit - 1));
            cd = codes[r];
            origin = org_code(cd & 0x7Fu, (uint32_t)r);
        } else {
            continue;  // deleted
        }
        const uint32_t n = cd & 0x7Fu;
        const bool here = n == kHere<D>;
        NbEntry& to = at(n);
        const uint64_t fw = here ? free : to.free, fr = fw & ge;
        if (!fr) {  // find_free_memory found nothing
            if (STATS) ++n_drop;
            continue;
        }
        const uint64_t fb = fr & (0 - fr);
        const int f = __builtin_ctzll(fb);
        ge = 0 - fb;
        if (STATS) ++n_moved;
        if (to.cell != kNoCell)
            org[org_at<D>(to.cell, (uint32_t)f, C32, K)] = (uint16_t)origin;
        if (here) {
            free ^= fb;
            if (f > ip) {  // the slot loop reaches it again
                left |= fb;
                again |= fb;
            }
        } else {
            to.free = fw ^ fb;
            if (cd & kRare) later(n, to, fb);
        }
    }
    pend |= again;
    return free;
}

// One cell of a phase.  free: its free slots; gap: its word of rare movers and
// arrivals to re-slot, on return with the slots re-slotted here added.  Returns
// the free slots after it.
template <int D, bool STATS, typename At, typename Later>
__device__ inline uint64_t run_cell(uint64_t mov, uint64_t stm, uint64_t& gap, uint64_t free,
                                    const uint32_t* row, const At& at, const Later& later,
                                    uint16_t* __restrict__ org, uint32_t S32, uint32_t C32,
                                    uint32_t K, int& n_moved, int& n_del, int& n_drop) {
    if (STATS) n_del += __popcll(mov & ~stm);
    NbEntry& own = at(kHere<D>);
    uint64_t after;
    if (gap) {
        uint64_t pend = mov | gap;
        after = run_rare<D, STATS>(pend, mov, stm, free, reinterpret_cast<const uint8_t*>(row),
                                   at, later, org, S32, C32, K, n_moved, n_drop);
        gap |= pend & ~mov;
    } else {
        own.free = 0;
        int moved = 0;
        const int n = __popcll(stm);
        if (n) run_movers<D, STATS>(n, row, at, org, C32, K, moved);
        after = free | mov;
        if (STATS) {
            n_moved += moved;
            n_drop += n - moved;
        }
    }
    own.free = after;
    return after;
}

__device__ inline void put_codes(uint32_t* row, const uint64_t (&w)[8], int nw) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (j < nw) {
            row[2 * j] = (uint32_t)w[j];
            row[2 * j + 1] = (uint32_t)(w[j] >> 32);
        }
}
__device__ inline void load_codes(const MoveScratch& ms, uint32_t S32, uint32_t C32, int nw,
                                  uint64_t (&w)[8]) {
    const uint64_t* __restrict__ cp = reinterpret_cast<const uint64_t*>(ms.code) + S32;
#pragma unroll
    for (int j = 0; j < 8; ++j) w[j] = j < nw ? cp[(int64_t)j * C32] : 0ull;
}

// one colour phase, one thread per colour cell; the neighbourhood's entries in
// a column of LDS per thread
template <int D, int BS, bool STATS>
__global__ void __launch_bounds__(BS) k_mv_phase(Grid<D> g, MoveScratch ms, Off3 off, int phase,
                                                 const int* __restrict__ flag, jp_stats* st) {
    __shared__ NbEntry s_nb[kNB<D>][BS];
    __shared__ uint32_t s_code[BS * kRow / 4];
    const int stop = *flag;  // far-jump path, or rejected grid: nothing moves here
    int n_moved = 0, n_del = 0, n_drop = 0;
    // (a phase has fewer than 2^31 cells: 32-bit divisions)
    uint32_t t = blockIdx.x * BS + threadIdx.x, ncol[D];
    int I[D];
    bool ok = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        ncol[d] = ((uint32_t)g.ni[d] + 2) / 3;
        const uint32_t q = d < D - 1 ? t / ncol[d] : 0;
        I[d] = 3 * (int)(t - q * ncol[d]) + off.o[d];
        ok = ok && I[d] < (int)g.ni[d];
        t = q;
    }
    if (ok) {
        // everything the cell needs, in one round of independent loads (cells
        // of one colour are 3 apart: no other thread of this phase touches
        // these neighbourhood words).  Unguarded: a neighbour outside the grid
        // loads the cell's own word, since guarded loads are waited for one by
        // one (27 round trips: a move of 30^3 cells without movers took 164 us, now 112)
        uint32_t str[D], S32 = 0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            str[d] = d == 0 ? 1u : str[d - 1] * (uint32_t)g.ni[d - 1];
            S32 += (uint32_t)I[d] * str[d];
        }
        const int tid = threadIdx.x;
        const uint32_t K = (uint32_t)g.K, C32 = (uint32_t)g.C;
        const uint64_t full = K == 64 ? ~0ull : ((1ull << K) - 1);
        const uint64_t mov = ms.mov[S32], stm = ms.stm[S32];
        uint64_t gap = ms.gap[S32];
        const int nw = ((int)K + 7) >> 3;
        uint64_t cw[8], word[kNB<D>];
        uint32_t cell[kNB<D>], in = 0;
        load_codes(ms, S32, C32, nw, cw);
#pragma unroll
        for (int n = 0; n < kNB<D>; ++n) {
            bool v = true;
            uint32_t c = S32;
            int r = n;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int o = r % 3 - 1;
                r /= 3;
                v = v && I[d] + o >= 0 && I[d] + o < (int)g.ni[d];
                c += (uint32_t)(o * (int)str[d]);
            }
            cell[n] = v ? c : S32;
            word[n] = ms.occ[cell[n]];
            in |= (uint32_t)v << n;
        }
        if (!stop && (mov | gap)) {
#pragma unroll
            for (int n = 0; n < kNB<D>; ++n)
                s_nb[n][tid] = NbEntry{(in >> n) & 1 ? ~word[n] & full : 0ull, cell[n], 0u};
            uint32_t* const row = s_code + tid * (kRow / 4);
            put_codes(row, cw, nw);
            const uint64_t gap0 = gap;
            auto at = [&](uint32_t cd) -> NbEntry& {
                return s_nb[D == 2 ? neighbour_of<D>(cd) : (int)cd][tid];
            };
            auto later = [&](uint32_t, NbEntry& to, uint64_t fb) {
                int64_t J[D];
                unlin<D>(g.ni, (int64_t)to.cell, J);
                if (phase_of<D>(J) > phase) ms.gap[to.cell] |= fb;
            };
            run_cell<D, STATS>(mov, stm, gap, s_nb[kCenter<D>][tid].free, row, at, later, ms.org,
                               S32, C32, K, n_moved, n_del, n_drop);
            // all words of the neighbourhood (unchanged ones too: comparing
            // would hold the old words in registers)
#pragma unroll
            for (int n = 0; n < kNB<D>; ++n)
                if ((in >> n) & 1) {
                    const NbEntry e = s_nb[n][tid];
                    ms.occ[e.cell] = ~e.free & full;
                }
            if (gap != gap0) ms.gap[S32] = gap;
        }
    }
    if (STATS) {
        stat_add(st, ST_MOVED, n_moved);
        stat_add(st, ST_DELETED, n_del);
        stat_add(st, ST_DROPPED, n_drop);
    }
}

// ------------------------------------------------------------ far jumps
// The colour phases when some particle jumps more than one cell (flag[0] has
// kFlagFar, flag[1] holds the largest jump R in cells), in one workgroup on
// the same words, codes and staged data as the regular phases; the scatter
// then moves the data as usual.  A cell's processing touches only cells
// within R of it, so two cells of one colour phase (3t + o) interact only
// when their colour coordinates t differ by at most q = floor(2R/3) in every
// dimension.  Within a phase the reference visits the cells in linear order
// of t; here they go in levels L(t) = sum_d m_d t_d with m_0 = 1 and
// m_d = 1 + sum_{e<d} m_e q_e (q_e = q capped at the colour count - 1): any
// two interacting cells have their linear order as level order, and cells of
// one level do not interact, so each level runs in parallel between
// barriers and the result is the reference's.  With a small R that is
// 3^D * (about (1 + m_1 + m_2) * the colour count per dimension) levels; a
// jump of the grid's size makes every level one cell (the serial order).
constexpr int kFarBlock = 256;

template <int D>
__device__ inline void far_origin(const MoveScratch& ms, uint32_t c, uint32_t k, uint32_t C,
                                  uint32_t K, uint32_t record) {
    const uint32_t at = org_at<D>(c, k, C, K);
    ms.orgf[at] = record;
    ms.org[at] = (uint16_t)kOrgFar;
}

// The reference slot loop of cell I in phase `phase` on the far-jump path
// (cells in an order that keeps apart any two that interact): kFar codes are
// resolved here from the staged positions, and a destination beyond the 3^D
// neighbourhood is updated in the global words directly.
template <int D, int BS, typename T>
__device__ inline void far_cell(const Grid<D>& g, const MoveScratch& ms, const int64_t* I,
                                int phase, NbEntry (&s_nb)[kNB<D>][BS],
                                uint32_t (&s_code)[BS * kRow / 4], int& n_moved, int& n_del,
                                int& n_drop, int& n_far) {
    const int64_t S = lin<D>(g.ni, I);
    const int tid = threadIdx.x;
    const int K = g.K;
    const int64_t C = g.C;
    const uint32_t S32 = (uint32_t)S, C32 = (uint32_t)C;
    const uint64_t full = K == 64 ? ~0ull : ((1ull << K) - 1);
    // everything this cell needs, in one round of independent loads: its
    // words, its code words and the occupancy words of its 3^D neighbourhood
    const uint64_t gapS = ms.gap[S];
    uint64_t pend = ms.mov[S] | gapS;
    const uint64_t pend0 = pend, occ0S = ms.occ0[S];
    const uint64_t stmS = ms.stm[S];  // staged movers (their record index)
    uint64_t cw[8];
    load_codes(ms, S32, C32, (K + 7) >> 3, cw);
    int64_t nbc[kNB<D>];
    uint64_t was[kNB<D>];
#pragma unroll
    for (int n = 0; n < kNB<D>; ++n) {
        bool v;
        nbc[n] = nb_cell<D>(g, I, n, v);
        was[n] = ms.occ[v ? nbc[n] : S];  // (unguarded: see k_mv_phase)
    }
    if (!pend) return;  // nothing leaves or re-slots here
#pragma unroll
    for (int n = 0; n < kNB<D>; ++n)
        s_nb[n][tid] = NbEntry{nbc[n] < 0 ? 0ull : ~was[n] & full,  // outside the grid: never free
                               nbc[n] < 0 ? kNoCell : (uint32_t)nbc[n], 0u};
    uint32_t* const row = s_code + tid * (kRow / 4);
    put_codes(row, cw, (K + 7) >> 3);
    uint64_t occC = was[kCenter<D>];  // this cell's occupancy
    uint64_t arrS = occC & ~occ0S;  // slots holding an arrival
    uint64_t selfm = 0;  // slots that received a re-slotted particle of this cell
    uint64_t again = 0;  // those the loop reaches (pending from then on)
    int sp = 0;
    while (pend) {
        const int ip = __builtin_ctzll(pend);
        pend &= pend - 1;
        const uint64_t bit = 1ull << ip;
        // a mover of this cell: its staged record and code; an arrival: the
        // record its origin staged, and (unless it was re-slotted here) the
        // destination from its position
        const bool arrival = (arrS & bit) != 0;
        const int rank = __popcll(stmS & (bit - 1));
        uint32_t origin = S32 * (uint32_t)K + (uint32_t)rank;
        uint32_t cd = kFar;
        if (arrival) {
            origin = ms.orgf[org_at<D>(S32, (uint32_t)ip, C32, (uint32_t)K)];
            // waited for here, on the rare path: otherwise every round of the loop
            // waits for it, and with it (one counter for loads and stores) for the
            // stores of the round before (split, 64^3 cells, CFL 2.5: 195 ms a move, now 187)
            __builtin_amdgcn_s_waitcnt(kVmcnt0);
        } else if (stmS & bit)
            cd = reinterpret_cast<const uint8_t*>(row)[rank];
        if (selfm & bit) cd = kHere<D>;
        occC &= ~bit;  // empty_particle! on the source slot
        arrS &= ~bit;
        selfm &= ~bit;
        if (!arrival && !(stmS & bit)) {
            ++n_del;
            continue;
        }
        if (cd == kFar) {
            // the destination from the staged position: bisection seeded
            // at this cell (FP64), the cell + floor(u) (split, whose staged
            // offset is renormalised to it here, for the scatter)
            int64_t J[D];
            bool near = true, inJ = true;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const T q = stg_coord<D, T>(ms, origin, d);
                if constexpr (std::is_same<T, float>::value) {
                    const int sd = (int)floorf(q);
                    J[d] = I[d] + sd;
                    stg_coord<D, T>(ms, origin, d) = (float)((double)q - (double)sd);
                } else {
                    J[d] = find_cell(q, g.xv[d], I[d]);
                    const double xl = g.xv[d].x[J[d]];
                    inJ = inJ && xl < q && q < xl + g.xv[d].dx[J[d]];
                }
                near = near && J[d] - I[d] <= 1 && I[d] - J[d] <= 1;
            }
            if (near) {  // inside the neighbourhood: the usual path
                int nn = 0, mult = 1;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    nn += (int)(J[d] - I[d] + 1) * mult;
                    mult *= 3;
                }
                cd = code_of<D>(nn);
                if (nn != kCenter<D> && !inJ) cd |= kRare;
            } else {
                ++n_far;
                const int64_t dcn = lin<D>(g.ni, J);
                const uint64_t od = ms.occ[dcn];
                const uint64_t fr = ~od & full & (~0ull << sp);
                if (!fr) {
                    ++n_drop;
                    continue;
                }
                const int f = __builtin_ctzll(fr);
                sp = f;
                const uint64_t fb = 1ull << f;
                ++n_moved;
                far_origin<D>(ms, (uint32_t)dcn, (uint32_t)f, C32, (uint32_t)K, origin);
                ms.occ[dcn] = od | fb;
                // an arrival that fails the strict test of its new cell is
                // looked up again when that cell comes later: in a later
                // phase, or later in this one (a jump by a multiple of 3
                // cells keeps the colour; cells of a phase go in linear
                // order)
                const int pj = phase_of<D>(J);
                if (!inJ && (pj > phase || (pj == phase && dcn > S)))
                    atomicOr(reinterpret_cast<unsigned long long*>(ms.gap + dcn),
                             (unsigned long long)fb);
                continue;
            }
        }
        const int n = neighbour_of<D>(cd & 0x7Fu);
        const NbEntry nb = s_nb[n][tid];
        const uint32_t dcn = nb.cell;
        const uint64_t fr = (n == kCenter<D> ? ~occC & full : nb.free) & (~0ull << sp);
        if (!fr) {  // find_free_memory found nothing: dropped
            ++n_drop;
            continue;
        }
        const int f = __builtin_ctzll(fr);
        sp = f;  // starting_point = free_idx
        const uint64_t fb = 1ull << f;
        s_nb[n][tid].free = nb.free & ~fb;  // (the centre's LDS copy is not read)
        ++n_moved;
        far_origin<D>(ms, dcn, (uint32_t)f, C32, (uint32_t)K, origin);
        if (n == kCenter<D>) {
            occC |= fb;
            arrS |= fb;
            if (f > ip) {  // the slot loop will reach this particle again
                pend |= fb;
                selfm |= fb;
                again |= fb;
            }
        } else if (cd & kRare) {
            // the arrival fails the strict test of its new cell: when that cell's
            // phase comes later, it is re-slotted there (bisection returns that cell)
            const int64_t Dc = dcn;
            int64_t J[D];
            unlin<D>(g.ni, Dc, J);
            if (phase_of<D>(J) > phase) {
                // (its destination is looked up again, as the reference does)
                ms.gap[Dc] |= fb;
            }
        }
    }
#pragma unroll
    for (int n = 0; n < kNB<D>; ++n) {
        if (n == kCenter<D>) continue;
        const NbEntry nb = s_nb[n][tid];
        const uint32_t dn = nb.cell;
        if (dn == 0xFFFFFFFFu) continue;
        const uint64_t now = ~nb.free & full;
        if (now != was[n]) ms.occ[dn] = now;
    }
    ms.occ[S] = occC;
    if (again & ~pend0) ms.gap[S] = gapS | again;
}

// (R: the largest jump; called by the whole workgroup of kFarBlock threads)
template <int D, typename T>
__device__ inline void far_phases(const Grid<D>& g, const MoveScratch& ms, int R,
                                  NbEntry (&s_nb)[kNB<D>][kFarBlock],
                                  uint32_t (&s_code)[kFarBlock * kRow / 4], jp_stats* st) {
    int64_t ncol[D], m[D];
#pragma unroll
    for (int d = 0; d < D; ++d) ncol[d] = (g.ni[d] + 2) / 3;
    const int64_t q = (2 * (int64_t)R) / 3;
    int64_t lmax = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        m[d] = 1;
        for (int e = 0; e < d; ++e) m[d] += m[e] * (q < ncol[e] - 1 ? q : ncol[e] - 1);
        lmax += m[d] * (ncol[d] - 1);
    }
    // the (t_1, ..., t_{D-1}) combinations, one per thread and round
    int64_t outer = 1;
#pragma unroll
    for (int d = 1; d < D; ++d) outer *= ncol[d];
    int n_moved = 0, n_del = 0, n_drop = 0, n_far = 0;
    for (int ph = 0; ph < kNB<D>; ++ph) {
        int o[D];
        int rr = ph;
#pragma unroll
        for (int d = D - 1; d >= 0; --d) {
            o[d] = rr % 3;
            rr /= 3;
        }
        for (int64_t lv = 0; lv <= lmax; ++lv) {
            for (int64_t i = threadIdx.x; i < outer; i += kFarBlock) {
                int64_t t[D], rest = i, l0 = lv;
#pragma unroll
                for (int d = 1; d < D; ++d) {
                    t[d] = rest % ncol[d];
                    rest /= ncol[d];
                    l0 -= m[d] * t[d];
                }
                t[0] = l0;
                if (t[0] < 0 || t[0] >= ncol[0]) continue;
                int64_t I[D];
                bool ok = true;
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    I[d] = 3 * t[d] + o[d];
                    ok = ok && I[d] < g.ni[d];
                }
                if (ok)
                    far_cell<D, kFarBlock, T>(g, ms, I, ph, s_nb, s_code, n_moved, n_del,
                                              n_drop, n_far);
            }
            __syncthreads();
        }
    }
    stat_add(st, ST_MOVED, n_moved);
    stat_add(st, ST_DELETED, n_del);
    stat_add(st, ST_DROPPED, n_drop);
    stat_add(st, ST_FAR, n_far);
}

template <int D, typename T>
__global__ void __launch_bounds__(kFarBlock) k_mv_far(Grid<D> g, MoveScratch ms,
                                                      const int* __restrict__ flag,
                                                      jp_stats* st) {
    __shared__ NbEntry s_nb[kNB<D>][kFarBlock];
    __shared__ uint32_t s_code[kFarBlock * kRow / 4];
    const int fl = flag[0];
    if (!(fl & kFlagFar) || (fl & kFlagRejected)) return;
    far_phases<D, T>(g, ms, flag[1], s_nb, s_code, st);
}

// ------------------------------------------------------------ 2'. 2D phases in tiles
// All nine colour phases of the 2D move in one launch.  A workgroup owns a
// tile of cells and replays the phases on the occupancy, pending, arrival and
// touched words of the tile plus a halo, all in LDS, with a barrier between
// phases; it keeps the results of its own cells.
//
// The halo is the dependency cone of the phases.  The processing of cell A in
// phase p reads and writes the words of A's 3x3 neighbourhood, so it depends
// on the processings, in earlier phases, of the cells B within 2 of A (their
// neighbourhoods overlap A's), and on theirs in turn.  A step from A to B
// moves, per dimension, by a multiple of 3 plus the difference of their
// colours, within [-2, 2]; taking the phases down from p, the offsets that can
// be reached lie in lo_p..hi_p with, for phase p = 3 c0 + c1 (c0 = I0 mod 3,
// the outer digit of the phase, c1 = I1 mod 3):
//   dimension 0: -c0 .. 2 c0,  dimension 1: -p .. 2 p.
// A processing is exact here when A + [lo_p - 1, hi_p + 1] lies inside the
// region (or leaves the grid there), and a processing that changes an exact
// one is itself exact, so only those run.  The final words of an owned cell
// come from the processings of its 3x3 neighbourhood, so the region is the
// tile widened by the largest cone plus 2: 4 cells below and 6 above in
// dimension 0, 10 below and 18 above in dimension 1.
//
// Tiles overlap, so a halo processing also runs in the tile that owns it;
// both compute the same slots from the same exact inputs.  Origins, counts and
// final words come from owned cells only.  (An arrival that is re-slotted has
// its origin read again, but stays in its cell: in a cell of another tile
// neither the read nor the store matters.)
//
// A pending slot that holds an arrival of this call is always re-slotted in
// its own cell (an arrival that fails the strict test of its new cell, or a
// particle re-slotted higher in its own cell), so the destination code of
// such a slot is the centre and the code words are read-only here.
constexpr int kTileHalo0Lo = 4, kTileHalo0Hi = 6, kTileHalo1Lo = 10, kTileHalo1Hi = 18;

__device__ inline int cone_lo(int p, int d) { return d == 0 ? -(p / 3) : -p; }
__device__ inline int cone_hi(int p, int d) { return d == 0 ? 2 * (p / 3) : 2 * p; }

// With a far jump one workgroup takes the far-jump path instead (a launch of its own
// for it, which nearly always returned at once, took 4.5 us of every move).
template <int TX, int TY, int BS, bool STATS, typename T>
__global__ void __launch_bounds__(BS) k_mv_tiles2(Grid<2> g, MoveScratch ms,
                                                  const int* __restrict__ flag, jp_stats* st) {
    constexpr int RX = TX + kTileHalo0Lo + kTileHalo0Hi;
    constexpr int RY = TY + kTileHalo1Lo + kTileHalo1Hi;
    constexpr int R = RX * RY;
    static_assert(((RX + 2) / 3) * ((RY + 2) / 3) <= BS, "one cell per thread and phase");
    static_assert(RX == kPitch2, "the codes' row pitch");
    static_assert(BS == kFarBlock, "the far-jump path's workgroup");
    union Entries {  // of the region, or of the far-jump path's cells
        struct {
            NbEntry nb[R];
            uint64_t gap[R];
        } tile;
        NbEntry far[kNB<2>][kFarBlock];
    };
    __shared__ __attribute__((aligned(16))) char s_raw[sizeof(Entries)];
    __shared__ uint32_t s_code[BS * kRow / 4];
    Entries& s_e = *reinterpret_cast<Entries*>(s_raw);
    if (*flag) {  // far jump or rejected grid
        if (blockIdx.x == 0 && (flag[0] & kFlagFar) && !(flag[0] & kFlagRejected))
            far_phases<2, T>(g, ms, flag[1], s_e.far, s_code, st);
        return;
    }
    NbEntry(&s_nb)[R] = s_e.tile.nb;
    uint64_t(&s_gap)[R] = s_e.tile.gap;
    const int n0 = (int)g.ni[0], n1 = (int)g.ni[1];
    const int ntx = (n0 + TX - 1) / TX;
    // neighbouring tiles read each other's halo words: consecutive tiles of
    // a row on one XCD
    const int tile = (int)xcd_block(blockIdx.x, gridDim.x);
    const int tx0 = (tile % ntx) * TX, ty0 = (tile / ntx) * TY;
    const int tx1 = (tx0 + TX < n0 ? tx0 + TX : n0) - 1;
    const int ty1 = (ty0 + TY < n1 ? ty0 + TY : n1) - 1;
    const int gx0 = tx0 - kTileHalo0Lo > 0 ? tx0 - kTileHalo0Lo : 0;
    const int gx1 = tx1 + kTileHalo0Hi < n0 - 1 ? tx1 + kTileHalo0Hi : n0 - 1;
    const int gy0 = ty0 - kTileHalo1Lo > 0 ? ty0 - kTileHalo1Lo : 0;
    const int gy1 = ty1 + kTileHalo1Hi < n1 - 1 ? ty1 + kTileHalo1Hi : n1 - 1;
    const int rw = gx1 - gx0 + 1, rh = gy1 - gy0 + 1;
    const uint32_t K = (uint32_t)g.K;
    const uint32_t C32 = (uint32_t)g.C;
    const uint64_t full = K == 64 ? ~0ull : ((1ull << K) - 1);
    for (int i = threadIdx.x; i < rw * rh; i += BS) {
        const int x = i % rw, y = i / rw;
        const uint32_t c = (uint32_t)(gx0 + x) + (uint32_t)n0 * (uint32_t)(gy0 + y);
        const int r = x + RX * y;
        const bool own = tx0 <= gx0 + x && gx0 + x <= tx1 && ty0 <= gy0 + y && gy0 + y <= ty1;
        s_nb[r] = NbEntry{~ms.occ0[c] & full, own ? c : kNoCell, 0u};
        s_gap[r] = ms.rar[c];  // (ms.gap: other tiles may have written theirs)
    }
    __syncthreads();
    const int nw = ((int)K + 7) >> 3;
    uint32_t* const row = s_code + threadIdx.x * (kRow / 4);
    int n_moved = 0, n_del = 0, n_drop = 0;
    // the colour-p cells whose processing is exact in the region: x = vx +
    // 3i (i < cx), y = vy + 3j (j < cy); this thread's one of them
    auto my_cell = [&](int p, int& x, int& y) {
        const int ax = gx0 == 0 ? 0 : gx0 - cone_lo(p, 0) + 1;
        const int bx = gx1 == n0 - 1 ? n0 - 1 : gx1 - cone_hi(p, 0) - 1;
        const int ay = gy0 == 0 ? 0 : gy0 - cone_lo(p, 1) + 1;
        const int by = gy1 == n1 - 1 ? n1 - 1 : gy1 - cone_hi(p, 1) - 1;
        const int vx = ax + (p / 3 - ax % 3 + 3) % 3;
        const int vy = ay + (p % 3 - ay % 3 + 3) % 3;
        const int cx = vx <= bx ? (bx - vx) / 3 + 1 : 0;
        const int cy = vy <= by ? (by - vy) / 3 + 1 : 0;
        const int t = threadIdx.x;
        if (t >= cx * cy) return false;
        x = vx + 3 * (t % cx);
        y = vy + 3 * (t / cx);
        return true;
    };
    // the words and code words of a phase's cell are loaded one phase ahead,
    // so that they are in flight during the phase before
    uint64_t nxt[8], mov = 0, stm = 0;
    int x = 0, y = 0;
    auto fetch = [&](int p) {
        const bool ok = my_cell(p, x, y);
        if (ok) {
            const uint32_t S32 = (uint32_t)x + (uint32_t)n0 * (uint32_t)y;
            load_codes(ms, S32, C32, nw, nxt);
            mov = ms.mov[S32];
            stm = ms.stm[S32];
        }
        return ok;
    };
    bool mine = fetch(0);
    for (int p = 0; p < kNB<2>; ++p) {
        const int px = x, py = y;
        const bool live = mine;
        const uint64_t mov_p = mov, stm_p = stm;
        if (live) put_codes(row, nxt, nw);
        if (p + 1 < kNB<2>) mine = fetch(p + 1);
        const int r = (px - gx0) + RX * (py - gy0);
        uint64_t gap = live ? s_gap[r] : 0ull;
        if (live && (mov_p | gap)) {
            const uint32_t S32 = (uint32_t)px + (uint32_t)n0 * (uint32_t)py;
            const int col0 = p / 3, col1 = p % 3;
            const uint64_t gap0 = gap;
            NbEntry* const nb0 = s_nb + (r - 1 - RX);
            auto at = [&](uint32_t cd) -> NbEntry& { return nb0[cd]; };
            auto later = [&](uint32_t cd, NbEntry& to, uint64_t fb) {
                const int n = neighbour_of<2>(cd), dx = n % 3 - 1, dy = n / 3 - 1;
                if (((col0 + dx + 3) % 3) * 3 + (col1 + dy + 3) % 3 > p)
                    atomicOr(reinterpret_cast<unsigned long long*>(&s_gap[&to - s_nb]),
                             (unsigned long long)fb);
            };
            int mv = 0, dl = 0, dr = 0;
            run_cell<2, STATS>(mov_p, stm_p, gap, s_nb[r].free, row, at, later, ms.org, S32, C32,
                               K, mv, dl, dr);
            if (gap != gap0) s_gap[r] = gap;
            if (STATS && tx0 <= px && px <= tx1 && ty0 <= py && py <= ty1) {
                n_moved += mv;
                n_del += dl;
                n_drop += dr;
            }
        }
        __syncthreads();
    }
    const int ow = tx1 - tx0 + 1, oh = ty1 - ty0 + 1;
    for (int i = threadIdx.x; i < ow * oh; i += BS) {
        const int cx = i % ow, cy = i / ow;
        const uint32_t c = (uint32_t)(tx0 + cx) + (uint32_t)n0 * (uint32_t)(ty0 + cy);
        const int r = (tx0 - gx0) + cx + RX * ((ty0 - gy0) + cy);
        ms.occ[c] = ~s_nb[r].free & full;
        if (s_gap[r]) ms.gap[c] = s_gap[r];
    }
    if (STATS) {
        stat_add(st, ST_MOVED, n_moved);
        stat_add(st, ST_DELETED, n_del);
        stat_add(st, ST_DROPPED, n_drop);
    }
}

// ------------------------------------------------------------ 3. scatter
// T: coordinate type (double: FP64 drop-in, float: split offsets)
template <int D, typename T>
struct TPtr3 {
    T* p[3];
};

// Bytes from a record's start to its fields.
template <int D, typename T>
constexpr int kFieldAt = (sizeof(T) * D + 7) / 8 * 8;

// FIELDS: nargs > 0.  REC16: 2D split with one field (16-byte records, one load
// per arrival)
template <int D, typename T, bool FIELDS, bool REC16 = false>
__global__ void __launch_bounds__(kBlock) k_mv_scatter(Grid<D> g, TPtr3<D, T> coords,
                                                       uint8_t* __restrict__ index, int nargs,
                                                       ArgPtrs args, MoveScratch ms,
                                                       const SplitGeom* __restrict__ geo,
                                                       int span, int* __restrict__ flag) {
    // the phases are over: the flag words are ready for the next move
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) flag[0] = flag[1] = 0;
    // one thread per cell and slot group (blockIdx.y, `span` slots), chunks of
    // 8 slot planes in lockstep across the wavefront (coalesced origin loads
    // and final stores); only the reads of the staged data are scattered.
    // Arrivals copy their staged data, vacated slots are emptied
    // (empty_particle!, src/Particles/move_safe.jl:243-251).  Nothing moves
    // when the split grid was rejected (geo: null in the FP64 form).
    if (geo && geo->bad) return;
    // 2D: XCD-contiguous cell ranges (a destination's sources are its
    // neighbour cells, whose staged lines other threads of the same L2 also
    // read; a row of cells above or below is only a few workgroups away, which
    // round-robin dealing puts on other XCDs); slot groups of one cell block
    // stay together.  3D keeps the dealt order: there the plane above or below
    // is a multiple of 8 workgroups away, already on the same XCD, and the
    // renumbering measured slower.
    const unsigned lb = D == 2 ? xcd_block(blockIdx.x + gridDim.x * blockIdx.y,
                                           gridDim.x * gridDim.y)
                               : blockIdx.x * gridDim.y + blockIdx.y;
    const int64_t c = (lb / gridDim.y) * (int64_t)blockDim.x + threadIdx.x;
    if (c >= g.C) return;
    const int kb = (int)(lb % gridDim.y) * span;
    const int ke = kb + span < g.K ? kb + span : g.K;
    const int64_t C = g.C;
    // the first chunk's origins go out with the cell's words: unguarded loads
    // (slot clamped to K - 1, values used for arrivals only), one round trip
    // fewer than loading them after the arrival bits are known
    uint16_t o0[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = kb + j < g.K ? kb + j : g.K - 1;
        o0[j] = ms.org[org_at<D>((uint32_t)c, (uint32_t)k, (uint32_t)C, (uint32_t)g.K)];
    }
    const uint64_t occ = ms.occ[c], occ0 = ms.occ0[c], gap = ms.gap[c];
    const uint64_t arr = arrivals(occ, occ0, ms.mov[c]);
    const uint64_t work = arr | (~occ & (occ0 | gap));  // arrivals, emptied slots
    if (!(work >> kb)) return;
    const int str1 = (int)g.ni[0], str2 = (int)(g.ni[0] * g.ni[1]);
    for (int k0 = kb; k0 < ke; k0 += 8) {
        const uint32_t wb = (uint32_t)(work >> k0) & 0xFFu;
        if (!wb) continue;
        const uint32_t ab = (uint32_t)(arr >> k0) & 0xFFu;
        uint32_t o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t at = org_at<D>((uint32_t)c, (uint32_t)(k0 + j), (uint32_t)C,
                                          (uint32_t)g.K);
            o[j] = k0 == kb ? (uint32_t)o0[j] : ((ab >> j) & 1) ? (uint32_t)ms.org[at] : 0u;
        }
        // the record numbers: of the source cell, its rank-th
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t src = (uint32_t)c - (uint32_t)move_offset<D>((o[j] >> 6) & 0x7Fu, str1,
                                                                        str2);
            if (((ab >> j) & 1) && o[j] == kOrgFar)
                o[j] = ms.orgf[org_at<D>((uint32_t)c, (uint32_t)(k0 + j), (uint32_t)C,
                                         (uint32_t)g.K)];
            else
                o[j] = src * (uint32_t)g.K + (o[j] & 63u);
        }
        if constexpr (REC16) {
            float u0[8], u1[8];
            double fv[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                u0[j] = u1[j] = __builtin_nanf("");
                fv[j] = dnan();
                if ((ab >> j) & 1) stg_get16(ms, o[j], u0[j], u1[j], fv[j]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (!((wb >> j) & 1)) continue;
                const int64_t e = c + C * (k0 + j);
                coords.p[0][e] = (T)u0[j];
                coords.p[D - 1][e] = (T)u1[j];
                index[e] = (uint8_t)((ab >> j) & 1);
                args.p[0][e] = fv[j];
            }
            continue;
        }
        // a record's coordinates and first field in one go: wide loads (of a pair of
        // doubles, of three floats) and no second round trip for the field (FP64,
        // 512^2: array by array 131 us, 120)
        T v[8][D];
        double av[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
#pragma unroll
            for (int d = 0; d < D; ++d) v[j][d] = (T)dnan();
            av[j] = dnan();
            if ((ab >> j) & 1) {
                const char* __restrict__ r = ms.stg + (int64_t)o[j] * ms.stride;
#pragma unroll
                for (int d = 0; d < D; ++d) v[j][d] = reinterpret_cast<const T*>(r)[d];
                if (FIELDS) av[j] = *reinterpret_cast<const double*>(r + kFieldAt<D, T>);
            }
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (!((wb >> j) & 1)) continue;
            const int64_t e = c + C * (k0 + j);
#pragma unroll
            for (int d = 0; d < D; ++d) coords.p[d][e] = v[j][d];
            index[e] = (uint8_t)((ab >> j) & 1);
            if (FIELDS) args.p[0][e] = av[j];
        }
        for (int a = 1; a < nargs; ++a) {
#pragma unroll
            for (int j = 0; j < 8; ++j) av[j] = ((ab >> j) & 1) ? stg_field<D>(ms, o[j], a) : dnan();
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if ((wb >> j) & 1) args.p[a][c + C * (k0 + j)] = av[j];
        }
    }
}

// ------------------------------------------------------------ split classify
// Split positions: the slot's cell plus an offset u in cell units.  A particle
// whose floor(u) is zero in every dimension stays; otherwise its destination
// is the cell + floor(u) (deleted when that lies outside the grid), and the
// staged offset is renormalised to the destination, u - floor(u), in FP64.
template <int D>
__global__ void __launch_bounds__(kClassifyMax)
    k_mv_classify_split(Grid<D> g, TPtr3<D, float> off, const uint8_t* __restrict__ index,
                        int nargs, ArgPtrs args, MoveScratch ms, int* flag,
                        const SplitGeom* __restrict__ geo) {
    __shared__ CellWords s_w;
    __shared__ uint32_t s_code[64 * kRow / 4];
    const ClassifySlots<D> cs = classify_slots<D, true>(g);
    if (geo->bad) {  // grid rejected: the later kernels of this move return at once
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(flag, kFlagRejected);
        return;  // (uniform over the block)
    }
    const int64_t c = cs.live ? cs.c : 0;
    const int kb = cs.kb, ke = cs.ke;  // slot chunk(s) kb..ke-1
    const int64_t C = g.C;
    int64_t I[D];
    unlin<D>(g.ni, c, I);
    const uint64_t occ = cs.live ? active_slots_in(index, c, C, kb, ke) : 0ull;
    uint64_t* __restrict__ cw = reinterpret_cast<uint64_t*>(ms.code) + c;
    uint32_t* row = s_code + (threadIdx.x & 63) * (kRow / 4);
    uint8_t* const crow = reinterpret_cast<uint8_t*>(row);
    fill_codes<D>(row, kb, kb + 8);
    constexpr int B = 8;
    const double* __restrict__ f0 = nargs ? args.p[0] : nullptr;
    for (int k0 = kb; k0 < ke; k0 += B) {
        // the offsets and the first field of the chunk's particles in one round
        // (the field of a particle that stays is loaded for nothing; loading it
        // after the movers are known would cost a round trip)
        float ub[B][D];
        double fb[B];
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const bool on = (occ >> (k0 + j)) & 1;
#pragma unroll
            for (int d = 0; d < D; ++d) ub[j][d] = on ? off.p[d][c + C * (k0 + j)] : 0.0f;
            fb[j] = (on && f0) ? f0[c + C * (k0 + j)] : 0.0;
        }
        uint32_t cd8[2] = {0, 0};  // the chunk's codes, by slot
        uint32_t mv8 = 0, stg = 0;
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const int k = k0 + j;
            if (!((occ >> k) & 1)) continue;
            int s[D];
            bool stay = true, out = false, far = false;
            int n = 0, mult = 1, jump = 0;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const bool fin = fabsf(ub[j][d]) < 1.0e6f;  // false for NaN/Inf
                s[d] = fin ? (int)floorf(ub[j][d]) : 0;
                out = out || !fin;
                const int64_t Jd = I[d] + s[d];
                out = out || Jd < 0 || Jd >= g.ni[d];
                stay = stay && s[d] == 0;
                far = far || s[d] > 1 || s[d] < -1;
                jump = s[d] < -jump ? -s[d] : (s[d] > jump ? s[d] : jump);
                n += (s[d] + 1) * mult;
                mult *= 3;
            }
            if (stay && !out) continue;
            mv8 |= 1u << j;
            if (out) continue;  // deleted
            uint32_t cd;
            if (far) {  // staged as it is: the far-jump path renormalises it
                atomicOr(flag, kFlagFar);
                atomicMax(flag + 1, jump);
                cd = kFar;
            } else {
                cd = code_of<D>(n);
#pragma unroll
                for (int d = 0; d < D; ++d)  // the staged value: the offset in the new cell
                    ub[j][d] = (float)((double)ub[j][d] - (double)s[d]);
            }
            stg |= 1u << j;
            cd8[j >> 2] |= cd << (8 * (j & 3));
        }
        // the chunk's staged movers, packed after the cell's earlier ones
        // (one chunk per thread)
        s_w.put(W_OCC, (uint32_t)(occ >> k0));
        s_w.put(W_MOV, mv8);
        s_w.put(W_STG, stg);
        __syncthreads();
        const int r0 = __popcll(s_w.get(W_STG) & ((1ull << k0) - 1));
#pragma unroll
        for (int j = 0; j < B; ++j)
            if ((stg >> j) & 1)
                crow[r0 + __popc(stg & ((1u << j) - 1))] = (uint8_t)(cd8[j >> 2] >> (8 * (j & 3)));
        const int64_t o0 = c * g.K + r0;
        __syncthreads();
        if (cs.live) {
            // (one code word per chunk-thread)
            if (__popcll(s_w.get(W_STG)) > kb) cw[(kb >> 3) * C] = code_word(row, kb >> 3);
            for (int w = (int)(threadIdx.x >> 6); w < W_COUNT; w += (int)(blockDim.x >> 6))
                store_word<D>(ms, c, w, w == W_GAP ? 0ull  // no ties: floor(u) is never the cell
                                                   : s_w.get(w));
            if (D == 2 && nargs == 1) {  // 16-byte records (the scatter reads them whole)
#pragma unroll
                for (int j = 0; j < B; ++j)
                    if ((stg >> j) & 1)
                        stg_put16(ms, o0 + __popc(stg & ((1u << j) - 1)), ub[j][0],
                                  ub[j][D - 1], fb[j]);
            } else {
#pragma unroll
                for (int j = 0; j < B; ++j)
                    if ((stg >> j) & 1) {
                        const int64_t o = o0 + __popc(stg & ((1u << j) - 1));
#pragma unroll
                        for (int d = 0; d < D; ++d) stg_coord<D, float>(ms, o, d) = ub[j][d];
                        if (f0) stg_field<D>(ms, o, 0) = fb[j];
                    }
                stage_args<D>(c, C, k0, stg, o0, nargs, args, ms, 1);
            }
        }
    }
}

ArgPtrs argptrs(double* const* a, int n) {
    ArgPtrs p;
    for (int i = 0; i < JP_MAX_ARGS; ++i) p.p[i] = i < n ? a[i] : nullptr;
    return p;
}

template <int D, typename T>
TPtr3<D, T> tptr3(T* const* c) {
    TPtr3<D, T> p{{nullptr, nullptr, nullptr}};
    for (int d = 0; d < D; ++d) p.p[d] = c[d];
    return p;
}

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// classify -> colour phases (2D: one tiled launch; 3D: 3^D launches) -> far-
// jump phases (one workgroup, of the tiled launch or of one that returns at once
// unless a particle jumped more than one cell; then the regular phases returned
// at once) -> scatter
template <int D, typename T>
int run_move(jp_ctx* ctx, const jp_cellgrid* gc, T* const* coords, uint8_t* index, int nargs,
             double* const* args, jp_stats* stats) {
    Grid<D> g = to_grid<D>(gc);
    const int64_t C = g.C, S = C * g.K;
    if (S >= ((int64_t)1 << 32))
        return fail(ctx, JP_ERR_ARG, "more than 2^32 slots%s");
    MoveScratch ms;
    size_t off = 0;
    const size_t o_occ0 = off; off = align_up(off + C * 8, 256);
    const size_t o_occ = off;  off = align_up(off + C * 8, 256);
    const size_t o_mov = off;  off = align_up(off + C * 8, 256);
    const size_t o_gap = off;  off = align_up(off + C * 8, 256);
    const size_t o_rar = off;  off = align_up(off + (D == 2 ? C * 8 : 0), 256);
    const size_t o_code = off; off = align_up(off + (size_t)C * 64, 256);
    const size_t o_org = off;  off = align_up(off + (size_t)S * 2, 256);
    const size_t o_orgf = off; off = align_up(off + (size_t)S * 4, 256);
    const size_t o_stm = off;  off = align_up(off + C * 8, 256);
    ms.S = S;
    ms.foff = kFieldAt<D, T>;
    ms.stride = ms.foff + 8 * nargs;
    const size_t stg_bytes = (size_t)S * (size_t)ms.stride;
    const size_t o_stg = off;  off = align_up(off + stg_bytes, 256);
    int rc = ensure_scratch(ctx, off);
    if (rc) return rc;
    char* base = static_cast<char*>(ctx->scratch);
    ms.occ0 = (uint64_t*)(base + o_occ0);
    ms.occ = (uint64_t*)(base + o_occ);
    ms.mov = (uint64_t*)(base + o_mov);
    ms.gap = (uint64_t*)(base + o_gap);
    ms.rar = (uint64_t*)(base + o_rar);
    ms.code = (uint8_t*)(base + o_code);
    ms.org = (uint16_t*)(base + o_org);
    ms.orgf = (uint32_t*)(base + o_orgf);
    ms.stm = (uint64_t*)(base + o_stm);
    ms.stg = base + o_stg;

    int* flag = dflags(ctx);
    // the flag words are zero here: a new context starts with them cleared, the
    // scatter, which runs on every move after the phases, clears them after use,
    // and a launch that fails after classify clears them here
    auto launched = [&]() -> int {
        const hipError_t e = hipGetLastError();
        if (e == hipSuccess) return JP_OK;
        if (!ctx->capturing) {
            (void)hipStreamSynchronize(ctx->stream);
            (void)hipMemset(flag, 0, 2 * sizeof(int));
        }
        return fail(ctx, JP_ERR_HIP, "HIP error %s", hipGetErrorString(e));
    };
    if ((rc = stats_begin(ctx, stats))) return rc;
    jp_stats* st = stats ? dstats(ctx) : nullptr;
    ArgPtrs ap = argptrs(args, nargs);
    TPtr3<D, T> cp = tptr3<D, T>(coords);
    // per-cell kernels: slot groups on blockIdx.y when the cells alone do not
    // fill the chip (up to 24 workgroups per CU: with one 8-slot chunk per
    // thread, no chunk's loads wait for an earlier chunk's stores)
    const int span = slot_span(ctx, blocks_for(C), g.K, 6144);
    const dim3 cgrid((unsigned)blocks_for(C), (unsigned)((g.K + span - 1) / span));
    // classify (classify_slots): a workgroup of one wavefront per 8-slot chunk
    // for each 64 cells (2D, 3D split), else a thread per cell
    const bool chunks = D == 2 || !std::is_same<T, double>::value;
    const unsigned kblocks = (unsigned)(chunks ? (C + 63) / 64 : blocks_for(C));
    const unsigned kthreads = (unsigned)(chunks ? 64 * ((g.K + 7) / 8) : kBlock);
    if constexpr (std::is_same<T, double>::value) {
        CPtr3 cc{{nullptr, nullptr, nullptr}};
        for (int d = 0; d < D; ++d) cc.p[d] = coords[d];
        k_mv_classify<D><<<kblocks, kthreads, 0, ctx->stream>>>(g, cc, index, nargs, ap, ms,
                                                               flag);
    } else {
        if ((rc = split_geometry(ctx, gc, nullptr))) return rc;
        k_mv_classify_split<D><<<kblocks, kthreads, 0, ctx->stream>>>(g, cp, index, nargs, ap,
                                                                     ms, flag, geo_ptr(ctx));
    }
    if ((rc = launched())) return rc;
    int64_t total = 1;
    for (int d = 0; d < D; ++d) total *= (g.ni[d] + 2) / 3;
    constexpr int BS = D == 2 ? 128 : 64;  // measured: 256 and 64 (2D), 128 (3D) slower
    const int nphase = (D == 2 && !ctx->opt_move_phases) ? 0 : kNB<D>;
    if (D == 2 && !ctx->opt_move_phases) {
        constexpr int TX = 32, TY = 16;
        const int64_t tiles = ((g.ni[0] + TX - 1) / TX) * ((g.ni[1] + TY - 1) / TY);
        if (tiles >= ((int64_t)1 << 31) || g.ni[0] >= ((int64_t)1 << 30) ||
            g.ni[1] >= ((int64_t)1 << 30))
            return fail(ctx, JP_ERR_ARG, "grid too large%s");
        Grid<2> g2 = to_grid<2>(gc);
        if (st)
            k_mv_tiles2<TX, TY, 256, true, T><<<(unsigned)tiles, 256, 0, ctx->stream>>>(g2, ms, flag,
                                                                                   st);
        else
            k_mv_tiles2<TX, TY, 256, false, T><<<(unsigned)tiles, 256, 0, ctx->stream>>>(g2, ms,
                                                                                    flag, st);
        if ((rc = launched())) return rc;
    }
    for (int ph = 0; ph < nphase; ++ph) {
        Off3 o{{0, 0, 0}};
        int r = ph;
        for (int d = D - 1; d >= 0; --d) {
            o.o[d] = r % 3;
            r /= 3;
        }
        const unsigned nb = (unsigned)((total + BS - 1) / BS);
        if (st)
            k_mv_phase<D, BS, true><<<nb, BS, 0, ctx->stream>>>(g, ms, o, ph, flag, st);
        else
            k_mv_phase<D, BS, false><<<nb, BS, 0, ctx->stream>>>(g, ms, o, ph, flag, st);
        if ((rc = launched())) return rc;
    }
    if (nphase) {
        k_mv_far<D, T><<<1, kFarBlock, 0, ctx->stream>>>(g, ms, flag, st);
        if ((rc = launched())) return rc;
    }
    const SplitGeom* geo = std::is_same<T, double>::value ? nullptr : geo_ptr(ctx);
    bool rec16 = false;  // 2D split, one field: 16-byte records
    if constexpr (D == 2 && std::is_same<T, float>::value) {
        rec16 = nargs == 1;
        if (rec16)
            k_mv_scatter<D, T, true, true><<<cgrid, kBlock, 0, ctx->stream>>>(g, cp, index, nargs, ap,
                                                                        ms, geo, span, flag);
    }
    if (!rec16 && nargs)
        k_mv_scatter<D, T, true><<<cgrid, kBlock, 0, ctx->stream>>>(g, cp, index, nargs, ap, ms,
                                                                   geo, span, flag);
    else if (!rec16)
        k_mv_scatter<D, T, false><<<cgrid, kBlock, 0, ctx->stream>>>(g, cp, index, nargs, ap, ms,
                                                                    geo, span, flag);
    if ((rc = launched())) return rc;

    if ((rc = stats_end(ctx, stats))) return rc;
    return std::is_same<T, double>::value ? finish(ctx) : split_finish(ctx);
}

int check_ptrs(jp_ctx* ctx, int n, const void* const* p, const char* what) {
    if (!p) return fail(ctx, JP_ERR_ARG, "null %s array", what);
    for (int i = 0; i < n; ++i)
        if (!p[i]) return fail(ctx, JP_ERR_ARG, "null %s pointer %lld", what, i);
    return JP_OK;
}

template <typename T>
int move_entry(jp_ctx* ctx, const jp_cellgrid* g, T* const* coords, uint8_t* index, int nargs,
               double* const* args, jp_stats* stats) {
    int rc = check_grid(ctx, g);
    if (rc) return rc;
    if ((rc = check_ptrs(ctx, g->ndim, (const void* const*)coords, "coords"))) return rc;
    if (!index) return fail(ctx, JP_ERR_ARG, "null index%s");
    if (nargs < 0 || nargs > JP_MAX_ARGS) return fail(ctx, JP_ERR_ARG, "nargs out of range%s");
    if (nargs && (rc = check_ptrs(ctx, nargs, (const void* const*)args, "args"))) return rc;
    return g->ndim == 2 ? run_move<2, T>(ctx, g, coords, index, nargs, args, stats)
                        : run_move<3, T>(ctx, g, coords, index, nargs, args, stats);
}

}  // namespace

extern "C" int jp_move_particles(jp_ctx* ctx, const jp_cellgrid* g, double* const* coords,
                                 uint8_t* index, int nargs, double* const* args, jp_stats* stats) {
    return move_entry<double>(ctx, g, coords, index, nargs, args, stats);
}

extern "C" int jp_move_particles_split(jp_ctx* ctx, const jp_cellgrid* g, float* const* off,
                                       uint8_t* index, int nargs, double* const* args,
                                       jp_stats* stats) {
    return move_entry<float>(ctx, g, off, index, nargs, args, stats);
}
