// k_sph.hip -- fixed-radius neighbour search, plain h-iteration, density, EOS and
// internal forces, all on the key-sorted working copies.
//
// Neighbour search.  The reference walks the tree once per particle with per-thread
// stacks (SPH::Kernel::fixedRadiusNN, sph.cu:93-281).  Here one wavefront owns 64
// consecutive key-sorted particles: it walks the tree once with the group's bounding box
// grown by the group's largest h, collecting the particle ranges of small cells (each
// cell is a contiguous range of sorted positions), then streams the candidates through
// LDS in tiles of 64 with coalesced SoA loads; every particle is tested against every candidate of
// the tile with the reference criterion d^2 < h_i^2 and d^2 < h_j^2, on the matrix cores where the
// result is clear and in FP64 otherwise, so the neighbour sets equal a brute-force search.
#include <algorithm>
#include <type_traits>

#include "mhpc_internal.h"

#define NN_WAVES 2
#define NN_CWIN 512   // group walk, list modes: the consumers' LDS window (in-window neighbours first)
#define NN_PB 4      // group walk, FP64 tests: candidates read from LDS per batch
#define NN_STACK_SLACK 192   // hard stack capacity above the soft one: a node a level opens
#define NN_RANGES 128
#define NN_LEAF 16           // per-particle walks: cells of at most this many particles are taken whole
#define NN_LEAF_GROUP 64     // group walks: the same for the 64-particle groups' boxes
static_assert(NN_LEAF_GROUP < NN_CWIN, "a clipped range crosses at most one end of the window");
#define NN_OUTLIER 4.0       // group-mode outlier: h above this factor x the group's smallest
#define NN_OUTLIER_MAX 32    // at most this many outliers per group are split off
#define NN_SPLIT_VOL 8.0     // group walks: a box of more than this many search cubes (2 h)^3 ...
#define NN_SPLIT_CAND 3072   // ... whose start cells hold more than this many particles is split
#define NN_PART_CAND 12288   // split-off parts of more candidates than this, and ...
#define NN_SPLIT_MIN 16      // ... of fewer particles go to the per-particle mode
static_assert(64 / NN_SPLIT_MIN <= MHPC_NN_PARTS_PER_GROUP, "the part list holds every group's parts");
// Re-lists: groups with at most NN_SPARSE flagged particles go per particle (lanes are
// candidates), the others are walked again.  A group walk costs as much as about ten
// per-particle searches: with 64 / 32 / 16 / 8 / 4 a step of the 128^3 blast takes
// 9.61 / 9.50 / 8.96 / 8.88 / 8.87 ms and the 1M cloud's RHS 7.45 / 7.41 / 6.91 / 6.68 / 6.63 ms.
// While few particles changed, the one group walk that any group needs is the launch's latency, and
// every flagged particle gets its own wavefront: the re-lists of 128^3 with 4,900 / 37,300 / 70,100
// particles changed take 71 / 170 / 249 us by NN_SPARSE, 44 / 162 / 279 us per particle (a ball of them;
// scattered ones cross at 150,000), those of the evolving Sedov run 130 / 42 us.  Sets of up to
// NN_SPARSE_SMALL particles always take them: their groups are one resident round, as long as its
// slowest group (RHS of a 40,000-particle Plummer sphere whose h all change: 2.94 / 1.57 ms).
#define NN_SPARSE 8
#define NN_SPARSE_CHANGED 32768
#define NN_SPARSE_SMALL 65536
#define NN_DRANGES 256       // direct form: candidate ranges per wavefront
#define NN_DSPAN 5           // direct form: start cells per axis - 1 (<= 216 cells)
#define NN_DIRECT_MAX 32768  // direct form: candidates per wavefront
// Up to this many particles every search is per particle: a group walk of 64 takes 65 us or more
// however few groups there are, a particle's direct search about 12 us.  RHS by group walks / per
// particle, us, lists from pass 0: lattices in Lebesgue order 25^3 423 / 269, 31^3 462 / 357, in
// Hilbert order 340 / 283 and 367 / 365; a lattice whose side is a power of two has no group that
// spans the domain (32^3 340 / 423).  Clustered sets gain most, although a search tests every
// particle of its start cells: Plummer spheres of 20,000 1568 / 636, of 32,768 1400 / 812, two clumps
// of 13,107 in a thin background 3147 / 2843, 28,500 of 30,000 in one start cell 9352 / 7479.
#define NN_FEW 32768
static_assert(NN_FEW <= NN_DIRECT_MAX && NN_DSPAN >= 1, "the direct form declines no box of so few particles");
#define NN_DU 4              // direct form: candidates per lane and round (loads in flight; 2 / 4 / 8 alike)

// candidate filter that keeps everything (per-particle walks test each candidate once)
struct KeepAll {
    __device__ __forceinline__ bool operator()(double, double, double, double) const { return true; }
};

struct NNArgs {
    int64_t n;
    const int32_t *perm;
    const double4 *sxm;
    const double *h;          // h used for the search (h_cur in the h-iteration)
    const int32_t *cstart, *cend, *cchild;
    const double *cbmin, *cbmax;
    int64_t cap_cells;
    // start table (levels 1..kmax) and the root box the keys were computed in
    const int32_t *stab;
    const int2 *srng;         // {first, count} of each table entry's node
    int kmax;
    const double *box;
    // list mode: entry s of particle k is nbr4[(s / 4) * stride + k].{x,y,z,w}[s % 4]
    int4 *nbr4;
    int64_t stride;
    int max_nb;
    int32_t *snoi;
    int32_t *noi_out;         // caller order
    double *sml_out;          // caller order (written when non-null)
    const int32_t *siters;
    int32_t *iters_out;       // caller order (written when non-null)
    // h-iteration mode
    double *h_next;
    uint8_t *done;
    int32_t *iters;
    const double *table;
    int tmax;
    int pass, max_counts, band_lo, band_hi;
    double sml_max;           // upper bound of h (0: none)
    // compacted lists of the particles still iterating: pass p reads list_in / count_in
    // (per-particle mode) and appends the particles that stay unconverged to list_out
    const int32_t *list_in;
    const uint32_t *count_in;
    int32_t *list_out;
    uint32_t *count_out;
    uint32_t *cnt_slot;       // split counting: neighbour count of list slot t
    const int32_t *slot_list; // split counting: the list slots it takes
    const uint32_t *slot_count;
    const uint32_t *changed_count;   // list mode with `only`: the particles whose change flagged them
    const uint8_t *only;      // list mode: when set, only particles with only[k] != 0
    uint8_t *dirty;           // dirty marking: particles whose list must be rebuilt
    double *h0_slot;          // pass 0 with lists: the pass-0 h of each unconverged particle
                              // (slot of list_out); read by the dirty marking
    int32_t *out_list;        // group mode: outlier particles deferred to the per-particle mode
    uint32_t *out_count;
    ulonglong2 *seg_list;     // group mode: {group, lanes} of the parts split off (see nn_split_group)
    uint32_t *seg_count;
    uint32_t *err;
    unsigned long long *counters;
    const double *chmax;      // per cell: an upper bound of its particles' h
    const uint8_t *lcp;       // key levels sorted particles k and k + 1 share (group splits)
    // h-iteration passes: the bounds the new h of the particles still iterating raise
    double *chmax_raise;
    const int32_t *ppar, *cpar;
    // tail passes: set when this pass changed the h of a particle that keeps iterating; a pass
    // whose previous pass changed none (prev_changed set and zero) repeats that pass's counts
    uint32_t *changed;
    const uint32_t *prev_changed;
};

// A tail pass after a pass that changed no h sees the same h everywhere as that pass (the
// particles that finished kept theirs), so every count it would take equals the count the
// previous pass stored in snoi: the counting kernels skip it and k_h_finish reuses snoi.
__device__ __forceinline__ bool h_pass_frozen(const NNArgs &A) {
    return A.prev_changed && *A.prev_changed == 0u;
}

// The positions a search is for -- one particle's, or the box of a group's (active) particles --
// and the largest h among them (the search radius).
struct NNCore {
    double x0, x1, y0, y1, z0, z1;
    double h;
};

// What a walk searches: the box [lo, hi] (the core grown by the search radius) and the core.
struct NNBounds {
    double lox, hix, loy, hiy, loz, hiz;
    NNCore core;
};

// per-wave LDS of the direct form: its candidate ranges (first particle less the number of
// candidates before the range) and where ranges begin among the candidates of a round
struct NNDirectLds {
    int off[NN_DRANGES];
    unsigned long long head[NN_DU];
};
// per-wave LDS of the group walks' matrix tests (nn_tile): one axis of a tile's 64 candidates in
// 16-bit parts, and the parts of their second norms
struct NNTileLds {
    uint2 part[3][64];
    uint16_t norm2[3][64];
    NNBounds bounds;                          // the group's
    double cx, cy, cz, scale, hm2s;           // middle of its box, scale and scaled largest h^2 (nn_tile)
};

// per-wave LDS of the walker; the filtered walk's tiles (TCAP = 128) have room to compact the
// candidates of two 64-particle loads before a full tile of 64 is handed on
template <int TCAP, int STACK, typename Extra>
struct NNWaveLdsT {
    static constexpr int soft = STACK;   // soft stack capacity (see nn_walk_box)
    int stack[STACK + NN_STACK_SLACK];
    int rstart[NN_RANGES];
    int rcnt[NN_RANGES];
    int rpre[64];
    double tx[TCAP], ty[TCAP], tz[TCAP], th2[TCAP];
    int tj[TCAP];
    Extra extra;
};
using NNWaveLds = NNWaveLdsT<64, 512, NNDirectLds>;
// 10 KB, so that 16 wavefronts fit a CU; the stack takes what is left, since it bounds the nodes opened
// per round (208 / 376 entries: 128^3 blast step 7.76 / 7.51 ms, 1M cloud RHS 4.94 / 4.82 ms)
using NNWaveLdsF = NNWaveLdsT<128, 376, NNTileLds>;
static_assert(sizeof(NNWaveLdsF) <= 163840 / 16, "16 wavefronts per CU");

// the squared distance of every neighbour test (and of the bounds that prune them):
// fma(dx, dx, fma(dy, dy, dz^2)), the oracle's form (two fused multiply-adds per test)
__device__ __forceinline__ double nn_d2(double dx, double dy, double dz) { return fma(dx, dx, fma(dy, dy, dz * dz)); }
__device__ __forceinline__ NNCore nn_point(double x, double y, double z, double h) {
    return NNCore{x, x, y, y, z, z, h};
}

// one particle's bounds: its search radius plus a relative margin far above FP64 rounding
__device__ __forceinline__ NNBounds nn_ball(const double4 &p, double h) {
    const double grow = h * (1.0 + 1e-9);
    return NNBounds{p.x - grow, p.x + grow, p.y - grow, p.y + grow, p.z - grow, p.z + grow, nn_point(p.x, p.y, p.z, h)};
}

// Can cell c hold a neighbour j of some particle i of the core?  A pair needs d < h_i^2 and
// d < h_j^2, and the squared distance from the core to the cell's particle box, taken per axis
// as max(0, lo_cell - hi_core, lo_core - hi_cell) and combined in the pair test's form
// (nn_d2), is at most every such pair's d (each rounding is monotone in exact values that
// grow with the per-axis distances), while h_i <= q.h and h_j <= chmax: a
// cell that fails d2 < min(q.h, chmax)^2 holds no neighbour of the core and its subtree is
// skipped.
__device__ __forceinline__ bool nn_cell_reaches(const NNArgs &A, const NNCore &q, int64_t c) {
    const int64_t cc = A.cap_cells;
    const double ex = fmax(fmax(A.cbmin[c] - q.x1, q.x0 - A.cbmax[c]), 0.0);
    const double ey = fmax(fmax(A.cbmin[cc + c] - q.y1, q.y0 - A.cbmax[cc + c]), 0.0);
    const double ez = fmax(fmax(A.cbmin[2 * cc + c] - q.z1, q.z0 - A.cbmax[2 * cc + c]), 0.0);
    const double hm = fmin(A.chmax[c], q.h);
    return nn_d2(ex, ey, ez) < hm * hm;
}

// Raise the cells' h bounds (chmax) to a particle's new h: every ancestor cell whose bound is
// smaller (an atomic maximum on the bits of the positive double, which orders like the value),
// stopping at the first ancestor that already bounds it.  Bounds never shrink within an RHS, so
// they stay upper bounds of the h every later search uses.
__device__ __forceinline__ void hmax_raise(double *chmax, const int32_t *__restrict__ ppar,
                                           const int32_t *__restrict__ cpar, int64_t cap_cells, int64_t k,
                                           double h) {
    const unsigned long long hb = (unsigned long long)__double_as_longlong(h);
    int64_t c = ppar[k];
    while (c >= 0 && c < cap_cells) {
        const unsigned long long old = atomicMax(reinterpret_cast<unsigned long long *>(chmax + c), hb);
        if (old >= hb || c == 0) break;
        c = cpar[c];
    }
}

// Level-K index along one axis of the cell containing v: the keys' bisection of [mn, mx]
// (lower half = key bit 1), counted upwards, so it is monotone in v.
__device__ __forceinline__ int nn_axis_index(double v, double mn, double mx, int K) {
    int idx = 0;
    for (int l = 0; l < K; l++) {
        const double m = 0.5 * (mn + mx);
        if (v < m) {
            mx = m;
            idx <<= 1;
        } else {
            mn = m;
            idx = (idx << 1) | 1;
        }
    }
    return idx;
}

#define NN_START_ALL (-1)     // walk start: table cells covering the box
#define NN_START_PART0 (-2)   // NN_START_PART0 - o: table cells of index = o (mod 8)

// The start level of a walk for the box [lo, hi] (see nn_start_push).
struct NNStart {
    int K, s;                          // start level K = kmax - s (< 1: whole tree)
    int ilx, ihx, ily, ihy, ilz, ihz;  // the box corners' cell indices at level kmax
};

// Called by all lanes together with the same box.  The six bisections run side by side, one per
// lane (one after the other they are a sixth of a direct search's instructions).
template <int SPAN = 3>
__device__ __forceinline__ NNStart nn_start_level(const NNArgs &A, double lox, double hix, double loy,
                                                  double hiy, double loz, double hiz) {
    NNStart S = {};
    const int K0 = A.stab ? A.kmax : 0;
    S.s = K0;
    if (K0 > 0) {
        const int side = wave_lane() & 7;   // {lo, hi} of x, y, z
        const double vx = side & 1 ? hix : lox, vy = side & 1 ? hiy : loy, vz = side & 1 ? hiz : loz;
        const int axis = side < 6 ? side >> 1 : 0;
        const int idx = nn_axis_index(axis == 0 ? vx : axis == 1 ? vy : vz, A.box[2 * axis], A.box[2 * axis + 1], K0);
        S.ilx = __builtin_amdgcn_readlane(idx, 0);
        S.ihx = __builtin_amdgcn_readlane(idx, 1);
        S.ily = __builtin_amdgcn_readlane(idx, 2);
        S.ihy = __builtin_amdgcn_readlane(idx, 3);
        S.ilz = __builtin_amdgcn_readlane(idx, 4);
        S.ihz = __builtin_amdgcn_readlane(idx, 5);
        int s = 0;
        while (s < K0 && ((S.ihx >> s) - (S.ilx >> s) > SPAN || (S.ihy >> s) - (S.ily >> s) > SPAN ||
                          (S.ihz >> s) - (S.ilz >> s) > SPAN))
            s++;
        S.s = s;
    }
    S.K = K0 - S.s;
    return S;
}

// Consumer window of a list walk: the particles [w0, w1) of the density and force kernels'
// LDS window that holds the walking group (w1 - w0 >= leaf; w0 == w1: none).  Their
// candidates are streamed first as one range, so every list holds its in-window neighbours
// first, and the tree walk skips them: a node or range inside the window is dropped (false)
// and a range of at most `leaf` (< NN_CWIN) particles is clipped to its part outside (it
// crosses at most one end of the window).  Larger nodes that cross an end are opened as usual.
__device__ __forceinline__ bool nn_win_clip(int w0, int w1, int &rs, int &rc, int leaf) {
    if (w0 == w1) return true;
    const int64_t e = (int64_t)rs + rc;
    if (rs >= w0 && e <= w1) return false;
    if (rc <= leaf) {
        if (rs < w0 && e > w0) rc = w0 - rs;
        else if (rs < w1 && e > w1) { rc = (int)(e - w1); rs = w1; }
    }
    return true;
}

// Lebesgue prefix of the level-K cell with the per-axis indices (ix, iy, iz) (the lower half of
// an axis sets its key bit, so the indices' bits enter inverted).
static_assert(MHPC_NN_KMAX <= 10, "a prefix of the start table has at most 30 bits");
__device__ __forceinline__ uint32_t nn_spread3(uint32_t v) {   // bit b of ten to bit 3 b
    v = (v | v << 16) & 0x030000ffu;
    v = (v | v << 8) & 0x0300f00fu;
    v = (v | v << 4) & 0x030c30c3u;
    return (v | v << 2) & 0x09249249u;
}
__device__ __forceinline__ uint32_t nn_cell_prefix(int ix, int iy, int iz, int K) {
    const uint32_t m = (1u << K) - 1u;
    return nn_spread3(~(uint32_t)ix & m) | nn_spread3(~(uint32_t)iy & m) << 1 | nn_spread3(~(uint32_t)iz & m) << 2;
}

// Particles in the start cells a walk for the box [lo, hi] would begin from (see nn_start_push):
// the candidates it has to stream, short of what the distance bounds prune.
__device__ __forceinline__ int nn_box_particles(const NNArgs &A, double lox, double hix, double loy, double hiy,
                                                double loz, double hiz) {
    const NNStart S = nn_start_level(A, lox, hix, loy, hiy, loz, hiz);
    if (S.K < 1) return (int)A.n;
    const int bx = S.ilx >> S.s, by = S.ily >> S.s, bz = S.ilz >> S.s;
    const int nx = (S.ihx >> S.s) - bx + 1, ny = (S.ihy >> S.s) - by + 1, nz = (S.ihz >> S.s) - bz + 1;
    const int lane = wave_lane();
    int cnt = 0;
    if (lane < nx * ny * nz) {
        const int64_t e = nn_tab_off(S.K) +
                          (int64_t)nn_cell_prefix(bx + lane % nx, by + (lane / nx) % ny, bz + lane / (nx * ny), S.K);
        if (A.stab[e] >= 0) cnt = A.srng[e].y;
    }
    return wave_sum(cnt);
}

// Start a walk for the box [lo, hi]: the deepest table level K <= kmax at which the box
// spans at most 4 cells per axis, and the table's node for every such cell (a cell of level
// K, a particle alone in it, or none).  Every particle inside the box lies in one of these
// cells (the keys use the same bisection), and the nodes' subtrees are disjoint, so the walk
// sees the same candidates as one from the root, in another order.  A node of at most
// `leaf` particles goes straight to the range list (its particles are candidates, as for a
// leaf the walk would take), any other onto the stack.  With nparts = 8, only cells of
// index = part (mod 8).  With a consumer window [w0, w1), its ranges come first -- the walking
// group's own particles [g0, g0 + 64) before the rest of the window -- and the nodes are
// clipped against it.  Returns the stack count; nr receives the range count.
template <typename LdsT>
__device__ __forceinline__ int nn_start_push(LdsT &L, const NNArgs &A, double lox, double hix, double loy,
                                             double hiy, double loz, double hiz, const NNCore &q, int part,
                                             int nparts, int w0, int w1, int g0, int &nr, int leaf) {
    const int lane = wave_lane();
    int node = -1;
    int2 rng = make_int2(0, 0x7fffffff);
    const NNStart S = nn_start_level(A, lox, hix, loy, hiy, loz, hiz);
    const int K = S.K, s = S.s;
    const int ilx = S.ilx, ihx = S.ihx, ily = S.ily, ihy = S.ihy, ilz = S.ilz, ihz = S.ihz;
    if (K < 1) {
        // box too large for the table (or no table): the whole tree
        if (lane == 0) node = nparts == 1 ? (int)A.n : A.cchild[part];
    } else {
        const int bx = ilx >> s, by = ily >> s, bz = ilz >> s;
        const int nx = (ihx >> s) - bx + 1, ny = (ihy >> s) - by + 1, nz = (ihz >> s) - bz + 1;
        if (lane < nx * ny * nz && lane % nparts == part) {
            const int ix = bx + lane % nx, iy = by + (lane / nx) % ny, iz = bz + lane / (nx * ny);
            const uint32_t P = nn_cell_prefix(ix, iy, iz, K);
            node = A.stab[nn_tab_off(K) + (int64_t)P];
            if (node >= 0) rng = A.srng[nn_tab_off(K) + (int64_t)P];
        }
    }
    if (node >= A.n && !nn_cell_reaches(A, q, node - A.n)) node = -1;
    if (node >= 0 && !nn_win_clip(w0, w1, rng.x, rng.y, leaf)) node = -1;
    int r0 = 0;   // the window's ranges: own group, then the window before and after it
    if (w1 > w0) {
        const int g1 = g0 + 64 < w1 ? g0 + 64 : w1;
        if (lane == 0) {
            L.rstart[0] = g0;
            L.rcnt[0] = g1 - g0;
            int r = 1;
            if (g0 > w0) {
                L.rstart[r] = w0;
                L.rcnt[r] = g0 - w0;
                r++;
            }
            if (w1 > g1) {
                L.rstart[r] = g1;
                L.rcnt[r] = w1 - g1;
            }
        }
        r0 = 1 + (g0 > w0 ? 1 : 0) + (w1 > g1 ? 1 : 0);
    }
    const uint64_t lt = lanemask_lt();
    const bool asRange = node >= 0 && rng.y <= leaf;
    const bool asNode = node >= 0 && !asRange;
    const uint64_t mR = wave_ballot(asRange), mN = wave_ballot(asNode);
    if (asRange) {
        const int pos = r0 + popc64(mR & lt);
        L.rstart[pos] = rng.x;
        L.rcnt[pos] = rng.y;
    }
    if (asNode) L.stack[popc64(mN & lt)] = node;
    nr = r0 + popc64(mR);
    return popc64(mN);
}

// Direct form of a per-particle search for the box [lo, hi]: the start cells of the box (up
// to NN_DSPAN + 1 per axis, at the deepest table level where they cover it) are taken whole as
// particle ranges -- no tree walk -- and every particle of them is handed to
// visit(valid, j, {x,y,z,m}_j, h_j), NN_DU candidates per lane and round with all their loads
// issued first; candidates come in ascending order of (round, slot, lane), and visit is called
// by all lanes together (it may use ballots).  Returns false, before any visit, when the box is
// too large for the table or has more than NN_DIRECT_MAX candidates.
// A search is a chain of waits, so each link is kept short: table entry, range and cell bounds of
// 128 cells are requested at once, and a candidate's range follows from one bit per range start
// (set in LDS) by counting bits, where a binary search would be eight dependent LDS reads per
// candidate (1M cloud: the first tail pass 320 -> 206 us, the re-list marking 311 -> 207 us).
#define NN_DROUNDS ((NN_DSPAN + 1) * (NN_DSPAN + 1) * (NN_DSPAN + 1) + 63) / 64
static_assert(NN_DRANGES >= (NN_DSPAN + 1) * (NN_DSPAN + 1) * (NN_DSPAN + 1), "every cell's range has room");
template <typename VisitFn>
__device__ __forceinline__ bool nn_direct(NNDirectLds &L, const NNArgs &A, const NNBounds &B, VisitFn &&visit) {
    const int lane = wave_lane();
    const uint64_t lt = lanemask_lt();
    const NNCore &q = B.core;
    const NNStart S = nn_start_level<NN_DSPAN>(A, B.lox, B.hix, B.loy, B.hiy, B.loz, B.hiz);
    if (S.K < 1) return false;
    const int K = S.K, s = S.s;
    const int bx = S.ilx >> s, by = S.ily >> s, bz = S.ilz >> s;
    const int nx = (S.ihx >> s) - bx + 1, ny = (S.ihy >> s) - by + 1, nz = (S.ihz >> s) - bz + 1;
    const int ncell = nx * ny * nz;
    // quotients of an index below 256 by nx, ny <= 6: exact with a 16-bit reciprocal rounded up
    const uint32_t rx = 65536u / (uint32_t)nx + 1u, ry = 65536u / (uint32_t)ny + 1u;
    const int64_t tab = nn_tab_off(K);
    constexpr int ROUNDS = NN_DROUNDS;
    int pre[ROUNDS];   // candidates before this lane's range of the round (-1: none)
    int nr = 0, total = 0;
#pragma unroll
    for (int r = 0; r < ROUNDS; r += 2) {
        pre[r] = -1;
        if (r + 1 < ROUNDS) pre[r + 1] = -1;
        if (64 * r >= ncell) continue;
        int first[2], num[2];
#pragma unroll
        for (int v = 0; v < 2; v++) {
            const uint32_t idx = 64 * (r + v) + lane;
            const bool in = idx < (uint32_t)ncell;
            const uint32_t iyz = (idx * rx) >> 16, iz = (iyz * ry) >> 16;
            const uint32_t P = nn_cell_prefix(bx + (int)(idx - iyz * nx), by + (int)(iyz - iz * ny), bz + (int)iz, K);
            const int64_t e = tab + (in ? (int64_t)P : 0);
            const int node = A.stab[e];
            const int2 rg = A.srng[e];   // read beside the node; unused where there is none
            // (cell 0 is read for particles and empty entries, and not looked at)
            const bool reach = nn_cell_reaches(A, q, node >= A.n ? node - A.n : 0);
            const bool keep = in && node >= 0 && (node < A.n || reach);
            first[v] = rg.x;
            num[v] = keep ? rg.y : 0;
        }
#pragma unroll
        for (int v = 0; v < 2; v++) {
            if (r + v >= ROUNDS) break;
            const uint64_t m = wave_ballot(num[v] > 0);
            const int incl = wave_incl_scan(num[v]);
            if (num[v] > 0) {
                pre[r + v] = total + incl - num[v];
                L.off[nr + popc64(m & lt)] = first[v] - pre[r + v];
            }
            nr += popc64(m);
            total += __builtin_amdgcn_readlane(incl, 63);
            if (total > NN_DIRECT_MAX) return false;
        }
    }
    int before = 0;   // ranges that begin before the round's candidates
    for (int base = 0; base < total; base += 64 * NN_DU) {
        if (lane < NN_DU) L.head[lane] = 0ull;
        wave_sync();
#pragma unroll
        for (int r = 0; r < ROUNDS; r++) {
            const uint32_t o = (uint32_t)(pre[r] - base);
            if (pre[r] >= 0 && o < 64u * NN_DU) atomicOr(&L.head[o >> 6], 1ull << (o & 63u));
        }
        wave_sync();
        int jj[NN_DU];
#pragma unroll
        for (int u = 0; u < NN_DU; u++) {
            const unsigned long long w = L.head[u];
            const int c = base + 64 * u + lane;
            // a candidate's range is the last one beginning at or before it
            const int own = before + popc64(w & (lt | 1ull << lane)) - 1;
            before += popc64(w);
            jj[u] = c < total ? L.off[own] + c : -1;
        }
        double4 pj[NN_DU];
        double hj[NN_DU];
#pragma unroll
        for (int u = 0; u < NN_DU; u++) {
            pj[u] = make_double4(0.0, 0.0, 0.0, 0.0);
            hj[u] = 0.0;
            if (jj[u] >= 0) {
                pj[u] = A.sxm[jj[u]];
                hj[u] = A.h[jj[u]];
            }
        }
#pragma unroll
        for (int u = 0; u < NN_DU; u++) visit(jj[u] >= 0, jj[u], pj[u], hj[u]);
    }
    wave_sync();
    return true;
}

// Walk the (sub)tree of node `start` (the root is node n) for the axis-aligned box [lo, hi]
// (the core q grown by the search radius) and hand the candidate particles to
// `tile` in LDS tiles of up to 64 (L.tx/ty/tz/th2/tj, count m).  Cells that cannot hold a
// neighbour of the core (nn_cell_reaches) are skipped with their subtrees.  Leaves of at most
// NN_LEAF particles (NN_LEAF_GROUP with FILTER: the group walks) and single particles are
// taken as ranges of sorted positions; larger cells are opened.  With FILTER, only candidates
// with keep(x, y, z, h^2) true reach the tiles (compacted in walk order, so the tile sequence
// is the unfiltered one minus the dropped candidates).  Returns false on stack overflow.
// Wave-uniform control flow.
// `bounds()` gives the box and the core: a group's are read from LDS where they are needed (they
// are the same in all lanes and would take 38 registers throughout).
template <bool FILTER, typename LdsT, typename BoundsFn, typename KeepFn, typename TileFn>
__device__ __forceinline__ bool nn_walk_box(LdsT &L, const NNArgs &A, BoundsFn &&bounds, int start, int w0, int w1,
                                            int g0, KeepFn &&keep, TileFn &&tile) {
    const int lane = wave_lane();
    const int64_t n = A.n;
    // a group's box spans a few 64-particle cells per axis: taken whole, their candidates come
    // in the order of the start cells, which is also the order the density and force kernels
    // gather best (same lists as sets, fewer distinct lines per gather step)
    constexpr int leaf = FILTER ? NN_LEAF_GROUP : NN_LEAF;
    int top = 1, nr = 0;
    if (start >= 0) {
        if (lane == 0) L.stack[0] = start;
    } else {
        const NNBounds B = bounds();
        top = nn_start_push(L, A, B.lox, B.hix, B.loy, B.hiy, B.loz, B.hiz, B.core,
                            start == NN_START_ALL ? 0 : NN_START_PART0 - start, start == NN_START_ALL ? 1 : 8, w0, w1,
                            g0, nr, leaf);
    }
    wave_sync();
    const uint64_t lt = lanemask_lt();
    int fill = 0;   // FILTER: kept candidates waiting in L.t*[0, fill)
    for (;;) {
        // walk until 64 ranges are pending or the stack is empty
        while (top > 0 && nr < 64) {
            int kpop = (LdsT::soft - top) / 7;
            kpop = kpop < 1 ? 1 : kpop;
            kpop = kpop > 64 ? 64 : kpop;
            kpop = kpop > top ? top : kpop;
            const int node = lane < kpop ? L.stack[top - kpop + lane] : -1;
            top -= kpop;
            wave_sync();
            bool take = false, open = false;
            int rs = 0, rc = 0;
            int64_t c = 0;
            if (node >= 0 && node < n) {
                const double4 r = A.sxm[node];
                const double px = r.x, py = r.y, pz = r.z;
                const NNBounds B = bounds();
                take = px >= B.lox && px <= B.hix && py >= B.loy && py <= B.hiy && pz >= B.loz && pz <= B.hiz;
                rs = node;
                rc = 1;
                take = take && nn_win_clip(w0, w1, rs, rc, leaf);
            } else if (node >= n) {
                c = node - n;
                const int64_t cc = A.cap_cells;
                const NNBounds B = bounds();
                const bool overlap = A.cbmin[c] <= B.hix && A.cbmax[c] >= B.lox &&
                                     A.cbmin[cc + c] <= B.hiy && A.cbmax[cc + c] >= B.loy &&
                                     A.cbmin[2 * cc + c] <= B.hiz && A.cbmax[2 * cc + c] >= B.loz &&
                                     nn_cell_reaches(A, B.core, c);
                if (overlap) {
                    rs = A.cstart[c];
                    rc = A.cend[c] - rs + 1;
                    if (nn_win_clip(w0, w1, rs, rc, leaf)) {
                        if (rc <= leaf) take = true; else open = true;
                    }
                }
            }
            const uint64_t mT = wave_ballot(take);
            if (take) {
                const int pos = nr + popc64(mT & lt);
                L.rstart[pos] = rs;
                L.rcnt[pos] = rc;
            }
            nr += popc64(mT);
            int ch[8];
            int nc = 0;
            if (open) {
                const int4 *cp = reinterpret_cast<const int4 *>(A.cchild + 8 * c);
                const int4 a = cp[0], b = cp[1];
                ch[0] = a.x; ch[1] = a.y; ch[2] = a.z; ch[3] = a.w;
                ch[4] = b.x; ch[5] = b.y; ch[6] = b.z; ch[7] = b.w;
#pragma unroll
                for (int s = 0; s < 8; s++) nc += ch[s] != -1;
            }
            const int incl = wave_incl_scan(nc);
            const int tot = __shfl(incl, 63);
            if (top + tot > LdsT::soft + NN_STACK_SLACK) return false;
            if (open) {
                int pos = top + incl - nc;
#pragma unroll
                for (int s = 7; s >= 0; s--)
                    if (ch[s] != -1) L.stack[pos++] = ch[s];
            }
            top += tot;
            wave_sync();
        }
        // nothing left: one more step hands on the candidates still waiting
        const bool last = nr == 0 && top == 0;
        if (last && fill == 0) return true;
        // stream the candidates of up to 64 ranges through LDS
        const int np = nr < 64 ? nr : 64;
        const int v = lane < np ? L.rcnt[lane] : 0;
        const int incl = wave_incl_scan(v);
        const int total = __shfl(incl, 63);
        const int pre = incl - v;
        L.rpre[lane] = pre;
        wave_sync();
        for (int base = 0; base < total || (FILTER && last); base += 64) {
            const int t = base + lane;
            // the ranges holding this chunk's first and last candidates bound every lane's
            // search (prefixes are non-decreasing): usually one or two ranges apart
            const int rf = popc64(wave_ballot(lane < np && pre <= base)) - 1;
            const int rl = popc64(wave_ballot(lane < np && pre <= base + 63)) - 1;
            if constexpr (!FILTER) {
                if (t < total) {
                    int rlo = rf, rhi = rl;
                    while (rlo < rhi) {
                        const int mid = (rlo + rhi + 1) >> 1;
                        if (L.rpre[mid] <= t) rlo = mid; else rhi = mid - 1;
                    }
                    const int j = L.rstart[rlo] + (t - L.rpre[rlo]);
                    const double hj = A.h[j];
                    const double4 r = A.sxm[j];
                    L.tx[lane] = r.x;
                    L.ty[lane] = r.y;
                    L.tz[lane] = r.z;
                    L.th2[lane] = hj * hj;
                    L.tj[lane] = j;
                }
                wave_sync();
                tile((total - base) < 64 ? (total - base) : 64);
                wave_sync();
            } else {
                bool kp = false;
                double rx = 0.0, ry = 0.0, rz = 0.0, h2 = 0.0;
                int j = 0;
                if (t < total) {
                    int rlo = rf, rhi = rl;
                    while (rlo < rhi) {
                        const int mid = (rlo + rhi + 1) >> 1;
                        if (L.rpre[mid] <= t) rlo = mid; else rhi = mid - 1;
                    }
                    j = L.rstart[rlo] + (t - L.rpre[rlo]);
                    const double hj = A.h[j];
                    const double4 r = A.sxm[j];
                    rx = r.x;
                    ry = r.y;
                    rz = r.z;
                    h2 = hj * hj;
                    kp = keep(rx, ry, rz, h2);
                }
                const uint64_t mk = wave_ballot(kp);
                if (kp) {
                    const int pos = fill + popc64(mk & lt);   // < fill + 64 <= 127
                    L.tx[pos] = rx;
                    L.ty[pos] = ry;
                    L.tz[pos] = rz;
                    L.th2[pos] = h2;
                    L.tj[pos] = j;
                }
                fill += popc64(mk);
                wave_sync();
                if (fill >= 64 || last) {
                    tile(fill < 64 ? fill : 64);
                    if (last) return true;
                    wave_sync();
                    // move the overflow [64, fill) to the front (disjoint ranges)
                    const int rest = fill - 64;
                    if (lane < rest) {
                        const double a0 = L.tx[64 + lane], a1 = L.ty[64 + lane], a2 = L.tz[64 + lane];
                        const double a3 = L.th2[64 + lane];
                        const int a4 = L.tj[64 + lane];
                        L.tx[lane] = a0;
                        L.ty[lane] = a1;
                        L.tz[lane] = a2;
                        L.th2[lane] = a3;
                        L.tj[lane] = a4;
                    }
                    fill = rest;
                    wave_sync();
                }
            }
        }
        const int rest = nr - np;
        if (lane < rest) {
            const int a = L.rstart[64 + lane], b = L.rcnt[64 + lane];
            L.rstart[lane] = a;
            L.rcnt[lane] = b;
        }
        nr = rest;
        wave_sync();
    }
}

// the plain h-iteration's per-particle update after a count N (sph.cu:909-935 in the
// Jacobi form): finish when N is in the band (or at the last pass) and below max_nb,
// else scale h by 1/2 (1 + (n_target / N)^(1/3)) from the table.  Returns fin.
__device__ __forceinline__ bool h_update(const NNArgs &A, int N, double hi, double &hn) {
    const bool inband = N >= A.band_lo && N <= A.band_hi;
    const bool last = A.pass == A.max_counts - 1;
    bool fin = false;
    hn = hi;
    if ((inband || last) && N < A.max_nb) {
        fin = true;
    } else {
        int Nc = N < 1 ? 1 : N;
        Nc = Nc > A.tmax ? A.tmax : Nc;
        hn = hi * A.table[Nc];
        if (A.sml_max > 0.0 && hn > A.sml_max) hn = A.sml_max;
        if (last) fin = true;
    }
    if (fin && (N >= A.max_nb || N == 0)) set_err(A.err, ERRF_CAP_NEIGHBOURS);
    return fin;
}

// bounding box of the active lanes' positions and their largest h
struct NNBox {
    double x0, x1, y0, y1, z0, z1, h;
};
__device__ __forceinline__ NNBox nn_box(bool active, double x, double y, double z, double h) {
    NNBox B;
    B.h = wave_max(active ? h : 0.0);
    B.x0 = wave_min(active ? x : 1e300); B.x1 = wave_max(active ? x : -1e300);
    B.y0 = wave_min(active ? y : 1e300); B.y1 = wave_max(active ? y : -1e300);
    B.z0 = wave_min(active ? z : 1e300); B.z1 = wave_max(active ? z : -1e300);
    return B;
}

// The neighbour tests of a group walk on the matrix cores.  For a particle i and a candidate j, both
// relative to the middle of the group's box and scaled by a power of two so that the largest h is
// below 2, (h_i^2 - d) / 2 = x_i . x_j + (h_i^2 - |x_i|^2) / 2 - |x_j|^2 / 2 is a row of six products
// per axis (each coordinate split exactly into three bfloat16 parts, the products of the parts but
// the smallest three) and three parts of each norm: 24 of the 32 products of one
// v_mfma_f32_16x16x32_bf16 element.  Its sign decides the test unless it is within `eps` of zero;
// then the pair is tested as in every other walk (FP64), so that the sets are the same.
// The error of an element, with M = (box half-diagonal + largest h)^2 bounding the terms' sum by
// 2.5 M: 32 FP32 additions, even truncated one after another, 32 2^-23 2.5 M = 2^-16.7 M; the dropped products
// 2^-20 M; the rounding of coordinates and norms to FP32 2^-22 M.  eps = 2^-16 M.  (Largest error
// measured over 67 million random pairs: 2^-21.2 M.)
// The FP64 tests were most of a walk that is bound by its instructions: 6 operations, 2
// comparisons and a bit per pair, against 1.5 to 2.5 instructions here (256^3 list walk 6.4 -> 5.2 ms,
// 47^3 RHS in two walks 884 -> 668 us, 1M cloud RHS 5.05 -> 4.80 ms, 128^3 blast step 7.69 -> 7.50 ms).
// Sets with a dense clump (40,000 particles, half of them in a ball of 1/1000 of the box): of a group
// that also holds particles from outside, those inside find every particle of the clump within eps,
// and the tests one by one cost more than the tile's by broadcast (k_nn_walk<1> 3.7 ms; 2.0 with such
// tiles tested by broadcast, 1.7 also without the matrix tests in the rest of such a group's walk).
#define NN_CLOSE_MAX 16      // a lane's candidates tested one by one in a tile
#define NN_CLOSE_OFF 48      // with more than these, no matrix tests in the group's further tiles
#define NN_MFMA_REACH 64.0   // largest M (h is 1 to 2): above, most tiles hold a pair too close to zero
typedef unsigned nn_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 nn_bf16x8 __attribute__((ext_vector_type(8)));
typedef float nn_f32x4 __attribute__((ext_vector_type(4)));

// x = parts a + b + c of eight significant bits each (exact), as FP32
struct NNParts {
    uint32_t a, b, c;
};
__device__ __forceinline__ NNParts nn_parts(float x) {
    NNParts p;
    p.a = __float_as_uint(x) & 0xffff0000u;
    const float r = x - __uint_as_float(p.a);
    p.b = __float_as_uint(r) & 0xffff0000u;
    p.c = __float_as_uint(r - __uint_as_float(p.b));
    return p;
}
// the upper halves of two words: lo's below hi's
__device__ __forceinline__ uint32_t nn_pack_hi(uint32_t hi, uint32_t lo) {
    return __builtin_amdgcn_perm(hi, lo, 0x07060302u);
}

// A group's particles as the matrix test needs them: lane (q, c) = 16 q + c holds, of axis q (none
// for q = 3) of the particles 16 a + c, the coordinate's parts {a, b} in ab, its part c and the first
// norm's part q in cn, and the second norm's part q with a one in n2.
struct NNTileI {
    bool on;
    float eps;
    uint32_t ab[4], cn[4], n2[4], one;
};

__device__ __forceinline__ void nn_tile_write(NNTileLds &T, int e, double X, double Y, double Z, float n1, float n2) {
    const NNParts x = nn_parts((float)X), y = nn_parts((float)Y), z = nn_parts((float)Z);
    const NNParts p = nn_parts(n1), r = nn_parts(n2);
    T.part[0][e] = make_uint2(nn_pack_hi(x.b, x.a), nn_pack_hi(p.a, x.c));
    T.part[1][e] = make_uint2(nn_pack_hi(y.b, y.a), nn_pack_hi(p.b, y.c));
    T.part[2][e] = make_uint2(nn_pack_hi(z.b, z.a), nn_pack_hi(p.c, z.c));
    T.norm2[0][e] = (uint16_t)(r.a >> 16);
    T.norm2[1][e] = (uint16_t)(r.b >> 16);
    T.norm2[2][e] = (uint16_t)(r.c >> 16);
}

// live: the lane's particle takes part
__device__ __forceinline__ NNTileI nn_tile_group(NNTileLds &T, bool live, double x, double y, double z, double h2,
                                                 const NNBox &B) {
    NNTileI I;
    const double cx = 0.5 * (B.x0 + B.x1), cy = 0.5 * (B.y0 + B.y1), cz = 0.5 * (B.z0 + B.z1);
    const double scale = ldexp(1.0, -ilogb(B.h));   // largest h in [1, 2)
    const double hs = B.h * scale;
    const double reach =
        0.5 * sqrt(nn_d2((B.x1 - B.x0) * scale, (B.y1 - B.y0) * scale, (B.z1 - B.z0) * scale)) + hs;
    const double M = reach * reach;
    // false where h is infinite; beyond these h the squares leave the normal numbers
    I.on = M <= NN_MFMA_REACH && B.h > 1e-140 && B.h < 1e140;
    I.eps = (float)(M * 1.52587890625e-05);
    if (!I.on) return I;
    const double X = live ? (x - cx) * scale : 0.0, Y = live ? (y - cy) * scale : 0.0,
                 Z = live ? (z - cz) * scale : 0.0;
    const double r2 = nn_d2(X, Y, Z);
    // a lane that takes no part is far from everything
    nn_tile_write(T, wave_lane(), X, Y, Z, live ? (float)(0.5 * (h2 * (scale * scale) - r2)) : -1e30f,
                  live ? (float)(-0.5 * r2) : -1e30f);
    if (wave_lane() == 0) {
        T.cx = cx;
        T.cy = cy;
        T.cz = cz;
        T.scale = scale;
        T.hm2s = hs * hs;
    }
    wave_sync();
    const int q = wave_lane() >> 4, c = wave_lane() & 15, ax = q < 3 ? q : 0;
    I.one = q < 3 ? 0x3f80u : 0u;
#pragma unroll
    for (int a = 0; a < 4; a++) {
        const uint2 v = T.part[ax][16 * a + c];
        I.ab[a] = q < 3 ? v.x : 0u;
        I.cn[a] = q < 3 ? v.y : 0u;
        I.n2[a] = q < 3 ? 0x3f800000u | T.norm2[ax][16 * a + c] : 0u;
    }
    wave_sync();
    return I;
}

// lane 16 q' + c gathers its particle's bits from the four rows of lanes: candidate 0 first
__device__ __forceinline__ void nn_tile_bits(const uint32_t w[4], uint32_t &lo, uint32_t &hi) {
    const auto s02 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
    const auto s13 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
    const auto r01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
    const auto r23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
    lo = __builtin_bitreverse32(r01[0] << 16 | r01[1]);
    hi = __builtin_bitreverse32(r23[0] << 16 | r23[1]);
}

// The tests of the tile's m candidates (bit e of lo, e - 32 of hi: candidate e; bits past m are any)
// for every lane's particle; `exact(e)` is the lane's test of candidate e in FP64.  SAME: every
// candidate's h^2 is at least the largest of the group, so h_i^2 alone decides.
// Returns false, with the bits of the candidates left to FP64, where some lane has more than
// NN_CLOSE_MAX of them: the caller tests the whole tile then.
template <bool SAME, typename LdsT, typename ExactFn>
__device__ __forceinline__ bool nn_tile(LdsT &L, const NNTileI &I, int m, uint32_t &lo, uint32_t &hi,
                                        ExactFn &&exact) {
    const int lane = wave_lane(), q = lane >> 4, ax = q < 3 ? q : 0;
    NNTileLds &T = L.extra;
    {
        const double sc = T.scale;
        const double dx = (L.tx[lane] - T.cx) * sc, dy = (L.ty[lane] - T.cy) * sc, dz = (L.tz[lane] - T.cz) * sc;
        const double r2 = nn_d2(dx, dy, dz);
        // past the tile, or no position (the filter lets a NaN pass): far from everything
        const bool in = lane < m && r2 == r2;
        const double X = in ? dx : 0.0, Y = in ? dy : 0.0, Z = in ? dz : 0.0;
        // beyond the largest h^2 the candidate's own never decides (and may be any size)
        const double h2 = SAME ? 0.0 : fmin(L.th2[lane] * (sc * sc), T.hm2s);
        nn_tile_write(T, lane, X, Y, Z, in ? (float)(-0.5 * r2) : -1e30f,
                      !SAME && in ? (float)(0.5 * (h2 - r2)) : SAME ? 0.f : -1e30f);
    }
    wave_sync();
    uint32_t w[4] = {0, 0, 0, 0}, close[4] = {0, 0, 0, 0};
    bool any_close = false;
    // row 4 q + r of step t is candidate 16 q + 4 t + r, so that a lane's bits of one q are in order
    const int row = 16 * ((lane & 15) >> 2) + (lane & 3);
    auto mfma = [](uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t p0, uint32_t p1, uint32_t p2,
                   uint32_t p3) {
        const nn_u32x4 c = {c0, c1, c2, c3}, p = {p0, p1, p2, p3};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(nn_bf16x8, c),
                                                       __builtin_bit_cast(nn_bf16x8, p),
                                                       nn_f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    };
    // take(a, r, v): v is the element of row r and the particles 16 a + c
    auto step = [&](int t, auto &&take) {
        // candidate slots {a b, a c, a b, 1 n}, particle slots {a a, b a, c b, n 1}
        const uint2 v = T.part[ax][row + 4 * t];
        const uint32_t ac = __builtin_amdgcn_perm(v.y, v.x, 0x05040100u);
        const uint32_t n = __builtin_amdgcn_perm(v.y, 0x3f80u, 0x07060100u);
        uint32_t n2 = 0;
        if constexpr (!SAME) n2 = (uint32_t)T.norm2[ax][row + 4 * t] << 16 | 0x3f80u;
#pragma unroll
        for (int a = 0; a < 4; a += 2) {
            nn_f32x4 d[2], d2[2];
#pragma unroll
            for (int g = 0; g < 2; g++) {
                uint32_t ab = I.ab[a + g], cn = I.cn[a + g];
                asm("" : "+v"(ab), "+v"(cn));   // unpacked in every step: kept unpacked, they cost registers
                const uint32_t p0 = __builtin_amdgcn_perm(ab, ab, 0x01000100u);
                const uint32_t p1 = __builtin_amdgcn_alignbit(ab, ab, 16);
                const uint32_t p2 = __builtin_amdgcn_perm(ab, cn, 0x07060100u);
                const uint32_t p3 = __builtin_amdgcn_alignbit(I.one, cn, 16);
                d[g] = mfma(v.x, ac, v.x, n, p0, p1, p2, p3);
                if constexpr (!SAME) d2[g] = mfma(v.x, ac, v.x, n2, p0, p1, p2, I.n2[a + g]);
            }
            __builtin_amdgcn_sched_barrier(0);
            // the smaller of two floats is the smaller integer, but that of two negative ones it is
            // the one nearer zero, which at most tests a pair again
#pragma unroll
            for (int g = 0; g < 2; g++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    take(a + g, r, SAME ? d[g][r] : __int_as_float(min(__float_as_int(d[g][r]), __float_as_int(d2[g][r]))));
        }
    };
#pragma unroll 1
    for (int t = 0; t < 4; t++) {
        float least = 3.0e38f;
        step(t, [&](int a, int, float v) {
            least = fminf(least, fabsf(v));
            w[a] = __builtin_amdgcn_alignbit(w[a], __float_as_uint(v), 31);   // the sign: no neighbour
        });
        if (wave_ballot(least <= I.eps) != 0) {   // once more, for where
            any_close = true;
            step(t, [&](int a, int r, float v) { close[a] |= (fabsf(v) <= I.eps ? 0x8000u : 0u) >> (4 * t + r); });
        }
    }
    wave_sync();
    nn_tile_bits(w, lo, hi);
    lo = ~lo;
    hi = ~hi;
    if (any_close) {
        uint32_t cl, ch;
        nn_tile_bits(close, cl, ch);
        if (wave_ballot(__popc(cl) + __popc(ch) > NN_CLOSE_MAX) != 0) {
            lo = cl;
            hi = ch;
            return false;
        }
        for (; cl != 0; cl &= cl - 1) {
            const int e = __builtin_ctz(cl);
            lo = exact(e) ? lo | 1u << e : lo & ~(1u << e);
        }
        for (; ch != 0; ch &= ch - 1) {
            const int e = __builtin_ctz(ch);
            hi = exact(32 + e) ? hi | 1u << e : hi & ~(1u << e);
        }
    }
    return true;
}

// does the box, grown by its largest h, hold more than `most` particles?
__device__ __forceinline__ bool nn_crowded(const NNArgs &A, const NNBox &B, int most) {
    return nn_box_particles(A, B.x0 - B.h, B.x1 + B.h, B.y0 - B.h, B.y1 + B.h, B.z0 - B.h, B.z1 + B.h) > most;
}

// A run of 64 keys can cross a boundary of a large cell.  The Lebesgue curve jumps there, so the
// run's box may hold a good part of the domain although each particle's surroundings are small:
// on a 47^3 lattice the worst such group streamed all 103,823 particles as candidates, and its
// one wavefront was the walk's whole time (1.75 ms; 0.22 ms with such groups split, and their
// parts take 0.09 ms).  The box is worth splitting when it is both large against the search
// radius and crowded; a group whose box is small against h, or holds few particles, gains nothing
// from a second walk.  Bounds measured: a volume of 6 / 8 / 12 search cubes gives 1052 / 1050 /
// 1186 us for the 47^3 RHS in two walks, 2048 / 3072 / 4096 / 8192 candidates 995 / 1006 / 1058 /
// 1234 us there and 9.80 / 9.60 / 9.61 / 9.62 ms for a step of the 128^3 blast.
__device__ __forceinline__ bool nn_split_wanted(const NNArgs &A, const NNBox &B, uint64_t m) {
    if ((m & (m - 1)) == 0) return false;   // one particle
    const double w = 2.0 * B.h, ex = B.x1 - B.x0, ey = B.y1 - B.y0, ez = B.z1 - B.z0;
    return (w + ex) * (w + ey) * (w + ez) > NN_SPLIT_VOL * (w * w * w) && nn_crowded(A, B, NN_SPLIT_CAND);
}

// Splits a group's active particles into runs that need no further split, cutting at the
// boundaries of the largest cells first (the smallest shared key prefix between consecutive
// particles; of several, the last).  Runs of at least NN_SPLIT_MIN particles are listed for
// k_nn_rest, one wavefront each; the others go to the per-particle mode, where lanes are
// candidates, and so do runs whose box holds a dense clump (NN_PART_CAND): the one wavefront streaming
// it would be all that the launch waits for (the clump of NN_CLOSE_MAX, RHS in two walks 10.4 -> 7.4 ms;
// a bound of NN_SPLIT_CAND: the same there, 4 to 5 % slower where a fifth of the particles around a
// wider clump meet it).  Every active particle ends up in exactly one of the two lists.
__device__ __forceinline__ void nn_split_group(const NNArgs &A, int64_t group, int64_t k, bool active, double x,
                                               double y, double z, double h) {
    const int lane = wave_lane();
    uint64_t todo = wave_ballot(active);
    while (todo != 0) {
        uint64_t m = todo;
        NNBox B;
        for (;;) {
            B = nn_box((m >> lane) & 1ull, x, y, z, h);
            if (!nn_split_wanted(A, B, m)) break;
            // lanes first .. last - 1 of the run own the boundary to their successor
            const int first = __builtin_ctzll(m), last = 63 - __builtin_clzll(m);
            const int cut = lane >= first && lane < last ? (int)A.lcp[k] * 64 + (63 - lane) : 0x7fffffff;
            const int at = 63 - (wave_min(cut) & 63);   // first <= at < last
            m &= (2ull << at) - 1ull;
        }
        todo &= ~m;
        const int num = popc64(m);
        const bool part = num >= NN_SPLIT_MIN && !nn_crowded(A, B, NN_PART_CAND);
        uint32_t b = 0;
        if (lane == 0) b = part ? atomicAdd(A.seg_count, 1u) : atomicAdd(A.out_count, (uint32_t)num);
        b = __shfl(b, 0);
        if (part) {
            if (lane == 0) A.seg_list[b] = make_ulonglong2((unsigned long long)group, m);
        } else if ((m >> lane) & 1ull) {
            A.out_list[b + popc64(m & lanemask_lt())] = (int32_t)k;
        }
    }
}

// Group mode: one wavefront owns 64 consecutive sorted particles and walks once with the
// bounding box of its active particles grown by their largest h, or once per part of the group
// where the box would be far larger than its particles' surroundings.
// MODE 0: build lists (only the particles flagged in `only` when it is set);
// MODE 1: one Jacobi pass of the h-iteration (count only; with list_out set, the
// unconverged particles are appended to it for the next pass);
// MODE 2: MODE 1 that also writes every particle's list with the h of this pass
// (speculative: kept for the particles whose list cannot change afterwards)
// SEG: `mSeg` lanes of the group only (a part that an earlier launch split off).
template <int MODE, bool SEG>
__device__ __forceinline__ void nn_group(NNWaveLdsF &L, const NNArgs &A, int64_t group, uint64_t mSeg) {
    const int lane = wave_lane();
    const int64_t k = group * 64 + lane;
    const int64_t n = A.n;
    const bool valid = k < n;
    bool active = valid;
    if (SEG) active = valid && ((mSeg >> lane) & 1ull);
    if (!SEG && MODE >= 1 && valid) active = A.done[k] == 0;
    if (!SEG && MODE == 0 && valid && A.only) active = A.only[k] != 0;
    uint64_t mActive = wave_ballot(active);
    if (mActive == 0) {
        if (MODE >= 1 && valid && !SEG) A.h_next[k] = A.h[k];
        return;
    }
    if (!SEG && MODE == 0 && A.only &&
        popc64(mActive) <= (n <= NN_SPARSE_SMALL || *A.changed_count <= NN_SPARSE_CHANGED ? 64 : NN_SPARSE)) {
        // a re-list of a few flagged particles: 64 lanes testing candidates for one or two of
        // them is wasted, so they go to the per-particle mode (lanes = candidates)
        uint32_t b = 0;
        if (lane == 0) b = atomicAdd(A.out_count, (uint32_t)popc64(mActive));
        b = __shfl(b, 0);
        if (active) A.out_list[b + popc64(mActive & lanemask_lt())] = (int32_t)k;
        return;
    }
    const double4 own = valid ? A.sxm[k] : make_double4(0.0, 0.0, 0.0, 0.0);
    const double xi = own.x, yi = own.y, zi = own.z;
    const double hi = valid ? A.h[k] : 0.0;
    const double hi2 = hi * hi;
    // outliers: a few active particles with h above NN_OUTLIER x the group's smallest would
    // grow the search box of all 64; they go to the per-particle mode instead.  So do particles whose
    // position is not finite or whose h is no number: a NaN would make the box, and with it every
    // branch below, differ between the lanes.
    bool outlier = SEG && !active;   // a part's other lanes belong to other waves
    if (!SEG) {
        const bool live = active && nn_d2(xi - xi, yi - yi, zi - zi) == 0.0 && hi2 >= 0.0;
        const double hmin = wave_min(live ? hi : 1e300);
        const bool big = live && hi > NN_OUTLIER * hmin;
        const bool few = popc64(wave_ballot(big)) <= NN_OUTLIER_MAX;
        outlier = (active && !live) || (big && few);
        const uint64_t mO = wave_ballot(outlier);
        if (mO != 0) {
            uint32_t b = 0;
            if (lane == 0) b = atomicAdd(A.out_count, (uint32_t)popc64(mO));
            b = __shfl(b, 0);
            if (outlier) A.out_list[b + popc64(mO & lanemask_lt())] = (int32_t)k;
            active = active && !outlier;
            mActive = wave_ballot(active);
            if (mActive == 0) {
                if (MODE >= 1 && valid && !outlier) A.h_next[k] = hi;
                return;
            }
        }
    }
    // search box: bounding box of the active lanes grown by their largest h (plus a
    // relative margin far above FP64 rounding, so pruning never drops a true pair)
    const NNBox B = nn_box(active, xi, yi, zi, hi);
    if (!SEG && A.seg_list && nn_split_wanted(A, B, mActive)) {
        nn_split_group(A, group, k, active, xi, yi, zi, hi);
        if (MODE >= 1 && valid && !active && !outlier) A.h_next[k] = hi;
        return;
    }
    if (lane == 0) {
        const double grow = B.h * (1.0 + 1e-9);
        L.extra.bounds = NNBounds{B.x0 - grow, B.x1 + grow, B.y0 - grow, B.y1 + grow, B.z0 - grow, B.z1 + grow,
                                  NNCore{B.x0, B.x1, B.y0, B.y1, B.z0, B.z1, B.h}};
    }
    NNTileI I = nn_tile_group(L.extra, active, xi, yi, zi, hi2, B);
    wave_sync();
    // candidate filter: squared distance from the box of the active positions, below both
    // hmax^2 and h_j^2.  Per axis fl(b0 - x) <= fl(x_i - x) for every x_i >= b0 (rounding is
    // monotone), and nn_d2 is monotone in each |axis distance|, so this distance never exceeds
    // the pair test's d for any active i, and every
    // pair with d < h_i^2 <= hmax^2 and d < h_j^2 passes: the tiles lose only non-pairs.
    auto keep = [&](double x, double y, double z, double h2) {
        const NNCore &q = L.extra.bounds.core;
        const double ex = fmax(fmax(q.x0 - x, x - q.x1), 0.0);
        const double ey = fmax(fmax(q.y0 - y, y - q.y1), 0.0);
        const double ez = fmax(fmax(q.z0 - z, z - q.z1), 0.0);
        const double d = nn_d2(ex, ey, ez);
        return d < q.h * q.h && d < h2;
    };

    int count = 0;
    // the last three hits, oldest first (a shift register): on every fourth hit they and the
    // new entry go out as one int4; the stale values left after a store are shifted out by
    // the next three hits before they are stored again
    int p0 = 0, p1 = 0, p2 = 0;
    int4 *wp = A.nbr4 + k;        // where the next four go
    // the count & 3 pending entries, in order, for the final partial int4
    auto tail4 = [&]() {
        const int r = count & 3;
        return r == 1 ? make_int4(p2, 0, 0, 0) : r == 2 ? make_int4(p1, p2, 0, 0) : make_int4(p0, p1, p2, 0);
    };
    // list modes: the group's consumer window (NN_CWIN-aligned) is streamed first
    int w0 = 0, w1 = 0;
    if (MODE != 1) {
        w0 = (int)(group * 64 / NN_CWIN * NN_CWIN);
        w1 = (int)(w0 + NN_CWIN < n ? w0 + NN_CWIN : n);
        if (w1 - w0 < NN_LEAF_GROUP) w0 = w1 = 0;
    }
    // with the window on, the group's own particles are the first candidates streamed, so all of
    // them that pass the filter are in the first tile: only its hits must skip j == k
    bool first_tile = true;
    const bool ok = nn_walk_box<true>(L, A, [&]() { return L.extra.bounds; }, NN_START_ALL, w0, w1,
                                      (int)(group * 64), keep, [&](int m) {
        uint32_t bits[2];
        bool done = false;
        if (I.on) {
            const double hm = L.extra.bounds.core.h;
            auto exact = [&](int e) {
                const double4 own = A.sxm[k];   // k < n: only live lanes have candidates that are close
                const double hk = A.h[k];
                const double d = nn_d2(own.x - L.tx[e], own.y - L.ty[e], own.z - L.tz[e]);
                return (d < hk * hk) & (d < L.th2[e]);
            };
            if (wave_ballot(lane < m && L.th2[lane] < hm * hm) == 0) done = nn_tile<true>(L, I, m, bits[0], bits[1], exact);
            else done = nn_tile<false>(L, I, m, bits[0], bits[1], exact);
            if (!done && wave_ballot(__popc(bits[0]) + __popc(bits[1]) > NN_CLOSE_OFF) != 0) I.on = false;
        }
        if (!done) {
            // FP64: candidates come as LDS broadcasts, NN_PB per batch with all their reads issued
            // first; one bit per test, the last candidate's lowest.  (The lane's own particle is read
            // again: kept, it would cost the matrix form its registers.)
            const int64_t ko = valid ? k : n - 1;
            const double4 own = A.sxm[ko];
            const double xi = own.x, yi = own.y, zi = own.z, hi2 = A.h[ko] * A.h[ko];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                uint32_t b = 0;
                for (int e = 32 * s; e < 32 * s + 32; e += NN_PB) {   // past the tile's end: any of its slots
                    double xs[NN_PB], ys[NN_PB], zs[NN_PB], h2s[NN_PB];
#pragma unroll
                    for (int u = 0; u < NN_PB; u++) {
                        xs[u] = L.tx[e + u];
                        ys[u] = L.ty[e + u];
                        zs[u] = L.tz[e + u];
                        h2s[u] = L.th2[e + u];
                    }
                    uint32_t hits = 0;
#pragma unroll
                    for (int u = 0; u < NN_PB; u++) {
                        const double dx = xi - xs[u];
                        const double dy = yi - ys[u];
                        const double dz = zi - zs[u];
                        const double d = nn_d2(dx, dy, dz);
                        hits |= ((d < hi2) & (d < h2s[u])) ? 1u << (NN_PB - 1 - u) : 0u;
                    }
                    b = b << NN_PB | hits;
                }
                bits[s] = __builtin_bitreverse32(b);
            }
        }
        if (m < 64) {
            bits[0] &= m < 32 ? (1u << m) - 1u : ~0u;
            bits[1] &= m < 32 ? 0u : (1u << (m - 32)) - 1u;
        }
        if (!active) return;
        if (MODE == 1) {   // the particle itself is taken off at the end
            count += __popc(bits[0]) + __popc(bits[1]);
            return;
        }
        // list modes: only the hits pass through the append code, bit by bit: every lane appends its
        // own next hit, so a wavefront runs it as often as its busiest lane has hits.  Every fourth
        // hit's 16-byte store is a branch; its capacity check is needed only when some lane could
        // reach max_nb within this tile.
        auto pairs = [&](auto check_cap, auto check_self) {
            auto append = [&](int j) {
                if (decltype(check_self)::value && j == (int)k) return;
                if ((count & 3) == 3) {
                    if (!decltype(check_cap)::value || count < A.max_nb) *wp = make_int4(p0, p1, p2, j);
                    wp += A.stride;
                }
                p0 = p1;
                p1 = p2;
                p2 = j;
                count++;
            };
#pragma unroll
            for (int s = 0; s < 2; s++) {
                uint32_t b = bits[s];
                while (b != 0) {
                    const int e = __builtin_ctz(b);
                    b &= b - 1;
                    append(L.tj[32 * s + e]);
                }
            }
        };
        const bool self = first_tile || w0 == w1;
        first_tile = false;
        if (wave_ballot(count + m > A.max_nb) == 0) {
            if (self) pairs(std::false_type{}, std::true_type{});
            else pairs(std::false_type{}, std::false_type{});
        } else {
            if (self) pairs(std::true_type{}, std::true_type{});
            else pairs(std::true_type{}, std::false_type{});
        }
    });
    if (!ok) {
        if (lane == 0) set_err(A.err, ERRF_STACK);
        return;
    }
    // every active particle is one of its own candidates, at distance 0
    if (MODE == 1 && active && hi2 > 0.0) count--;
    if (MODE == 2 && active && (count & 3) != 0 && count < A.max_nb)
        A.nbr4[(int64_t)(count >> 2) * A.stride + k] = tail4();
    if (MODE == 0 && A.only) {
        // re-list of flagged particles: counts and caller-order outputs are published for
        // all particles by the density kernel afterwards
        if (active) {
            if ((count & 3) != 0 && count < A.max_nb)
                A.nbr4[(int64_t)(count >> 2) * A.stride + k] = tail4();
            A.snoi[k] = count;
            if (count > A.max_nb) set_err(A.err, ERRF_CAP_NEIGHBOURS);
        }
    } else if (MODE == 0) {
        const bool own_list = valid && !outlier;
        if (own_list && (count & 3) != 0 && count < A.max_nb)
            A.nbr4[(int64_t)(count >> 2) * A.stride + k] = tail4();
        if (own_list) {
            A.snoi[k] = count;
            const int32_t i = A.perm[k];
            A.noi_out[i] = count;
            if (A.sml_out) A.sml_out[i] = hi;
            if (A.iters_out) A.iters_out[i] = A.siters[k];
            if (count > A.max_nb) set_err(A.err, ERRF_CAP_NEIGHBOURS);
        }
        unsigned long long s = (unsigned long long)wave_sum(own_list ? count : 0);
        int mx = wave_max(own_list ? count : 0);
        if (lane == 0) {
            atomicAdd(&cnt_slot(A.counters)[CNT_NEIGHBOURS], s);
            atomicMax(&cnt_slot(A.counters)[CNT_MAX_NOI], (unsigned long long)mx);
        }
    } else {
        bool stay = false;
        if (valid && !outlier) {
            if (active) {
                A.iters[k] = A.pass + 1;
                A.snoi[k] = count;
                double hn;
                const bool fin = h_update(A, count, hi, hn);
                A.h_next[k] = hn;
                if (fin) A.done[k] = 1;
                stay = !fin;
            } else {
                A.h_next[k] = hi;
            }
        }
        if (A.list_out) {
            // append the unconverged particles (wave-aggregated; list order is free, the
            // next pass's results do not depend on it)
            const uint64_t mS = wave_ballot(stay);
            uint32_t b = 0;
            if (lane == 0 && mS) b = atomicAdd(A.count_out, (uint32_t)popc64(mS));
            b = __shfl(b, 0);
            if (stay) {
                const uint32_t pos = b + popc64(mS & lanemask_lt());
                A.list_out[pos] = (int32_t)k;
                if (A.h0_slot) A.h0_slot[pos] = hi;   // the h this pass's list was built with
            }
        }
        if (lane == 0) atomicAdd(&cnt_slot(A.counters)[CNT_H_COUNTS], (unsigned long long)popc64(mActive));
    }
}

// Four wavefronts per SIMD (128 registers): free, the matrix tests would take 140 and run at two.
template <int MODE>
__global__ __launch_bounds__(64 * NN_WAVES, 4) void k_nn_walk(NNArgs A) {
    __shared__ NNWaveLdsF lds_all[NN_WAVES];
    const int w = threadIdx.x / 64;
    const int64_t group = xcd_block(blockIdx.x, gridDim.x) * NN_WAVES + w;
    if (group * 64 >= A.n) return;
    nn_group<MODE, false>(lds_all[w], A, group, 0ull);
}

// Per-particle mode: one wavefront per listed particle, searching the particle's own box
// x +- h with the 64 lanes testing 64 candidates at a time.  Used for the outliers of the
// group mode (particles whose h is far above the rest of their group) and for list fix-ups.
// MODE 1: count and h update (identical to the group mode's; the new h goes to h_next[k]);
// MODE 2: MODE 1 plus the list; MODE 0: the list only.  Lists are written in candidate
// order, one 4-byte entry per lane.
#define NN1_WAVES 4
#define NN1_MAX_BLOCKS 1024   // about one resident round: 4096 wavefronts loop over the list
// the same for the kernels that search in the direct form only: little LDS, five wavefronts a SIMD
#define NN_DIRECT_BLOCKS 1280
inline unsigned nn_direct_grid(int64_t n) { return (unsigned)std::min<int64_t>(ceil_div(n, NN1_WAVES), NN_DIRECT_BLOCKS); }
// Workgroups [first, first + blocks) of the launch.
template <int MODE>
__device__ __forceinline__ void nn_one(NNWaveLds &L, const NNArgs &A, unsigned first, unsigned blocks) {
    const int w = threadIdx.x / 64, lane = wave_lane();
    const int64_t cnt = A.list_in ? (int64_t)*A.count_in : A.n;   // no list: every particle
    const int64_t nwaves = (int64_t)blocks * NN1_WAVES;
    const uint64_t lt = lanemask_lt();
    int32_t *nbr32 = reinterpret_cast<int32_t *>(A.nbr4);
    for (int64_t t = (int64_t)(blockIdx.x - first) * NN1_WAVES + w; t < cnt; t += nwaves) {
        const int64_t k = A.list_in ? A.list_in[t] : t;
        const double4 own = A.sxm[k];
        const double hi = A.h[k];
        const double hi2 = hi * hi;
        int count = 0;
        // one candidate per lane: pair test, then the hits appended in lane order
        auto take = [&](bool v, int j, double x, double y, double z, double h2) {
            bool hit = false;
            if (v) {
                const double dx = own.x - x;
                const double dy = own.y - y;
                const double dz = own.z - z;
                const double d = nn_d2(dx, dy, dz);
                hit = d < hi2 && d < h2 && j != (int)k;
            }
            const uint64_t mh = wave_ballot(hit);
            if (MODE != 1 && hit) {
                const int s = count + popc64(mh & lt);
                if (s < A.max_nb) nbr32[((int64_t)(s >> 2) * A.stride + k) * 4 + (s & 3)] = j;
            }
            count += popc64(mh);
        };
        const bool direct = nn_direct(L.extra, A, nn_ball(own, hi),
                                      [&](bool v, int j, const double4 &p, double h) { take(v, j, p.x, p.y, p.z, h * h); });
        if (!direct) {
            const bool ok = nn_walk_box<false>(L, A, [&]() { return nn_ball(own, hi); }, NN_START_ALL, 0, 0, -1, KeepAll(), [&](int m) {
                const bool v = lane < m;
                take(v, v ? L.tj[lane] : -1, v ? L.tx[lane] : 0.0, v ? L.ty[lane] : 0.0, v ? L.tz[lane] : 0.0,
                     v ? L.th2[lane] : 0.0);
            });
            if (!ok) {
                if (lane == 0) set_err(A.err, ERRF_STACK);
                return;
            }
        }
        if (MODE == 0) {
            if (lane == 0) {
                A.snoi[k] = count;
                if (A.noi_out) A.noi_out[A.perm[k]] = count;
                if (count > A.max_nb) set_err(A.err, ERRF_CAP_NEIGHBOURS);
                if (A.counters) {
                    atomicAdd(&cnt_slot(A.counters)[CNT_NEIGHBOURS], (unsigned long long)count);
                    atomicMax(&cnt_slot(A.counters)[CNT_MAX_NOI], (unsigned long long)count);
                }
            }
        } else {
            double hn;
            const bool fin = h_update(A, count, hi, hn);
            if (lane == 0) {
                A.iters[k] = A.pass + 1;
                A.snoi[k] = count;
                A.h_next[k] = hn;
                if (fin) A.done[k] = 1;
                else {
                    const uint32_t pos = atomicAdd(A.count_out, 1u);
                    A.list_out[pos] = (int32_t)k;
                    if (A.h0_slot) A.h0_slot[pos] = hi;
                }
                atomicAdd(&cnt_slot(A.counters)[CNT_H_COUNTS], 1ull);
            }
        }
        wave_sync();
    }
}

template <int MODE>
__global__ __launch_bounds__(64 * NN1_WAVES) void k_nn_one(NNArgs A) {
    __shared__ NNWaveLds lds_all[NN1_WAVES];
    nn_one<MODE>(lds_all[threadIdx.x / 64], A, 0, gridDim.x);
}

// What a group walk left to others, in one launch: workgroups [0, part_blocks) take the parts of
// the groups it split (one wavefront each), the others the particles it deferred (k_nn_one).
template <int MODE>
__global__ __launch_bounds__(64 * NN1_WAVES) void k_nn_rest(NNArgs A, unsigned part_blocks) {
    __shared__ union Lds {
        NNWaveLds one;
        NNWaveLdsF group;
    } lds_all[NN1_WAVES];
    Lds &L = lds_all[threadIdx.x / 64];
    if (blockIdx.x < part_blocks) {
        const uint32_t cnt = *A.seg_count;
        for (int64_t t = (int64_t)blockIdx.x * NN1_WAVES + threadIdx.x / 64; t < cnt;
             t += (int64_t)part_blocks * NN1_WAVES) {
            const ulonglong2 s = A.seg_list[t];
            nn_group<MODE, true>(L.group, A, (int64_t)s.x, s.y);
            wave_sync();
        }
    } else {
        nn_one<MODE>(L.one, A, part_blocks, gridDim.x - part_blocks);
    }
}

// Dirty marking after a speculative pass 0: for every particle j whose h changed after
// pass 0 (list_in, with its pass-0 h in h0_slot), flag j and every particle i whose pair
// membership with j changed, (d < min(h_i, h_j0)) != (d < min(h_i, h_j1)) with h_j1 the final
// h: the only pairs whose membership d < h_i and d < h_j can differ from pass 0 (an unflagged
// particle keeps its pass-0 h).  Such an i lies within max(h_j0, h_j1) of x_j.  One wavefront
// per changed particle; lanes are candidates; d is the pair test's (symmetric) value.  The boxes
// the direct form declines (DIRECT) go to a second launch that walks the tree for them: the
// walk's LDS would keep half of the direct searches off the chip.
template <bool DIRECT>
__global__ __launch_bounds__(64 * NN1_WAVES) void k_nn_mark_dirty(NNArgs A) {
    using Lds = std::conditional_t<DIRECT, NNDirectLds, NNWaveLds>;
    __shared__ Lds lds_all[NN1_WAVES];
    const int w = threadIdx.x / 64, lane = wave_lane();
    Lds &L = lds_all[w];
    const uint32_t cnt = DIRECT ? *A.count_in : *A.slot_count;
    const int64_t nwaves = (int64_t)gridDim.x * NN1_WAVES;
    for (int64_t tt = (int64_t)blockIdx.x * NN1_WAVES + w; tt < cnt; tt += nwaves) {
        const int64_t t = DIRECT ? tt : A.slot_list[tt];
        const int64_t jc = A.list_in[t];
        const double4 own = A.sxm[jc];
        const double h0 = A.h0_slot[t], h1 = A.h[jc];
        const double h02 = h0 * h0, h12 = h1 * h1;
        const double hq = h0 > h1 ? h0 : h1;
        if (DIRECT && lane == 0) A.dirty[jc] = 1;
        auto mark = [&](bool v, int i, double x, double y, double z, double hi2) {
            if (v) {
                const double dx = own.x - x;
                const double dy = own.y - y;
                const double dz = own.z - z;
                const double d = nn_d2(dx, dy, dz);
                if (((d < hi2) & (d < h02)) != ((d < hi2) & (d < h12))) A.dirty[i] = 1;
            }
        };
        if constexpr (DIRECT) {
            const bool direct = nn_direct(L, A, nn_ball(own, hq),
                                          [&](bool v, int i, const double4 &p, double h) { mark(v, i, p.x, p.y, p.z, h * h); });
            if (!direct && lane == 0) A.list_out[atomicAdd(A.count_out, 1u)] = (int32_t)t;
        } else {
            const bool ok = nn_walk_box<false>(L, A, [&]() { return nn_ball(own, hq); }, NN_START_ALL, 0, 0, -1, KeepAll(), [&](int m) {
                if (lane < m) mark(true, L.tj[lane], L.tx[lane], L.ty[lane], L.tz[lane], L.th2[lane]);
            });
            if (!ok) {
                if (lane == 0) set_err(A.err, ERRF_STACK);
                return;
            }
        }
        wave_sync();
    }
}

// Counting pass of the h-iteration for the listed particles, direct form (nn_direct): one
// wavefront per particle tests every particle of the start cells of its box x +- h, with no
// tree walk.  (Sharing large boxes among several wavefronts gained 0.07 ms on an evolved state
// and cost more than that on the others: the extra wavefronts of the small boxes.)  A box the
// direct form declines (too large for the table, too many cells or candidates) is appended to
// hard_list for k_nn_count_split.  The count goes to cnt_slot[t] (integer, exact).
__global__ __launch_bounds__(64 * NN1_WAVES) void k_nn_count_direct(NNArgs A) {
    __shared__ NNDirectLds lds_all[NN1_WAVES];
    const int w = threadIdx.x / 64, lane = wave_lane();
    NNDirectLds &L = lds_all[w];
    if (h_pass_frozen(A)) return;
    const uint32_t cnt = *A.count_in;
    const int64_t nwaves = (int64_t)gridDim.x * NN1_WAVES;
    for (int64_t t = (int64_t)blockIdx.x * NN1_WAVES + w; t < cnt; t += nwaves) {
        const int64_t k = A.list_in[t];
        const double4 own = A.sxm[k];
        const double hi = A.h[k];
        const double hi2 = hi * hi;
        int count = 0;
        const bool direct = nn_direct(L, A, nn_ball(own, hi),
                                      [&](bool v, int j, const double4 &p, double h) {
            if (v) {
                const double dx = own.x - p.x;
                const double dy = own.y - p.y;
                const double dz = own.z - p.z;
                const double d = nn_d2(dx, dy, dz);
                count += (d < hi2 && d < h * h && j != (int)k) ? 1 : 0;
            }
        });
        if (!direct) {
            if (lane == 0) A.list_out[atomicAdd(A.count_out, 1u)] = (int32_t)t;   // hard_list (slots)
            continue;
        }
        count = wave_sum(count);
        if (lane == 0) A.cnt_slot[t] = (uint32_t)count;
        wave_sync();
    }
}

// Counting pass of the h-iteration for the particles the direct form left (slots in
// slot_list), split eight ways: wavefront (t, o) counts particle list_in[t]'s neighbours
// under the start cells of index = o (mod 8) (the root's child o when the box is too large
// for the start table) and adds them to cnt_slot[t] (integer sums: exact and order-free).
// A particle with a large h (a free-boundary particle whose h keeps growing) is so shared
// by eight wavefronts; k_h_finish then applies the update.
__global__ __launch_bounds__(64 * NN1_WAVES) void k_nn_count_split(NNArgs A) {
    __shared__ NNWaveLds lds_all[NN1_WAVES];
    const int w = threadIdx.x / 64, lane = wave_lane();
    NNWaveLds &L = lds_all[w];
    if (h_pass_frozen(A)) return;
    const int64_t work = 8 * (int64_t)*A.slot_count;
    const int64_t nwaves = (int64_t)gridDim.x * NN1_WAVES;
    for (int64_t tt = (int64_t)blockIdx.x * NN1_WAVES + w; tt < work; tt += nwaves) {
        const int64_t t = A.slot_list[tt >> 3];
        const int o = (int)(tt & 7);
        const int64_t k = A.list_in[t];
        const double4 own = A.sxm[k];
        const double hi = A.h[k];
        const double hi2 = hi * hi;
        const int start = NN_START_PART0 - o;   // eighth o of the start cells
        int count = 0;
        const bool ok = nn_walk_box<false>(L, A, [&]() { return nn_ball(own, hi); }, start, 0, 0, -1, KeepAll(), [&](int m) {
            bool hit = false;
            if (lane < m) {
                const double dx = own.x - L.tx[lane];
                const double dy = own.y - L.ty[lane];
                const double dz = own.z - L.tz[lane];
                const double d = nn_d2(dx, dy, dz);
                hit = d < hi2 && d < L.th2[lane] && L.tj[lane] != (int)k;
            }
            count += popc64(wave_ballot(hit));
        });
        if (!ok) {
            if (lane == 0) set_err(A.err, ERRF_STACK);
            return;
        }
        if (lane == 0 && count > 0) atomicAdd(&A.cnt_slot[t], (uint32_t)count);
        wave_sync();
    }
}

// the h update of the listed particles from their counts (after the counting pass, so every
// count saw the h of this pass; each thread writes only its own particle's h): clears
// cnt_slot for the next pass and appends the unconverged particles to list_out, a block at a time
// (every append waits for the one counter) and enough threads for one step over the first list
// (1M cloud RHS, 64 blocks and an append per wavefront / now: 5.12 / 5.03 ms)
#define H_FINISH_THREADS 256
#define H_FINISH_BLOCKS 512
__global__ __launch_bounds__(H_FINISH_THREADS) void k_h_finish(NNArgs A) {
    __shared__ uint32_t wave_stay[H_FINISH_THREADS / 64], block_pos;
    const uint32_t cnt = *A.count_in;
    const bool frozen = h_pass_frozen(A);
    const int lane = wave_lane(), w = threadIdx.x / 64;
    const uint64_t lt = lanemask_lt();
    for (int64_t t0 = blockIdx.x * (int64_t)blockDim.x; t0 < cnt; t0 += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = t0 + threadIdx.x;
        const bool valid = t < cnt;
        bool stay = false, changed = false;
        int64_t k = 0;
        double hn = 0.0;
        if (valid) {
            k = A.list_in[t];
            const int N = frozen ? A.snoi[k] : (int)A.cnt_slot[t];
            A.cnt_slot[t] = 0u;
            const double hi = A.h[k];
            const bool fin = h_update(A, N, hi, hn);
            A.iters[k] = A.pass + 1;
            A.snoi[k] = N;
            A.h_next[k] = hn;
            if (fin) A.done[k] = 1;
            stay = !fin;
            changed = stay && hn != hi;
        }
        const uint64_t mS = wave_ballot(stay);
        if (lane == 0) wave_stay[w] = (uint32_t)popc64(mS);
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int v = 0; v < H_FINISH_THREADS / 64; v++) {
            before += v < w ? wave_stay[v] : 0u;
            all += wave_stay[v];
        }
        if (threadIdx.x == 0) {
            block_pos = all != 0 ? atomicAdd(A.count_out, all) : 0u;
            const int64_t left = (int64_t)cnt - t0;
            atomicAdd(&cnt_slot(A.counters)[CNT_H_COUNTS],
                      (unsigned long long)(left < H_FINISH_THREADS ? left : H_FINISH_THREADS));
        }
        // the next pass counts with hn: the cell bounds must cover it (they cover hi)
        if (changed && A.chmax_raise) hmax_raise(A.chmax_raise, A.ppar, A.cpar, A.cap_cells, k, hn);
        if (A.changed && wave_ballot(changed) != 0 && lane == 0) *A.changed = 1u;
        __syncthreads();
        if (stay) A.list_out[block_pos + before + popc64(mS & lt)] = (int32_t)k;
    }
}

// A whole pass of the h-iteration in one launch, for few particles (NN_FEW): one wavefront per
// particle that has not finished tests every particle of the start cells of its box x +- h, with
// no tree walk (nn_direct; it declines no box of so few), and applies the h update at once.  The
// pass reads one h array and writes the other: a particle that finished holds the same h in both
// (its last count left it unchanged), so only the unfinished ones are written.  No lists: with a
// few particles per wavefront, looking at a flag costs less than appending to one counter, whose
// atomics serialise (47^3: 26 us per pass with lists appended here, 11 + 6 us with counts and a
// wave-aggregated update, so larger sets keep those).
__global__ __launch_bounds__(64 * NN1_WAVES) void k_h_pass(NNArgs A) {
    __shared__ NNDirectLds lds_all[NN1_WAVES];
    const int w = threadIdx.x / 64, lane = wave_lane();
    NNDirectLds &L = lds_all[w];
    const bool frozen = h_pass_frozen(A);
    const int64_t nwaves = (int64_t)gridDim.x * NN1_WAVES;
    bool changed = false, stays = false;
    unsigned counted = 0;
    // the wavefront's particles whose h changed (lane i holds the i-th): their cells' bounds are
    // raised together
    int32_t rk = 0;
    double rh = 0.0;
    int rn = 0;
    auto raise = [&]() {
        if (lane < rn) hmax_raise(A.chmax_raise, A.ppar, A.cpar, A.cap_cells, rk, rh);
        rn = 0;
    };
    for (int64_t t = (int64_t)blockIdx.x * NN1_WAVES + w; t < A.n; t += nwaves) {
        const int32_t k = (int32_t)t;
        if (A.done[k]) continue;
        const double hi = A.h[k];
        int N = 0;
        if (frozen) {
            N = A.snoi[k];
        } else {
            const double4 own = A.sxm[k];
            const double hi2 = hi * hi;
            const bool direct =
                nn_direct(L, A, nn_ball(own, hi), [&](bool v, int j, const double4 &p, double h) {
                    if (v) {
                        const double dx = own.x - p.x;
                        const double dy = own.y - p.y;
                        const double dz = own.z - p.z;
                        const double d = nn_d2(dx, dy, dz);
                        N += (d < hi2 && d < h * h && j != k) ? 1 : 0;
                    }
                });
            // cannot happen: no more candidates than particles, and a box spans at most the two cells
            // per axis of level 1; a count of zero instead would pass for a result
            if (!direct && lane == 0) set_err(A.err, ERRF_STACK);
            N = wave_sum(N);
            wave_sync();
        }
        counted++;
        double hn;
        const bool fin = h_update(A, N, hi, hn);
        if (lane == 0) {
            A.iters[k] = A.pass + 1;
            A.snoi[k] = N;
            A.h_next[k] = hn;
            if (fin) A.done[k] = 1;
        }
        if (fin) continue;
        stays = true;
        if (hn != hi) {   // the next pass counts with hn: the cell bounds must cover it
            changed = true;
            if (lane == rn) {
                rk = k;
                rh = hn;
            }
            if (++rn == 64) raise();
        }
    }
    raise();
    if (lane == 0) {
        if (counted != 0) atomicAdd(&cnt_slot(A.counters)[CNT_H_COUNTS], (unsigned long long)counted);
        if (stays) *A.count_out = 1u;   // not a length here: some particle goes on
        if (changed) *A.changed = 1u;
    }
}

// Start table of the current tree: a particle alone in its level-l prefix for every
// l >= its leaf level, and every cell of level <= kmax, written at their Lebesgue prefix.
__global__ __launch_bounds__(256) void k_nn_start_table(int64_t n, int kmax, const uint8_t *__restrict__ lcp,
                                                        const uint64_t *__restrict__ slkey,
                                                        const int32_t *__restrict__ cell_base,
                                                        const int32_t *__restrict__ cstart,
                                                        const int32_t *__restrict__ cend,
                                                        const int32_t *__restrict__ clevel, int64_t cap_cells,
                                                        int32_t *__restrict__ tab, int2 *__restrict__ rng) {
    // particles, then the cells of levels 1..kmax (cells are numbered level by level, so these
    // are cells 1 .. cell_base[kmax + 1] - 1); grid-stride over the actual counts
    const int64_t ncells = cell_base[MHPC_LEVELS + 1];
    if (ncells > cap_cells) return;   // capacity error already flagged; cells are incomplete
    const int64_t ctop = cell_base[kmax + 1] < ncells ? cell_base[kmax + 1] : ncells;
    const int64_t items = n + (ctop > 1 ? ctop - 1 : 0);
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < items;
         t += (int64_t)gridDim.x * blockDim.x) {
        if (t < n) {
            const int a = t > 0 ? (int)lcp[t - 1] : 0;
            const int b = (int)lcp[t];
            const int lp = (a > b ? a : b) + 1;
            const uint64_t key = slkey[t];
            for (int l = lp; l <= kmax; l++) {
                const int64_t e = nn_tab_off(l) + (int64_t)(key >> (3 * (MHPC_LEVELS - l)));
                tab[e] = (int32_t)t;
                rng[e] = make_int2((int)t, 1);
            }
        } else {
            const int64_t c = t - n + 1;   // cells 1 .. ctop-1 (cell 0 is the root)
            const int L = clevel[c];
            if (L < 1 || L > kmax) continue;
            const int32_t s0 = cstart[c];
            const int64_t e = nn_tab_off(L) + (int64_t)(slkey[s0] >> (3 * (MHPC_LEVELS - L)));
            tab[e] = (int32_t)(n + c);
            rng[e] = make_int2((int)s0, (int)(cend[c] - s0 + 1));
        }
    }
}

// cleared: the table was just emptied (with the h-iteration's flags, k_h_init)
static void ensure_nn_start(mhpc_ctx *c, bool cleared = false) {
    if (c->nn_start_valid || c->n <= 0) return;
    if (!cleared)
        launch_fill_u32(c, reinterpret_cast<uint32_t *>(c->nn_start), 0xffffffffu, nn_tab_off(c->nn_kmax + 1));
    const uint64_t *slkey = (c->p.curve == MHPC_CURVE_HILBERT) ? c->slkey : c->skey;
    const int64_t items = c->n + c->cap_cells;
    hipLaunchKernelGGL(k_nn_start_table, dim3((unsigned)std::min<int64_t>(ceil_div(items, 256), 8192)), dim3(256),
                       0, c->stream, c->n,
                       c->nn_kmax, c->lcp, slkey, c->cell_base, c->cstart, c->cend, c->clevel, c->cap_cells,
                       c->nn_start, c->nn_start_rng);
    c->nn_start_valid = true;
}

static NNArgs nn_common(mhpc_ctx *c) {
    ensure_nn_start(c);
    NNArgs a = {};
    a.stab = c->nn_start;
    a.srng = c->nn_start_rng;
    a.kmax = c->nn_kmax;
    a.box = c->box;
    a.n = c->n;
    a.perm = c->perm;
    a.sxm = c->sxm;
    a.cstart = c->cstart; a.cend = c->cend; a.cchild = c->cchild;
    a.cbmin = c->cbmin; a.cbmax = c->cbmax;
    a.cap_cells = c->cap_cells;
    a.max_nb = c->p.max_nb;
    a.err = c->err;
    a.counters = c->counters;
    a.chmax = c->chmax;
    a.lcp = c->lcp;
    return a;
}

// the split parts and the deferred particles of the group walk queued before, with its arguments:
// about one resident round of wavefronts each, looping over their lists
template <int MODE>
static void launch_nn_rest(mhpc_ctx *c, const NNArgs &a) {
    const unsigned parts = (unsigned)std::min<int64_t>(ceil_div(nn_parts_max(c->n), NN1_WAVES), NN1_MAX_BLOCKS);
    const unsigned ones = (unsigned)std::min<int64_t>(ceil_div(c->n, NN1_WAVES), NN1_MAX_BLOCKS);
    hipLaunchKernelGGL(k_nn_rest<MODE>, dim3(parts + ones), dim3(64 * NN1_WAVES), 0, c->stream, a, parts);
}
bool nn_few(const mhpc_ctx *c) { return c->n <= NN_FEW; }
static unsigned nn_grid(mhpc_ctx *c) { return (unsigned)ceil_div(ceil_div(c->n, 64), NN_WAVES); }

// done flags, iteration counts and dirty flags to zero, the walks' start table empty; the per-pass
// list counters, the per-pass changed flags and the outlier counters (pass 0, list fix-up) to zero
static_assert(offsetof(DevStatus, hchanged) == offsetof(DevStatus, hlist_count) + sizeof(DevStatus::hlist_count),
              "k_h_init zeroes the list counters and the changed flags as one range");
__global__ void k_h_init(int64_t n, uint8_t *done, int32_t *iters, uint8_t *dirty, uint32_t *list_counts,
                         int nlc, uint32_t *ocount, uint32_t *cnt_slot, uint32_t *tab, int64_t ntab) {
    int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (int64_t e = k; e < ntab; e += (int64_t)gridDim.x * blockDim.x) tab[e] = 0xffffffffu;   // empty start table
    if (k < n) {
        done[k] = 0;
        iters[k] = 0;
        dirty[k] = 0;
        cnt_slot[k] = 0u;
    }
    if (k < nlc) list_counts[k] = 0;
    if (k < 4) ocount[k] = 0;
}

// the raise for the listed particles (after pass 0: the particles still iterating are the ones
// whose h changed)
__global__ __launch_bounds__(256) void k_hmax_raise(const int32_t *__restrict__ list, const uint32_t *count,
                                                    const double *__restrict__ h, const int32_t *__restrict__ ppar,
                                                    const int32_t *__restrict__ cpar, double *chmax,
                                                    int64_t cap_cells) {
    const uint32_t cnt = *count;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < cnt; t += (int64_t)gridDim.x * blockDim.x) {
        const int32_t k = list[t];
        hmax_raise(chmax, ppar, cpar, cap_cells, k, h[k]);
    }
}

static void launch_hmax_raise(mhpc_ctx *c, const int32_t *list, const uint32_t *count) {
    hipLaunchKernelGGL(k_hmax_raise, dim3((unsigned)std::min<int64_t>(ceil_div(c->n, 1024), 512)), dim3(256), 0, c->stream, list, count, c->sh, c->ppar, c->cpar,
                       c->chmax, c->cap_cells);
}

// a9: the plain h-iteration as Jacobi passes; sh holds the final h afterwards.  Sets of up to NN_FEW
// particles take every pass per particle and write no lists (k_h_pass).  Larger ones take pass 0 in
// group mode over all particles, with the outliers and split parts behind it, and list the
// unconverged ones; later passes search per particle over that list only.
void launch_h_iterate(mhpc_ctx *c, int passes, bool speculative, hipEvent_t *walk_events) {
    if (c->n <= 0) return;
    hipLaunchKernelGGL(k_h_init, dim3((unsigned)ceil_div(c->n > 64 ? c->n : 64, 256)), dim3(256), 0, c->stream,
                       c->n, c->sdone, c->siters, c->sdirty, c->hlist_count, 3 * (MHPC_MAX_PASSES + 1), c->ocount,
                       c->hcnt, reinterpret_cast<uint32_t *>(c->nn_start),
                       c->nn_start_valid ? (int64_t)0 : nn_tab_off(c->nn_kmax + 1));
    ensure_nn_start(c, true);
    NNArgs a = nn_common(c);
    a.done = c->sdone;
    a.iters = c->siters;
    a.snoi = c->snoi;
    a.table = c->htable;
    a.tmax = MHPC_HTABLE_MAX;
    a.max_counts = passes;
    a.band_lo = c->p.band_lo;
    a.band_hi = c->p.band_hi;
    a.sml_max = c->p.sml_max;
    const unsigned g1 = (unsigned)std::min<int64_t>(ceil_div(c->n, NN1_WAVES), NN1_MAX_BLOCKS);
    if (nn_few(c)) {
        // every pass in the per-particle mode, from one h array to the other; the lists are built
        // once from the final h (launch_neighbours_fixup)
        a.chmax_raise = c->chmax;
        a.ppar = c->ppar;
        a.cpar = c->cpar;
        for (int pass = 0; pass < passes; pass++) {
            a.pass = pass;
            a.h = c->sh;
            a.h_next = c->sh2;
            a.count_out = c->hlist_count + pass;
            a.changed = c->dstatus->hchanged + pass;   // zeroed by k_h_init
            a.prev_changed = pass >= 1 ? c->dstatus->hchanged + (pass - 1) : nullptr;
            if (walk_events && pass == 0) (void)hipEventRecord(walk_events[0], c->stream);
            hipLaunchKernelGGL(k_h_pass, dim3(nn_direct_grid(c->n)), dim3(64 * NN1_WAVES), 0, c->stream, a);
            if (walk_events && pass == 0) (void)hipEventRecord(walk_events[1], c->stream);
            std::swap(c->sh, c->sh2);
        }
        return;
    }
    // pass 0, group mode; its list of unconverged particles (hlist[2]) is also the list
    // of particles whose h changed after pass 0
    a.pass = 0;
    a.h = c->sh;
    a.h_next = c->sh2;
    a.list_out = c->hlist[2];
    a.count_out = c->hlist_count + 0;
    a.h0_slot = c->h0slot;
    a.out_list = c->olist;
    a.out_count = c->ocount;   // zeroed by k_h_init
    a.seg_list = c->seglist;
    a.seg_count = c->ocount + 2;
    if (walk_events) (void)hipEventRecord(walk_events[0], c->stream);
    if (speculative) {
        a.nbr4 = reinterpret_cast<int4 *>(c->nbr);
        a.stride = c->cap_pad;
        hipLaunchKernelGGL(k_nn_walk<2>, dim3(nn_grid(c)), dim3(64 * NN_WAVES), 0, c->stream, a);
    } else {
        hipLaunchKernelGGL(k_nn_walk<1>, dim3(nn_grid(c)), dim3(64 * NN_WAVES), 0, c->stream, a);
    }
    if (walk_events) (void)hipEventRecord(walk_events[1], c->stream);
    // the group mode's split parts and outliers, same pass
    a.list_in = c->olist;
    a.count_in = c->ocount;
    if (speculative) launch_nn_rest<2>(c, a);
    else launch_nn_rest<1>(c, a);
    a.nbr4 = nullptr;
    a.out_list = nullptr;
    a.h0_slot = nullptr;   // the pass-0 slots stay for the dirty marking
    std::swap(c->sh, c->sh2);
    // the particles still iterating are the ones whose h changed
    launch_hmax_raise(c, c->hlist[2], c->hlist_count + 0);
    // passes 1.., per-particle mode over the list of the previous pass
    for (int pass = 1; pass < passes; pass++) {
        a.pass = pass;
        a.h = c->sh;
        a.list_in = pass == 1 ? c->hlist[2] : c->hlist[(pass - 1) & 1];
        a.count_in = c->hlist_count + (pass - 1);
        a.list_out = c->hlist[pass & 1];
        a.count_out = c->hlist_count + pass;
        a.h_next = c->sh;   // k_h_finish updates h in place once every count is done
        a.cnt_slot = c->hcnt;
        a.changed = c->dstatus->hchanged + pass;   // zeroed by k_h_init
        a.prev_changed = pass >= 2 ? c->dstatus->hchanged + (pass - 1) : nullptr;
        // direct counts; the particles they cannot take go to the split walk
        uint32_t *hard_count = c->hlist_count + MHPC_MAX_PASSES + 1 + pass;   // zeroed by k_h_init
        NNArgs d = a;
        d.list_out = c->hhard;
        d.count_out = hard_count;
        hipLaunchKernelGGL(k_nn_count_direct, dim3(nn_direct_grid(c->n)), dim3(64 * NN1_WAVES), 0, c->stream, d);
        a.slot_list = c->hhard;
        a.slot_count = hard_count;
        // the split work is 8 wavefronts per particle the direct form declined: usually none
        hipLaunchKernelGGL(k_nn_count_split, dim3(std::min(g1, 256u)), dim3(64 * NN1_WAVES), 0, c->stream, a);
        NNArgs f = a;
        f.chmax_raise = c->chmax;
        f.ppar = c->ppar;
        f.cpar = c->cpar;
        hipLaunchKernelGGL(k_h_finish, dim3(H_FINISH_BLOCKS), dim3(H_FINISH_THREADS), 0, c->stream, f);
    }
}

// After a speculative h-iteration (launch_h_iterate with lists from pass 0; its k_h_init
// zeroed the dirty flags and the second outlier counter): re-list exactly the particles whose
// pass-0 list may differ from the list with the final h (the changed particles and every
// particle within its own h of one).  The lists then equal those of a full list walk with the
// final h as sets (order may differ); the density kernel publishes the counts.
// For few particles the iteration built no lists: all are listed, one wavefront each.
void launch_neighbours_fixup(mhpc_ctx *c) {
    if (c->n <= 0) return;
    NNArgs a = nn_common(c);
    a.h = c->sh;
    if (nn_few(c)) {
        a.nbr4 = reinterpret_cast<int4 *>(c->nbr);
        a.stride = c->cap_pad;
        a.snoi = c->snoi;
        a.counters = nullptr;   // the density kernel counts every particle
        hipLaunchKernelGGL(k_nn_one<0>, dim3((unsigned)std::min<int64_t>(ceil_div(c->n, NN1_WAVES), NN1_MAX_BLOCKS)),
                           dim3(64 * NN1_WAVES), 0, c->stream, a);
        return;
    }
    a.list_in = c->hlist[2];
    a.count_in = c->hlist_count + 0;
    a.dirty = c->sdirty;
    a.h0_slot = c->h0slot;
    const unsigned g1 = (unsigned)std::min<int64_t>(ceil_div(c->n, NN1_WAVES), NN1_MAX_BLOCKS);
    // declined boxes: the list the counting passes used, its length in the entry pass 0 leaves unused
    a.list_out = c->hhard;
    a.count_out = c->hlist_count + MHPC_MAX_PASSES + 1;   // zeroed by k_h_init
    hipLaunchKernelGGL(k_nn_mark_dirty<true>, dim3(nn_direct_grid(c->n)), dim3(64 * NN1_WAVES), 0, c->stream, a);
    a.slot_list = c->hhard;
    a.slot_count = a.count_out;
    hipLaunchKernelGGL(k_nn_mark_dirty<false>, dim3(std::min(g1, 256u)), dim3(64 * NN1_WAVES), 0, c->stream, a);
    NNArgs b = nn_common(c);
    b.h = c->sh;
    b.nbr4 = reinterpret_cast<int4 *>(c->nbr);
    b.stride = c->cap_pad;
    b.snoi = c->snoi;
    b.only = c->sdirty;
    b.changed_count = a.count_in;
    b.out_list = c->olist;
    b.out_count = c->ocount + 1;
    b.seg_list = c->seglist;
    b.seg_count = c->ocount + 3;
    hipLaunchKernelGGL(k_nn_walk<0>, dim3(nn_grid(c)), dim3(64 * NN_WAVES), 0, c->stream, b);
    b.list_in = c->olist;
    b.count_in = c->ocount + 1;
    b.counters = nullptr;   // the density kernel counts every particle
    b.noi_out = nullptr;
    launch_nn_rest<0>(c, b);
    // h, counts and the neighbour sums go to caller order with the density kernel
    // (launch_density_eos(c, true)), which runs next and visits every particle
}

void launch_neighbours(mhpc_ctx *c) {
    if (c->n <= 0) return;
    NNArgs a = nn_common(c);
    a.h = c->sh;
    a.nbr4 = reinterpret_cast<int4 *>(c->nbr);
    a.stride = c->cap_pad;
    a.snoi = c->snoi;
    a.noi_out = c->noi;
    a.sml_out = nullptr;
    a.siters = c->siters;
    a.iters_out = nullptr;
    const unsigned g1 = (unsigned)std::min<int64_t>(ceil_div(c->n, NN1_WAVES), NN1_MAX_BLOCKS);
    if (nn_few(c)) {
        hipLaunchKernelGGL(k_nn_one<0>, dim3(g1), dim3(64 * NN1_WAVES), 0, c->stream, a);
        return;
    }
    launch_fill_u32(c, c->ocount, 0u, 4);
    a.out_list = c->olist;
    a.out_count = c->ocount;
    a.seg_list = c->seglist;
    a.seg_count = c->ocount + 2;
    hipLaunchKernelGGL(k_nn_walk<0>, dim3(nn_grid(c)), dim3(64 * NN_WAVES), 0, c->stream, a);
    a.list_in = c->olist;
    a.count_in = c->ocount;
    launch_nn_rest<0>(c, a);
}

// ------------------------------------------------------------------------------------
// a11 density (density.cu:8-72): rho_i = m_i W(0, h_i) + sum_j m_j W(r_ij, h_ij).
// Neighbour records are read as one 32-byte {x,y,z,m} plus h; the loop is unrolled so a
// wave keeps several independent gathers in flight.
#define K8PI 2.5464790894703255   // 8 / pi

// a10 cubic spline (kernel.cu:50-83), support radius h, q = r / h: W = 8/pi h^-3 w(q) with
// w = 1 + 6 q^2 (q - 1) up to q = 1/2, 2 (1 - q)^3 up to 1, and 0 beyond.  The pair loops evaluate
// both branches and select: their lanes take different ones, so a wavefront pays for both anyway.
// A NaN q selects 0 (the forces of coincident particles).
template <typename T>
__device__ __forceinline__ T cubic_w(T q) {
    const T t = T(1) - q;
    const T a = fma(T(6) * q * q, q - T(1), T(1)), b = (t + t) * (t * t);
    const T w = q <= T(0.5) ? a : b;
    return q <= T(1) ? w : T(0);
}
// (dW/dr) / r without its factor 6 * 8/pi h^-4: (3 q - 2) / h up to q = 1/2 (q / r = 1 / h), else
// -(1 - q)^2 / r
template <typename T>
__device__ __forceinline__ T cubic_grad(T q, T ih, T rinv) {
    const T t = T(1) - q;
    const T a = ih * fma(T(3), q, T(-2)), b = -(rinv * (t * t));
    const T s = q <= T(0.5) ? a : b;
    return q <= T(1) ? s : T(0);
}

// 1/x of a positive normal x from the hardware estimate (2^-23 at least) and one third-order step
// y (1 + e + e^2), e = 1 - x y: the error of a correctly rounded division (0.998 x 2^-53 largest
// over 2^20 arguments), in three instructions after the estimate.  1/sqrt(x): rsq_f64.
__device__ __forceinline__ double rcp_f64(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
}
// the same in FP32, one Newton step from the estimate: 0.5 ulp and a little
__device__ __forceinline__ float rcp_f32(float x) {
    const float y = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(y, __builtin_fmaf(-x, y, 1.f), y);
}
// n/d from the estimate of 1/d, corrected by the quotient's exact residual: 0.5 ulp and a little, in
// four instructions (a correctly rounded division takes about ten)
__device__ __forceinline__ float div_f32(float n, float d) {
    const float y = __builtin_amdgcn_rcpf(d);
    const float q = n * y;
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}
// sqrt(x), x >= 0, from the estimate of 1/sqrt(x) and its square's exact residual: 0.5 ulp and a
// little, 0 for 0; rinv receives 1/sqrt(x) to 1 ulp (large for 0).  Below the normal numbers
// (separations under 1e-19) the result is only of that size.
__device__ __forceinline__ float sqrt_f32(float x, float &rinv) {
    const float y = __builtin_amdgcn_rsqf(fmaxf(x, 1.17549435e-38f));
    const float r = x * y, half = 0.5f * y;
    rinv = __builtin_fmaf(half, __builtin_fmaf(-r, y, 1.f), y);
    return __builtin_fmaf(__builtin_fmaf(-r, r, x), half, r);
}

// a10, the five kernels of SPH::SmoothingKernel (kernel.cu:14-183, 3D branches; Dehnen & Aly
// 2012 for the Wendland functions), selected by mhpc_params.smoothing_kernel as the
// reference's Smoothing::Kernel (parameter.h:177-180).  Normalised form: for q = r/h <= 1,
// W = sigma/h^3 w(q) and dW/dr = sigma/h^4 w'(q); both are 0 beyond.  The cubic spline keeps
// its own inlined form in the density and force loops; the others go through kernel_shape.
// The Wendland C4 gradient is the reference's expression (kernel.cu:140), which is not the
// derivative of its W; it is followed as written so that results are the reference's.
__device__ __forceinline__ double kernel_sigma(int kind) {
    switch (kind) {
        case MHPC_KERNEL_SPIKY: return 15.0 / M_PI;
        case MHPC_KERNEL_WENDLAND_C2: return 21.0 / (2.0 * M_PI);
        case MHPC_KERNEL_WENDLAND_C4: return 495.0 / (32.0 * M_PI);
        case MHPC_KERNEL_WENDLAND_C6: return 1365.0 / (64.0 * M_PI);
        default: return 8.0 / M_PI;
    }
}

template <typename T>
__device__ __forceinline__ void kernel_shape(int kind, T q, T &w, T &dw) {
    const T t = T(1) - q;
    const T t2 = t * t, t3 = t2 * t;
    switch (kind) {
        case MHPC_KERNEL_SPIKY:
            w = t3;
            dw = T(-3) * t2;
            break;
        case MHPC_KERNEL_WENDLAND_C2:
            w = t2 * t2 * (T(1) + T(4) * q);
            dw = T(-20) * q * t3;
            break;
        case MHPC_KERNEL_WENDLAND_C4:
            w = t3 * t3 * (T(1) + q * (T(6) + T(35.0 / 3.0) * q));
            dw = T(-6) * t3 * t2 * (T(1) + q * q * (T(-35) + T(105) * q));
            break;
        case MHPC_KERNEL_WENDLAND_C6:
            w = t2 * t2 * t2 * t2 * (T(1) + q * (T(8) + q * (T(25) + T(32) * q)));
            dw = T(-22) * q * t3 * t2 * t2 * (T(1) + q * (T(7) + T(16) * q));
            break;
        default:   // cubic spline
            if (q <= T(0.5)) {
                w = T(1) + T(6) * q * q * (q - T(1));
                dw = T(6) * q * (T(3) * q - T(2));
            } else {
                w = T(2) * t3;
                dw = T(-6) * t2;
            }
            break;
    }
}

// ------------------------------------------------------------------------------------
// a12 / a13 sound speed (soundspeed.cu:38-97) and pressure (pressure.cu:6-87), fused;
// also writes the records the force loop gathers: cs into {vx,vy,vz,cs} and
// {rho, p/rho^2, m/rho, h}.
// cs_const > 0: the constant sound speed of MHPC_EOS_ISOTHERMAL_CONST_CS (otherwise that EOS
// keeps each particle's uploaded cs)
__device__ __forceinline__ double eos_cs(int eos, double gamma, double K, double cs_const, double rho, double p,
                                         double cs) {
    switch (eos) {
        case MHPC_EOS_POLYTROPIC: return sqrt(K * pow(rho, gamma - 1.0));
        case MHPC_EOS_IDEAL_GAS: return sqrt(gamma * p / rho);
        case MHPC_EOS_LOCALLY_ISOTHERMAL: return 0.0;
        case MHPC_EOS_ISOTHERMAL_CONST_CS: return cs_const > 0.0 ? cs_const : cs;
        default: return cs;
    }
}

__device__ __forceinline__ double eos_p(int eos, double gamma, double K, double rho, double e,
                                        double cs) {
    switch (eos) {
        case MHPC_EOS_POLYTROPIC: return K * pow(rho, gamma);
        case MHPC_EOS_ISOTHERMAL: return 41255.407 * rho;
        case MHPC_EOS_IDEAL_GAS: return (gamma - 1) * rho * e;
        case MHPC_EOS_LOCALLY_ISOTHERMAL:
        case MHPC_EOS_ISOTHERMAL_CONST_CS: return cs * cs * rho;
        default: return 0.0;
    }
}

// EOS of one particle and the records the force loop reads (shared by k_eos and the
// density kernel's fused form)
struct EosArgs {
    int eos, cs_before_p;
    double gamma, K, cs_const;
    const double *se;
    double *sp, *scs;
    double4 *sv4, *sr4;
    double *p_out, *cs_out;
};

__device__ __forceinline__ void eos_particle(const EosArgs &E, int64_t k, int32_t i, double rho, double m,
                                             double h) {
    const double e = E.se[k];
    double p = E.sp[k], cs = E.scs[k];
    if (E.eos == MHPC_EOS_ISOTHERMAL_CONST_CS) cs = eos_cs(E.eos, E.gamma, E.K, E.cs_const, rho, p, cs);
    if (E.cs_before_p) {
        cs = eos_cs(E.eos, E.gamma, E.K, E.cs_const, rho, p, cs);
        p = eos_p(E.eos, E.gamma, E.K, rho, e, cs);
    } else {
        p = eos_p(E.eos, E.gamma, E.K, rho, e, cs);
        cs = eos_cs(E.eos, E.gamma, E.K, E.cs_const, rho, p, cs);
    }
    E.sp[k] = p;
    E.scs[k] = cs;
    E.sv4[k].w = cs;
    E.sr4[k] = make_double4(rho, p / (rho * rho), m / rho, h);
    E.p_out[i] = p;
    E.cs_out[i] = cs;
}

static EosArgs eos_args(mhpc_ctx *c) {
    EosArgs E;
    E.eos = c->p.eos;
    E.cs_before_p = c->p.cs_before_p;
    E.gamma = c->p.gamma;
    E.K = c->p.K;
    E.cs_const = c->p.cs_const;
    E.se = c->se;
    E.sp = c->sp;
    E.scs = c->scs;
    E.sv4 = c->sv4;
    E.sr4 = c->sr4;
    E.p_out = c->f[MHPC_F_P];
    E.cs_out = c->f[MHPC_F_CS];
    return E;
}

// one density pair term m_j W added into acc.  FP32: W in FP32 from FP64 differences, without the
// kernel's constant (density_sum puts it in), times the FP64 mass: a rounded constant or mass is the
// same error in every term (8/pi: -4.0e-8 of the density), and with these gone an FP64 sum costs no
// more than a compensated one.
template <bool FP64, bool CUBIC>
__device__ __forceinline__ void density_pair(const double4 &pi, double hi, const double4 &pj, double hj,
                                             int sml_avg, int kind, double &acc) {
    const double hb = sml_avg ? 0.5 * (hi + hj) : hi;
    if constexpr (FP64) {
        const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        const double ih = rcp_f64(hb);
        const double q = fmax(r2 * rsq_f64(r2) * ih, 0.0);   // r = 0: 0 inf, no number, to 0
        const double ih3 = ih * ih * ih;
        if constexpr (CUBIC) {
            acc = fma(pj.w * (K8PI * ih3), cubic_w(q), acc);
        } else if (q <= 1.0) {
            double w, dw;
            kernel_shape<double>(kind, q, w, dw);
            acc = fma(pj.w, kernel_sigma(kind) * ih3 * w, acc);
        }
    } else {
        const float dx = (float)(pi.x - pj.x), dy = (float)(pi.y - pj.y), dz = (float)(pi.z - pj.z);
        const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
        const float ih = rcp_f32((float)hb);
        float rinv;
        const float q = sqrt_f32(r2, rinv) * ih;
        const float ih3 = ih * ih * ih;
        if constexpr (CUBIC) {
            acc = fma(pj.w, (double)(ih3 * cubic_w(q)), acc);
        } else if (q <= 1.0f) {
            float w, dw;
            kernel_shape<float>(kind, q, w, dw);
            acc = fma(pj.w, (double)(ih3 * w), acc);
        }
    }
}
template <bool FP64, bool CUBIC>
__device__ __forceinline__ double density_sum(int kind, double acc) {
    return FP64 ? acc : acc * (CUBIC ? K8PI : kernel_sigma(kind));
}

// caller-order h, neighbour and iteration counts and the neighbour sum / maximum, published by
// the density kernel when noi is set (the RHS with lists from pass 0, after the list fix-up)
struct DensPub {
    const int32_t *siters;
    double *sml;
    int32_t *noi, *iters;
    unsigned long long *counters;
};

// Neighbour window.  Per-lane gathers of neighbour records are bound by the L1 address path
// (each 16-byte load of a wave touches ~50 distinct cache lines).  A block covers a
// contiguous range of sorted particles -- a compact region of the curve -- and stages that
// range's records in LDS: a neighbour j inside the window is read from LDS at j - base (no
// lookup), the others are gathered (the masked loads of the out-of-window lanes are all the
// address path sees).  On a lattice 67 % of the pairs fall in a 512-particle window and 58 %
// in a 256-particle one.  Same arithmetic and order as a pure gather.
#define DENS_WIN 512
// Up to this many particles a list is shared by 16 lanes instead (k_density_split,
// k_forces_split): RHS of 31^3 598 -> 558 us, of 36^3 625 -> 605 us, but of 45^3 712 -> 738 us,
// where the windows' saved gathers count more than idle lanes
#define SPLIT_MAX 49152

// EOS: the sound speed / pressure of the particle follow in the same kernel (the RHS path)
template <bool FP64, bool EOS, bool CUBIC>
__global__ __launch_bounds__(DENS_WIN) void k_density(int64_t n, const double4 *__restrict__ sxm,
                                                      const double *__restrict__ sh,
                                                      const int32_t *__restrict__ snoi,
                                                      const int32_t *__restrict__ nbr, int64_t stride,
                                                      int max_nb, int sml_avg, int kind,
                                                      const int32_t *__restrict__ perm,
                                                      double *__restrict__ srho, double *__restrict__ rho,
                                                      uint32_t *err, EosArgs E, DensPub P) {
    __shared__ double4 wp[DENS_WIN];
    __shared__ double wh[DENS_WIN];
    const int64_t base = xcd_block(blockIdx.x, gridDim.x) * (int64_t)DENS_WIN;
    const int tid = threadIdx.x;
    const int64_t k = base + tid;
    if (k < n) {
        wp[tid] = sxm[k];
        wh[tid] = sh[k];
    }
    __syncthreads();
    int pub_cnt = 0;   // the neighbour count this thread publishes (0 beyond n)
    if (k < n) {
        const double4 pi = wp[tid];
        const double hi = wh[tid];
        int cnt = snoi[k];
        cnt = cnt > max_nb ? max_nb : cnt;
        const int4 *nrow = reinterpret_cast<const int4 *>(nbr) + k;   // row r at nrow[r * stride]
        double acc = 0.0;
        // two list rows (eight neighbours) per iteration: the eight records are requested
        // together, then the pairs are evaluated in list order; the next two rows are
        // requested a step ahead.  The window copy is read unconditionally (clamped index),
        // the gather only where j is outside the window.
        int4 qn0 = make_int4(0, 0, 0, 0), qn1 = qn0;
        if (cnt > 0) qn0 = nrow[0];
        if (cnt > 4) qn1 = nrow[stride];
        for (int r = 0; 4 * r < cnt; r += 2) {
            const int4 qa = qn0, qb = qn1;
            const int m = cnt - 4 * r;   // entries left (>= 1)
            if (m > 8) qn0 = nrow[(int64_t)(r + 2) * stride];
            if (m > 12) qn1 = nrow[(int64_t)(r + 3) * stride];
            const int32_t jj[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
            double4 pj[8];
            double hj[8];
    #pragma unroll
            for (int e = 0; e < 8; e++) {
                const int32_t j = e < m ? jj[e] : (int32_t)k;
                const uint32_t o = (uint32_t)(j - (int32_t)base);
                const bool in = o < (uint32_t)DENS_WIN;
                const int oc = in ? (int)o : 0;
                pj[e] = wp[oc];
                hj[e] = wh[oc];
                if (!in) {
                    pj[e] = sxm[j];
                    hj[e] = sh[j];
                }
            }
    #pragma unroll
            for (int e = 0; e < 8; e++)
                if (e < m) density_pair<FP64, CUBIC>(pi, hi, pj[e], hj[e], sml_avg, kind, acc);
        }
        const double self = CUBIC ? K8PI / (hi * hi * hi) : kernel_sigma(kind) / (hi * hi * hi);   // W(0)
        const double r = pi.w * self + density_sum<FP64, CUBIC>(kind, acc);
        srho[k] = r;
        const int32_t i = perm[k];
        rho[i] = r;
        if (!(r > 0.0)) set_err(err, ERRF_RHO);
        if (EOS) eos_particle(E, k, i, r, pi.w, hi);
        if (P.noi) {
            pub_cnt = snoi[k];
            P.noi[i] = pub_cnt;
            P.sml[i] = hi;
            P.iters[i] = P.siters[k];
        }
    }
    if (P.noi) {
        // every thread of the block takes part: one sum / max and one pair of atomics per block
        // (a pair per wavefront would queue tens of thousands of atomics on one address)
        __shared__ unsigned long long psum[DENS_WIN / 64];
        __shared__ int pmax[DENS_WIN / 64];
        const unsigned long long sum = wave_sum((unsigned long long)pub_cnt);
        const int mx = wave_max(pub_cnt);
        if (wave_lane() == 0) {
            psum[tid / 64] = sum;
            pmax[tid / 64] = mx;
        }
        __syncthreads();
        if (tid == 0) {
            unsigned long long t = 0;
            int m = 0;
            for (int w = 0; w < DENS_WIN / 64; w++) {
                t += psum[w];
                m = pmax[w] > m ? pmax[w] : m;
            }
            atomicAdd(&cnt_slot(P.counters)[CNT_NEIGHBOURS], t);
            atomicMax(&cnt_slot(P.counters)[CNT_MAX_NOI], (unsigned long long)m);
        }
    }
}

// The same for few particles: 16 lanes per particle, each taking every 16th list row (four
// neighbours), their sums added across the lanes; neighbours are gathered (no window).  With one
// lane per particle, 4096 particles are eight workgroups whose lanes walk their lists alone
// (30 us; this 7 us).
#define SPLIT_LANES 16
template <bool FP64, bool EOS, bool CUBIC>
__global__ __launch_bounds__(256) void k_density_split(int64_t n, const double4 *__restrict__ sxm,
                                                       const double *__restrict__ sh,
                                                       const int32_t *__restrict__ snoi,
                                                       const int32_t *__restrict__ nbr, int64_t stride, int max_nb,
                                                       int sml_avg, int kind, const int32_t *__restrict__ perm,
                                                       double *__restrict__ srho, double *__restrict__ rho,
                                                       uint32_t *err, EosArgs E, DensPub P) {
    const int64_t k = xcd_block(blockIdx.x, gridDim.x) * (256 / SPLIT_LANES) + threadIdx.x / SPLIT_LANES;
    const int sub = threadIdx.x % SPLIT_LANES;
    double sum = 0.0, hi = 0.0;
    double4 pi = make_double4(0.0, 0.0, 0.0, 0.0);
    int noi = 0;
    if (k < n) {
        pi = sxm[k];
        hi = sh[k];
        noi = snoi[k];
        const int cnt = noi > max_nb ? max_nb : noi;
        const int4 *nrow = reinterpret_cast<const int4 *>(nbr) + k;
        double acc = 0.0;
        for (int r = sub; 4 * r < cnt; r += SPLIT_LANES) {
            const int4 q = nrow[(int64_t)r * stride];
            const int m = cnt - 4 * r;
            const int32_t jj[4] = {q.x, q.y, q.z, q.w};
            double4 pj[4];
            double hj[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int32_t j = e < m ? jj[e] : (int32_t)k;
                pj[e] = sxm[j];
                hj[e] = sh[j];
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (e < m) density_pair<FP64, CUBIC>(pi, hi, pj[e], hj[e], sml_avg, kind, acc);
        }
        sum = density_sum<FP64, CUBIC>(kind, acc);
    }
    sum = row_sum(sum);
    if (k < n && sub == 0) {
        const double self = CUBIC ? K8PI / (hi * hi * hi) : kernel_sigma(kind) / (hi * hi * hi);   // W(0)
        const double r = pi.w * self + sum;
        srho[k] = r;
        const int32_t i = perm[k];
        rho[i] = r;
        if (!(r > 0.0)) set_err(err, ERRF_RHO);
        if (EOS) eos_particle(E, k, i, r, pi.w, hi);
        if (P.noi) {
            P.noi[i] = noi;
            P.sml[i] = hi;
            P.iters[i] = P.siters[k];
        }
    }
    if (P.noi) {
        const unsigned long long tot = wave_sum((unsigned long long)(sub == 0 ? noi : 0));
        const int mx = wave_max(noi);
        if (wave_lane() == 0) {
            atomicAdd(&cnt_slot(P.counters)[CNT_NEIGHBOURS], tot);
            atomicMax(&cnt_slot(P.counters)[CNT_MAX_NOI], (unsigned long long)mx);
        }
    }
}

template <bool FP64, bool EOS>
static void launch_density_p(mhpc_ctx *c, const EosArgs &E, const DensPub &P) {
    const bool cubic = c->p.smoothing_kernel == MHPC_KERNEL_CUBIC_SPLINE;
    const bool split = c->n <= SPLIT_MAX;
    auto kernel = split ? (cubic ? k_density_split<FP64, EOS, true> : k_density_split<FP64, EOS, false>)
                        : (cubic ? k_density<FP64, EOS, true> : k_density<FP64, EOS, false>);
    const unsigned threads = split ? 256 : DENS_WIN;
    const unsigned g = (unsigned)ceil_div(c->n * (split ? SPLIT_LANES : 1), threads);
    hipLaunchKernelGGL(kernel, dim3(g), dim3(threads), 0, c->stream, c->n, c->sxm, c->sh, c->snoi, c->nbr, c->cap_pad,
                       c->p.max_nb, c->p.sml_avg, c->p.smoothing_kernel, c->perm, c->srho, c->f[MHPC_F_RHO], c->err, E,
                       P);
}

template <bool EOS>
static void launch_density_t(mhpc_ctx *c, bool publish) {
    if (c->n <= 0) return;
    const EosArgs E = eos_args(c);
    DensPub P = {};
    if (publish) P = DensPub{c->siters, c->f[MHPC_F_SML], c->noi, c->h_iters, c->counters};
    if (c->p.precision == MHPC_PREC_FP64) launch_density_p<true, EOS>(c, E, P);
    else launch_density_p<false, EOS>(c, E, P);
}

void launch_density(mhpc_ctx *c) { launch_density_t<false>(c, false); }

void launch_density_eos(mhpc_ctx *c, bool publish) { launch_density_t<true>(c, publish); }

__global__ __launch_bounds__(256) void k_eos(int64_t n, EosArgs E, const double *__restrict__ srho,
                                             const double4 *__restrict__ sxm, const double *__restrict__ sh,
                                             const int32_t *__restrict__ perm) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= n) return;
    eos_particle(E, k, perm[k], srho[k], sxm[k].w, sh[k]);
}

void launch_eos(mhpc_ctx *c) {
    if (c->n <= 0) return;
    hipLaunchKernelGGL(k_eos, dim3((unsigned)ceil_div(c->n, 256)), dim3(256), 0, c->stream, c->n, eos_args(c),
                       c->srho, c->sxm, c->sh, c->perm);
}

// ------------------------------------------------------------------------------------
// a14 internal forces (internal_forces.cu:4-668): SPH_EQU_VERSION 1 pressure term,
// Monaghan viscosity, drho/dt, de/dt (INTEGRATE_ENERGY), dh/dt (INTEGRATE_SML).
// Per pair: grad W = dW/dr (r_ij / r); pressure factor pf = -m_j (p_i/rho_i^2 +
// p_j/rho_j^2); a_i += (pf - m_j Pi_ij) grad W; drho_i += rho_i (m_j/rho_j) v_ij.gradW;
// dh_i -= h_i/3 (m_j/rho_j) v_ij.gradW; de_i += 1/2 (m_j Pi_ij - pf) v_ij.gradW (the
// reference's 1/2 m_j Pi v.gradW + 1/2 a^p_ij . (-v_ij), with a^p_ij = pf gradW).
struct ForceArgs {
    int64_t n;
    const double4 *sxm, *sv4, *sr4;
    const double *sh;
    const int32_t *snoi, *nbr;
    int64_t stride;
    int max_nb, sml_avg, kind;
    double alpha, beta;
    const int32_t *perm;
    double *ax, *ay, *az, *drhodt, *dedt, *dsmldt, *muijmax;
    double *curlv, *gradrho;   // learned-h features (FEAT)
};

// Per-lane force accumulators.  FEAT also accumulates curl v = sum (m_j/rho_j) grad W x
// (v_j - v_i) and grad rho = sum m_j grad W, the learned-h features (plain sums in the pair
// precision).
template <bool FP64>
struct ForceAcc;
template <>
struct ForceAcc<true> {
    double a0 = 0, a1 = 0, a2 = 0, dvv = 0, de = 0;
};
template <>
struct ForceAcc<false> {
    Kahan a0, a1, a2, dvv, de;
};

struct ForceI {   // particle i's data and the constants of the pair loop
    double4 p, v, r;
    double h;
    int sml_avg, kind;
    double alpha, beta;
};

// one pair (i, j) of the force loop; j's records {x,y,z,m}, {vx,vy,vz,cs},
// {rho, p/rho^2, m/rho, h}.  The loop is bound by its instructions as much as by its gathers, so
// every shared factor is taken out: with grad W = gs r_ij, v.grad W = gs (v.r_ij) and the
// acceleration is (fa gs) r_ij; the viscosity Pi_ij = (beta mu - alpha c) mu / rho with
// mu = h v.r / D, D = r^2 + 0.01 h^2, is taken in FP64 as one quotient over D^2 rho (two reciprocals
// fewer instructions than dividing by D and by rho).  112 -> 96 vector instructions per FP64 pair
// (256^3 RHS 18.1 -> 17.9 ms).  In FP32 numerator and D^2, which grow like h^4, would leave the
// range in which every other term of the pair stays (h of 50 km in metres): there mu, of the size of
// v, is formed first.
// mu is negative wherever it is used, so the largest mu_ij, which starts at 0
// (internal_forces.cu:135, :383-385), is always 0.
template <bool FP64, bool FEAT, bool CUBIC>
__device__ __forceinline__ void force_pair(const ForceI &I, const double4 &pj, const double4 &vj, const double4 &rj,
                                           ForceAcc<FP64> &acc, double *feat) {
    typedef typename std::conditional<FP64, double, float>::type T;
    const double4 pi = I.p, vi = I.v, ri = I.r;
    const T hs = (T)(I.h + rj.w);
    const T hb = T(0.5) * hs;
    const T sml = I.sml_avg ? hb : (T)I.h;
    const T d0 = (T)(pi.x - pj.x), d1 = (T)(pi.y - pj.y), d2 = (T)(pi.z - pj.z);
    const T v0 = (T)(vi.x - vj.x), v1 = (T)(vi.y - vj.y), v2 = (T)(vi.z - vj.z);
    const T r2 = fma(d0, d0, fma(d1, d1, d2 * d2));
    T rinv, ih, q;
    if constexpr (FP64) {
        rinv = rsq_f64(r2);
        ih = rcp_f64(sml);
        q = r2 * rinv * ih;
    } else {
        ih = rcp_f32(sml);
        q = sqrt_f32(r2, rinv) * ih;
    }
    const T ih2 = ih * ih;
    // grad W = gs r_ij, gs = (dW/dr) / r; in FP32 without the kernel's constant, which multiplies the
    // sums instead (ForceSums): rounded, it would be the same error in every term
    T gs = T(0);
    if constexpr (CUBIC) {
        const T norm = FP64 ? T(6 * K8PI) * (ih2 * ih2) : ih2 * ih2;
        gs = norm * cubic_grad(q, ih, rinv);
    } else if (q <= T(1) && r2 > T(0)) {
        T w, dw;
        kernel_shape<T>(I.kind, q, w, dw);
        gs = (FP64 ? (T)kernel_sigma(I.kind) : T(1)) * (ih2 * ih2) * dw * rinv;
    }
    const T vr = fma(v0, d0, fma(v1, d1, v2 * d2));
    const T mj = (T)pj.w;
    // Pi_ij = (beta mu - alpha c) mu / rho, mu = h v.r / D, c and rho the pair's means
    const T D = fma(hb * hb, T(1e-2), r2);
    T mpij;
    if constexpr (FP64) {
        // m (2 h v.r) (beta/2 (2 h v.r) - alpha c D) / (D^2 (rho_i + rho_j))
        const T x = hs * vr;
        const T cD = T(0.5) * (vi.w + vj.w) * D;
        const T num = mj * x * fma(T(0.5) * I.beta, x, -I.alpha * cD);
        mpij = num * rcp_f64(D * D * (ri.x + rj.x));
    } else {
        const T mu = div_f32(hb * vr, D);
        const T c = T(0.5) * (T)(vi.w + vj.w), rho = T(0.5) * (T)(ri.x + rj.x);
        mpij = div_f32(mj * fma((T)I.beta, mu, -(T)I.alpha * c) * mu, rho);
    }
    mpij = vr < T(0) ? mpij : T(0);
    const T pf = -mj * (T)(ri.y + rj.y);
    const T f = pf - mpij;
    if constexpr (FP64) {
        const T vv = gs * vr, fa = f * gs;   // vv = v.grad W
        acc.a0 = fma(fa, d0, acc.a0);
        acc.a1 = fma(fa, d1, acc.a1);
        acc.a2 = fma(fa, d2, acc.a2);
        acc.dvv = fma(rj.z, vv, acc.dvv);   // the drho/dt and dh/dt sums are the same sum
        acc.de = fma(-f, vv, acc.de);
    } else {
        // v.grad W from the rounded components: the roundings of the three products are independent
        // (de/dt, rms error over 2.4e5 particles: 1.59e-7, as gs (v.r_ij) 1.66e-7)
        const T g0 = gs * d0, g1 = gs * d1, g2 = gs * d2;
        const T vv = fma(v0, g0, fma(v1, g1, v2 * g2));
        acc.a0.add(f * g0);
        acc.a1.add(f * g1);
        acc.a2.add(f * g2);
        acc.dvv.add((T)rj.z * vv);
        acc.de.add(-f * vv);
    }
    if (FEAT) {
        const T rg = (T)rj.z * gs, mg = mj * gs;
        feat[0] += rg * (v1 * d2 - v2 * d1);
        feat[1] += rg * (v2 * d0 - v0 * d2);
        feat[2] += rg * (v0 * d1 - v1 * d0);
        feat[3] += mg * d0;
        feat[4] += mg * d1;
        feat[5] += mg * d2;
    }
}

// a particle's accumulated sums (drho/dt and dh/dt share one)
struct ForceSums {
    double a[3], dvv, de, feat[6];
    __device__ __forceinline__ void take(const ForceAcc<true> &s, const double *f, double) {
        a[0] = s.a0; a[1] = s.a1; a[2] = s.a2;
        dvv = s.dvv;
        de = s.de;
        for (int q = 0; q < 6; q++) feat[q] = f[q];
    }
    // c: the kernel's constant, left out of the FP32 terms
    __device__ __forceinline__ void take(const ForceAcc<false> &s, const double *f, double c) {
        a[0] = c * s.a0.value(); a[1] = c * s.a1.value(); a[2] = c * s.a2.value();
        dvv = c * s.dvv.value();
        de = c * s.de.value();
        for (int q = 0; q < 6; q++) feat[q] = c * f[q];
    }
};

template <bool FEAT>
__device__ __forceinline__ void force_store(const ForceArgs &A, int64_t k, const ForceI &I, const ForceSums &S) {
    const int32_t i = A.perm[k];
    A.ax[i] = S.a[0];
    A.ay[i] = S.a[1];
    A.az[i] = S.a[2];
    A.drhodt[i] = I.r.x * S.dvv;
    A.dedt[i] = 0.5 * S.de;
    A.dsmldt[i] = -(1.0 / 3.0) * I.h * S.dvv;
    A.muijmax[i] = 0.0;   // see force_pair
    if (FEAT) {
        const double *f = S.feat;
        A.curlv[i] = sqrt(f[0] * f[0] + f[1] * f[1] + f[2] * f[2]);
        A.gradrho[i] = sqrt(f[3] * f[3] + f[4] * f[4] + f[5] * f[5]);
    }
}

// One block per window of FORCE_WIN consecutive sorted particles, their records staged in
// LDS (see the density kernel): in-window neighbours are read there, the others gathered.
#define FORCE_WIN 512
static_assert(FORCE_WIN == NN_CWIN && DENS_WIN == NN_CWIN, "lists hold the neighbours of the consumers' window first");

template <bool FP64, bool FEAT, bool CUBIC>
__global__ __launch_bounds__(FORCE_WIN) void k_forces(ForceArgs A) {
    __shared__ double4 wp[FORCE_WIN], wv[FORCE_WIN], wr[FORCE_WIN];
    const int64_t base = xcd_block(blockIdx.x, gridDim.x) * (int64_t)FORCE_WIN;
    const int tid = threadIdx.x;
    const int64_t k = base + tid;
    if (k < A.n) {
        wp[tid] = A.sxm[k];
        wv[tid] = A.sv4[k];
        wr[tid] = A.sr4[k];
    }
    __syncthreads();
    if (k >= A.n) return;
    ForceI I;
    I.p = wp[tid];
    I.v = wv[tid];
    I.r = wr[tid];
    I.h = A.sh[k];
    I.sml_avg = A.sml_avg;
    I.kind = A.kind;
    I.alpha = A.alpha;
    I.beta = A.beta;
    int cnt = A.snoi[k];
    cnt = cnt > A.max_nb ? A.max_nb : cnt;
    ForceAcc<FP64> acc;
    double feat[6] = {0, 0, 0, 0, 0, 0};
    const int4 *nrow = reinterpret_cast<const int4 *>(A.nbr) + k;   // row r at nrow[r * stride]
    const int64_t stride = A.stride;
    // two neighbours per step, both requested before either pair is evaluated (see the
    // density kernel); list rows a row ahead
    int4 qn = make_int4(0, 0, 0, 0);
    if (cnt > 0) qn = nrow[0];
    for (int r = 0; 4 * r < cnt; r++) {
        const int4 q4 = qn;
        const int m = cnt - 4 * r;
        if (m > 4) qn = nrow[(int64_t)(r + 1) * stride];
        const int32_t jj[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
        for (int h = 0; h < 4; h += 2) {
            double4 pj[2], vj[2], rj[2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int32_t j = h + e < m ? jj[h + e] : (int32_t)k;
                const uint32_t o = (uint32_t)(j - (int32_t)base);
                const bool in = o < (uint32_t)FORCE_WIN;
                const int oc = in ? (int)o : 0;
                pj[e] = wp[oc];
                vj[e] = wv[oc];
                rj[e] = wr[oc];
                if (!in) {
                    pj[e] = A.sxm[j];
                    vj[e] = A.sv4[j];
                    rj[e] = A.sr4[j];
                }
            }
#pragma unroll
            for (int e = 0; e < 2; e++)
                if (h + e < m) force_pair<FP64, FEAT, CUBIC>(I, pj[e], vj[e], rj[e], acc, feat);
        }
    }
    ForceSums S;
    S.take(acc, feat, CUBIC ? 6 * K8PI : kernel_sigma(I.kind));
    force_store<FEAT>(A, k, I, S);
}

// the same for few particles, 16 lanes per particle (see k_density_split; 4096 particles: 49 -> 6 us)
template <bool FP64, bool FEAT, bool CUBIC>
__global__ __launch_bounds__(256) void k_forces_split(ForceArgs A) {
    const int64_t k = xcd_block(blockIdx.x, gridDim.x) * (256 / SPLIT_LANES) + threadIdx.x / SPLIT_LANES;
    const int sub = threadIdx.x % SPLIT_LANES;
    ForceAcc<FP64> acc;
    double feat[6] = {0, 0, 0, 0, 0, 0};
    ForceI I = {};
    if (k < A.n) {
        I.p = A.sxm[k];
        I.v = A.sv4[k];
        I.r = A.sr4[k];
        I.h = A.sh[k];
        I.sml_avg = A.sml_avg;
        I.kind = A.kind;
        I.alpha = A.alpha;
        I.beta = A.beta;
        int cnt = A.snoi[k];
        cnt = cnt > A.max_nb ? A.max_nb : cnt;
        const int4 *nrow = reinterpret_cast<const int4 *>(A.nbr) + k;
        for (int r = sub; 4 * r < cnt; r += SPLIT_LANES) {
            const int4 q = nrow[(int64_t)r * A.stride];
            const int m = cnt - 4 * r;
            const int32_t jj[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int h = 0; h < 4; h += 2) {
                double4 pj[2], vj[2], rj[2];
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int32_t j = h + e < m ? jj[h + e] : (int32_t)k;
                    pj[e] = A.sxm[j];
                    vj[e] = A.sv4[j];
                    rj[e] = A.sr4[j];
                }
#pragma unroll
                for (int e = 0; e < 2; e++)
                    if (h + e < m) force_pair<FP64, FEAT, CUBIC>(I, pj[e], vj[e], rj[e], acc, feat);
            }
        }
    }
    ForceSums S;
    S.take(acc, feat, CUBIC ? 6 * K8PI : kernel_sigma(I.kind));
#pragma unroll
    for (int q = 0; q < 3; q++) S.a[q] = row_sum(S.a[q]);
    S.dvv = row_sum(S.dvv);
    S.de = row_sum(S.de);
    if (FEAT)
#pragma unroll
        for (int q = 0; q < 6; q++) S.feat[q] = row_sum(S.feat[q]);
    if (k < A.n && sub == 0) force_store<FEAT>(A, k, I, S);
}

template <bool FP64, bool FEAT>
static void launch_forces_p(mhpc_ctx *c, const ForceArgs &a) {
    const bool cubic = a.kind == MHPC_KERNEL_CUBIC_SPLINE;
    const bool split = c->n <= SPLIT_MAX;
    auto kernel = split ? (cubic ? k_forces_split<FP64, FEAT, true> : k_forces_split<FP64, FEAT, false>)
                        : (cubic ? k_forces<FP64, FEAT, true> : k_forces<FP64, FEAT, false>);
    const unsigned threads = split ? 256 : FORCE_WIN;
    hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(c->n * (split ? SPLIT_LANES : 1), threads)), dim3(threads), 0,
                       c->stream, a);
}

void launch_forces(mhpc_ctx *c, bool features) {
    if (c->n <= 0) return;
    ForceArgs a;
    a.n = c->n;
    a.sxm = c->sxm; a.sv4 = c->sv4; a.sr4 = c->sr4; a.sh = c->sh;
    a.snoi = c->snoi; a.nbr = c->nbr; a.stride = c->cap_pad;
    a.max_nb = c->p.max_nb; a.sml_avg = c->p.sml_avg; a.kind = c->p.smoothing_kernel;
    a.alpha = c->p.alpha; a.beta = c->p.beta;
    a.perm = c->perm;
    a.ax = c->f[MHPC_F_AX]; a.ay = c->f[MHPC_F_AY]; a.az = c->f[MHPC_F_AZ];
    a.drhodt = c->f[MHPC_F_DRHODT]; a.dedt = c->f[MHPC_F_DEDT]; a.dsmldt = c->f[MHPC_F_DSMLDT];
    a.muijmax = c->f[MHPC_F_MUIJMAX];
    a.curlv = c->f[MHPC_F_CURLV];
    a.gradrho = c->f[MHPC_F_GRADRHO];
    if (c->p.precision == MHPC_PREC_FP64) {
        if (features) launch_forces_p<true, true>(c, a);
        else launch_forces_p<true, false>(c, a);
    } else {
        if (features) launch_forces_p<false, true>(c, a);
        else launch_forces_p<false, false>(c, a);
    }
}

// ------------------------------------------------------------------------------------
// neighbour lists back to the reference layout nnl[i * max_nb + k], original indices
__global__ __launch_bounds__(256) void k_nnl_to_caller(int64_t n, const int32_t *__restrict__ perm,
                                                       const int32_t *__restrict__ snoi,
                                                       const int32_t *__restrict__ nbr, int64_t stride,
                                                       int cap_nb, int32_t *__restrict__ nnl,
                                                       int32_t *__restrict__ noi, int max_nb) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int32_t i = perm[k];
    int cnt = snoi[k];
    noi[i] = cnt;
    cnt = cnt > cap_nb ? cap_nb : cnt;
    cnt = cnt > max_nb ? max_nb : cnt;
    for (int s = 0; s < cnt; s++) {
        const int32_t j = nbr[((int64_t)(s >> 2) * stride + k) * 4 + (s & 3)];
        nnl[(int64_t)i * max_nb + s] = perm[j];
    }
}

void launch_neighbours_to_caller(mhpc_ctx *c, int32_t *dst_nnl, int32_t *dst_noi, int max_nb) {
    if (c->n <= 0) return;
    hipLaunchKernelGGL(k_nnl_to_caller, dim3((unsigned)ceil_div(c->n, 256)), dim3(256), 0, c->stream,
                       c->n, c->perm, c->snoi, c->nbr, c->cap_pad, c->p.max_nb, dst_nnl, dst_noi, max_nb);
}

// after the h-iteration: final h, iteration counts and last counts to caller order
__global__ __launch_bounds__(256) void k_scatter_h(int64_t n, const int32_t *__restrict__ perm,
                                                   const double *__restrict__ sh,
                                                   const int32_t *__restrict__ siters,
                                                   const int32_t *__restrict__ snoi,
                                                   double *__restrict__ sml, int32_t *__restrict__ iters,
                                                   int32_t *__restrict__ noi) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int32_t i = perm[k];
    sml[i] = sh[k];
    iters[i] = siters[k];
    noi[i] = snoi[k];
}

void launch_scatter_h(mhpc_ctx *c) {
    if (c->n <= 0) return;
    hipLaunchKernelGGL(k_scatter_h, dim3((unsigned)ceil_div(c->n, 256)), dim3(256), 0, c->stream, c->n,
                       c->perm, c->sh, c->siters, c->snoi, c->f[MHPC_F_SML], c->h_iters, c->noi);
}
