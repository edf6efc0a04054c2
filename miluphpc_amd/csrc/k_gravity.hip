// k_gravity.hip -- Barnes-Hut force, wavefront-cooperative.
//
// The reference walks the tree once per particle (computeForces_v1, gravity.cu:252-396)
// or once per warp of 32 sorted particles with a warp vote on the acceptance test
// (computeForces_v2, gravity.cu:726-903).  Here one wavefront, or a workgroup of several, owns
// a GROUP of 64 consecutive key-sorted particles and walks the tree once for all of them:
//   * the 64 lanes of a wavefront test up to 64 stacked nodes at a time (FP64, exact, the
//     acceptance test the oracle restates), so the traversal itself is parallel across lanes.
//     Vote form (the reference v2's warp vote, gravity.cu:836, over the group of 64): a cell is
//     accepted only if every member accepts it with its own distance.  A lane's cell that
//     passes the test against the group's bounding box passes it for every member (the box
//     distance is a lower bound of each member's, also after rounding), so only the other
//     cells are put to the vote: first the lane tests its cell against the member furthest out
//     in the cell's direction, whose rejection already decides; for the cells left, all 64
//     lanes test against their own particle and one ballot decides.  Box form: the
//     bounding-box test alone (one test per group); it opens more cells;
//   * leaves and accepted cells go to LDS interaction lists of the wavefront;
//   * each time a list holds 64 entries all 64 lanes evaluate it, every lane reading
//     the same LDS entry (broadcast) for its own particle.  FP32 mode: entries are
//     staged as FP32 positions relative to the group's centre (each rounded once from the
//     FP64 difference), each batch of up to 64 entries is summed in FP32 (potentials in two
//     chains) and the batch sums are added with Kahan compensation.  FP64 mode: plain FP64 throughout.
// The stack lives in LDS; the number of nodes popped per round shrinks as the stack
// fills so it cannot overflow (a hard bound still sets ERRF_STACK).
//
// Several wavefronts per group (MULTI) share the group's stack: each round pops up to 64 nodes
// per wavefront, every wavefront keeps its own interaction lists and partial sums over its nodes,
// and the partial sums are added in wavefront order at the end (same interactions, same counts).
// With one wavefront per group, 65,536 particles are 1024 wavefronts, one per SIMD, and every
// dependent FP64 operation and LDS read shows its latency (launch_bh chooses the width).
#include <type_traits>

#include "mhpc_internal.h"

#define BH_WAVES 2                       // one wavefront per group: groups per block
#define BH_MULTI_MAX 8                   // wavefronts per group at most
static_assert(MHPC_BH_GROUP == 64, "one Barnes-Hut group per wavefront");
#define BH_STACK 768                     // soft stack capacity
#define BH_STACK_PHYS (BH_STACK + 192)   // hard capacity
// a group with several wavefronts pops up to 64 nodes per wavefront and round: its stack holds
// as many more children
__host__ __device__ constexpr int bh_stack_soft(int waves) { return BH_STACK + 448 * (waves - 1); }
__host__ __device__ constexpr int bh_stack_phys(int waves) { return bh_stack_soft(waves) + 192; }
#define BH_LIST 128
#define BH_FILL_WAVES 16384              // see bh_waves_per_group

// Interaction lists of one wavefront.  `p` holds the particles (id = sorted position) and,
// without quadrupoles, the accepted cells too (id = -1): both are the same monopole term.
// FP64 mode: {x, y, z, m}; FP32 mode: FP32 {x, y, z, m} relative to the group's centre (rounded
// once per entry from the FP64 difference, instead of once per lane and interaction).
template <bool FP64, bool QUAD>
struct BHLists {
    typedef typename std::conditional<FP64, double4, float4>::type rec;
    rec p[BH_LIST];
    int id[BH_LIST];
    // cells with their quadrupole
    rec c[QUAD ? BH_LIST : 1];
    float4 q0[QUAD ? BH_LIST : 1];
    float2 q1[QUAD ? BH_LIST : 1];
};

template <bool FP64>
struct BHAcc;

template <>
struct BHAcc<false> {
    Kahan x, y, z, phi;
};

template <>
struct BHAcc<true> {
    Plain64 x, y, z, phi;
};

// 1/sqrt(x) for normal x > 0.  SOFT: x is known to be at least the softening, a normal number.
// Otherwise x = 0 (the particle itself, unsoftened) and x = inf give 0, and smaller x are raised to
// the smallest normal number, so that the bare hardware estimates apply (no denormal scaling).
template <bool SOFT>
__device__ __forceinline__ float rsq_pos(float x) {
    if (SOFT) return __builtin_amdgcn_rsqf(x);
    return x > 0.f ? __builtin_amdgcn_rsqf(fmaxf(x, 1.17549435e-38f)) : 0.f;
}
template <bool SOFT>
__device__ __forceinline__ double rsq_pos(double x) {
    const double y = rsq_f64(SOFT ? x : fmax(x, 2.2250738585072014e-308));
    return SOFT || (x > 0.0 && x <= 1.7976931348623157e308) ? y : 0.0;   // rsq_f64(inf) is no number
}

// Monopole batch, FP32: plain FP32 sums over the (at most 64) entries, then one compensated
// (Kahan) addition of each batch sum into the running total.  13 instructions and the
// reciprocal square root per interaction.
template <bool POT, bool SOFT, typename ListT>
__device__ __forceinline__ void eval_mono(const ListT &L, int cnt, float px, float py, float pz, int self,
                                          float eps2, BHAcc<false> &acc) {
    float bx = 0.f, by = 0.f, bz = 0.f, bp[2] = {0.f, 0.f};
#pragma unroll 4
    for (int e = 0; e < cnt; e++) {
        const float4 q = L.p[e];
        const float dx = q.x - px, dy = q.y - py, dz = q.z - pz;
        const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, eps2)));
        const float rinv = rsq_pos<SOFT>(r2);
        const float mr = q.w * rinv;
        const float mr3 = mr * rinv * rinv;
        bx = __builtin_fmaf(mr3, dx, bx);
        by = __builtin_fmaf(mr3, dy, by);
        bz = __builtin_fmaf(mr3, dz, bz);
        // two chains: all terms have one sign, so that a chain's roundings grow with its length
        if (POT && L.id[e] != self) {
            if (e & 1) bp[1] -= mr;
            else bp[0] -= mr;
        }
    }
    acc.x.add(bx);
    acc.y.add(by);
    acc.z.add(bz);
    if (POT) acc.phi.add(bp[0]);
    if (POT) acc.phi.add(bp[1]);
}

// The same in FP64, summed as it comes.
template <bool POT, bool SOFT, typename ListT>
__device__ __forceinline__ void eval_mono(const ListT &L, int cnt, double px, double py, double pz, int self,
                                          double eps2, BHAcc<true> &acc) {
#pragma unroll 4
    for (int e = 0; e < cnt; e++) {
        const double4 q = L.p[e];
        const double dx = q.x - px, dy = q.y - py, dz = q.z - pz;
        const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
        const double rinv = rsq_pos<SOFT>(r2);
        const double mr = q.w * rinv;
        const double mr3 = mr * (rinv * rinv);
        acc.x.s = fma(mr3, dx, acc.x.s);
        acc.y.s = fma(mr3, dy, acc.y.s);
        acc.z.s = fma(mr3, dz, acc.z.s);
        if (POT && L.id[e] != self) acc.phi.s -= mr;
    }
}

// Cells with the traceless quadrupole: a = (m r^-3 + 5/2 (d.Qd) r^-7) d - r^-5 Qd, the two terms
// along d taken together (33 instead of 39 instructions per interaction: the 16.7M Plummer walk
// is bound by its instruction rate, 34.7 -> 32.6 ms).
template <bool POT, bool SOFT, typename ListT, typename AccT, typename T>
__device__ __forceinline__ void eval_quad(const ListT &L, int cnt, T px, T py, T pz, T eps2, AccT &acc) {
    constexpr bool FP64 = sizeof(T) == 8;
    T bx = 0, by = 0, bz = 0, bp = 0;
#pragma unroll 2
    for (int e = 0; e < cnt; e++) {
        const auto q = L.c[e];
        const float4 a = L.q0[e];
        const float2 b = L.q1[e];
        const T qxx = a.x, qxy = a.y, qxz = a.z, qyy = a.w, qyz = b.x, qzz = b.y;
        const T dx = q.x - px, dy = q.y - py, dz = q.z - pz;
        const T r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
        const T rinv = rsq_pos<SOFT>(r2);
        const T u = rinv * rinv;
        const T r3 = rinv * u;
        const T r5 = r3 * u;
        const T qdx = fma(qxx, dx, fma(qxy, dy, qxz * dz));
        const T qdy = fma(qxy, dx, fma(qyy, dy, qyz * dz));
        const T qdz = fma(qxz, dx, fma(qyz, dy, qzz * dz));
        const T dqd = fma(dx, qdx, fma(dy, qdy, dz * qdz));
        const T k = r3 * fma(T(2.5), (dqd * u) * u, q.w);
        bx = fma(k, dx, fma(-r5, qdx, bx));
        by = fma(k, dy, fma(-r5, qdy, by));
        bz = fma(k, dz, fma(-r5, qdz, bz));
        if (POT) bp -= fma(T(0.5) * dqd, r5, q.w * rinv);
    }
    acc.x.add(bx);
    acc.y.add(by);
    acc.z.add(bz);
    if (POT) acc.phi.add(bp);
}

// a uniform lane's double (l must be the same in every lane)
__device__ __forceinline__ double readlane_d(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

struct BHArgs {
    int64_t n;
    const int32_t *perm;
    const double4 *sxm;
    const int32_t *clevel, *cchild;
    const double *cmass, *cx, *cy, *cz;
    const float4 *cquadf;
    const double *box;
    double theta, eps2, G;
    int mac;
    double *gax, *gay, *gaz, *u;
    uint32_t *err;
    unsigned long long *counters;
};

// LDS of a block: the stacks, the vote's outermost members, and the wavefronts' lists
template <bool FP64, bool QUAD>
struct BHBlock {
    typedef BHLists<FP64, QUAD> Lists;
    // MULTI: one stack; otherwise one per wavefront
    static __host__ __device__ constexpr size_t stack_ints(bool multi, int waves) {
        return multi ? (size_t)bh_stack_phys(waves) : (size_t)BH_STACK_PHYS * waves;
    }
    static constexpr size_t bytes(bool multi, int waves) {
        return sizeof(Lists) * waves + (multi ? 1 : waves) * 8 * 3 * sizeof(double) + stack_ints(multi, waves) * 4 +
               4 * BH_MULTI_MAX;
    }
};

template <bool FP64, bool POT, bool QUAD, bool VOTE, bool MULTI>
__global__ __launch_bounds__(64 * (MULTI ? BH_MULTI_MAX : BH_WAVES)) void k_bh_walk(BHArgs A) {
    typedef BHBlock<FP64, QUAD> Blk;
    typedef typename Blk::Lists Lists;
    typedef typename std::conditional<FP64, double, float>::type T;
    extern __shared__ __align__(32) unsigned char lds[];
    const int nw = blockDim.x / 64, w = threadIdx.x / 64, lane = wave_lane();
    Lists &L = reinterpret_cast<Lists *>(lds)[w];
    double *const ends_all = reinterpret_cast<double *>(lds + sizeof(Lists) * nw);
    double *const ends = ends_all + (MULTI ? 0 : w * 24);   // [axis][octant] outermost member
    int *const stack0 = reinterpret_cast<int *>(ends_all + (MULTI ? 1 : nw) * 24);
    int *const stack = stack0 + (MULTI ? 0 : w * BH_STACK_PHYS);
    int *const wtot = stack0 + Blk::stack_ints(MULTI, nw);   // MULTI: children pushed per wavefront
    const int stack_soft = MULTI ? bh_stack_soft(nw) : BH_STACK;
    const int stack_phys = MULTI ? bh_stack_phys(nw) : BH_STACK_PHYS;
    const int64_t block = xcd_block(blockIdx.x, gridDim.x);
    const int64_t group = MULTI ? block : block * nw + w;
    const int64_t k = group * 64 + lane;
    const int64_t n = A.n;
    if (group * 64 >= n) return;   // MULTI: the whole block, else the whole wave
    const bool valid = k < n;
    const double4 own = valid ? A.sxm[k] : make_double4(0.0, 0.0, 0.0, 0.0);
    const double px = own.x, py = own.y, pz = own.z;
    // group bounding box (exact)
    const double glo_x = wave_min(valid ? px : 1e300), ghi_x = wave_max(valid ? px : -1e300);
    const double glo_y = wave_min(valid ? py : 1e300), ghi_y = wave_max(valid ? py : -1e300);
    const double glo_z = wave_min(valid ? pz : 1e300), ghi_z = wave_max(valid ? pz : -1e300);
    const uint64_t mInvalid = ~wave_ballot(valid);
    const int nvalid = 64 - popc64(mInvalid);
    // acceptance constants, same expressions as the oracle
    const double R = 0.5 * (A.box[1] - A.box[0]);
    const double s2_0 = 4.0 * R * R;
    const double dp_1 = R * R / A.theta;
    const double theta2 = A.theta * A.theta;
    const double eps2 = A.eps2;
    const bool classic = A.mac == MHPC_MAC_CLASSIC;
    // FP32 mode: positions relative to the group's centre
    const double refx = 0.5 * (glo_x + ghi_x), refy = 0.5 * (glo_y + ghi_y), refz = 0.5 * (glo_z + ghi_z);
    const T tx = FP64 ? (T)px : (T)(px - refx), ty = FP64 ? (T)py : (T)(py - refy),
            tz = FP64 ? (T)pz : (T)(pz - refz);
    const T teps2 = (T)eps2;
    // every squared distance a positive normal number: softened, and (FP64) no box whose square leaves FP64
    const bool soft = teps2 >= (FP64 ? (T)2.2250738585072014e-308 : (T)1.17549435e-38f) && (!FP64 || R < 1e150);
    auto flush_p = [&](int cnt, BHAcc<FP64> &acc) {
        if (soft) eval_mono<POT, true>(L, cnt, tx, ty, tz, (int)k, teps2, acc);
        else eval_mono<POT, false>(L, cnt, tx, ty, tz, (int)k, teps2, acc);
    };
    auto flush_c = [&](int cnt, BHAcc<FP64> &acc) {
        if (soft) eval_quad<POT, true>(L, cnt, tx, ty, tz, teps2, acc);
        else eval_quad<POT, false>(L, cnt, tx, ty, tz, teps2, acc);
    };

    if (VOTE) {
        // the member furthest out in each octant direction: a cell in that direction is nearest
        // to it or to a member beside it, so its rejection settles most votes.  (Any member
        // would do: a choice that rejects nothing only leaves the cell to the ballot.)
        const double ux = valid ? px - refx : 0.0, uy = valid ? py - refy : 0.0, uz = valid ? pz - refz : 0.0;
        if (!MULTI || w == 0) {
#pragma unroll
            for (int o = 0; o < 8; o++) {
                const float d = (float)((o & 1 ? ux : -ux) + (o & 2 ? uy : -uy) + (o & 4 ? uz : -uz));
                const uint64_t m = wave_ballot(valid && d == wave_max(valid ? d : -3.0e38f));
                if (m != 0 && lane == __builtin_ctzll(m)) {
                    ends[o] = px;
                    ends[8 + o] = py;
                    ends[16 + o] = pz;
                } else if (m == 0 && lane == 0) {   // non-finite positions: any member
                    ends[o] = px;
                    ends[8 + o] = py;
                    ends[16 + o] = pz;
                }
            }
        }
    }

    BHAcc<FP64> acc;
    int top = 1, pl_n = 0, cl_n = 0;
    long long n_cells = 0, n_parts = 0;
    if (lane == 0 && (!MULTI || w == 0)) stack[0] = (int)n;   // root
    if (MULTI) __syncthreads(); else wave_sync();
    const uint64_t lt = lanemask_lt();
    bool overflow = false;
    while (top > 0) {
        int kpop = (stack_soft - top) / 7;
        kpop = kpop < 1 ? 1 : kpop;
        kpop = kpop > 64 * (MULTI ? nw : 1) ? 64 * (MULTI ? nw : 1) : kpop;
        kpop = kpop > top ? top : kpop;
        // MULTI: the popped nodes are dealt to the wavefronts in turn, each its share of lanes
        const int slot = MULTI ? lane * nw + w : lane;
        const int node = slot < kpop ? stack[top - kpop + slot] : -1;
        top -= kpop;
        if (!MULTI) wave_sync();
        const bool isPart = node >= 0 && node < n;
        const bool isCell = node >= n;
        bool accept = false, open = false;
        double ccx = 0, ccy = 0, ccz = 0;
        int64_t c = 0;
        double size = 0.0;
        // the acceptance test of distance^2 d2 for a cell of size term S (same expressions as the
        // oracle)
        auto mac_size = [&](int L) {
            return classic ? s2_0 * ldexp(1.0, -2 * L) : dp_1 * ldexp(1.0, -2 * (L - 1));
        };
        auto mac_ok = [&](double d2, double S) { return classic ? (d2 + eps2) * theta2 > S : S <= d2 + eps2; };
        // everything the round may need of its node is requested together, before the test
        // decides which of it is used: one memory round trip per round instead of one for the
        // test and one more for the children or the list entries
        int4 cha = make_int4(-1, -1, -1, -1), chb = cha;
        double cmass = 0.0;
        float4 qa = make_float4(0.f, 0.f, 0.f, 0.f), qb = qa;
        double4 prec = make_double4(0.0, 0.0, 0.0, 0.0);
        if (isPart) prec = A.sxm[node];
        if (isCell) {
            c = node - n;
            const int4 *cp = reinterpret_cast<const int4 *>(A.cchild + 8 * c);
            cha = cp[0];
            chb = cp[1];
            cmass = A.cmass[c];
            if (QUAD) {
                qa = A.cquadf[2 * c];
                qb = A.cquadf[2 * c + 1];
            }
            ccx = A.cx[c];
            ccy = A.cy[c];
            ccz = A.cz[c];
            size = mac_size(A.clevel[c]);
            const double dx = fmax(fmax(glo_x - ccx, ccx - ghi_x), 0.0);
            const double dy = fmax(fmax(glo_y - ccy, ccy - ghi_y), 0.0);
            const double dz = fmax(fmax(glo_z - ccz, ccz - ghi_z), 0.0);
            accept = mac_ok(dx * dx + dy * dy + dz * dz, size);
        }
        if constexpr (VOTE) {
            // cells the box test rejects: one member's rejection settles the vote, and the
            // outermost member towards the cell is the likeliest to reject
            bool amb = isCell && !accept;
            if (amb) {
                const int o = (ccx > refx ? 1 : 0) | (ccy > refy ? 2 : 0) | (ccz > refz ? 4 : 0);
                const double dx = ccx - ends[o], dy = ccy - ends[8 + o], dz = ccz - ends[16 + o];
                amb = mac_ok(dx * dx + dy * dy + dz * dz, size);
            }
            // the others: every member tests each with its own distance
            uint64_t mAmb = wave_ballot(amb);
            uint64_t mVote = 0;
            while (mAmb) {
                const int b = __builtin_ctzll(mAmb);
                mAmb &= mAmb - 1;
                const double bx = readlane_d(ccx, b), by = readlane_d(ccy, b), bz = readlane_d(ccz, b);
                const double bs = readlane_d(size, b);
                const double dx = bx - px, dy = by - py, dz = bz - pz;
                const bool ok = mac_ok(dx * dx + dy * dy + dz * dz, bs);
                if ((wave_ballot(ok) | mInvalid) == ~0ull) mVote |= 1ull << b;
            }
            accept = accept || ((mVote >> lane) & 1ull);
        }
        open = isCell && !accept;
        // children of opened cells
        int ch[8];
        int nc = 0;
        if (open) {
            ch[0] = cha.x; ch[1] = cha.y; ch[2] = cha.z; ch[3] = cha.w;
            ch[4] = chb.x; ch[5] = chb.y; ch[6] = chb.z; ch[7] = chb.w;
#pragma unroll
            for (int s = 0; s < 8; s++) nc += ch[s] != -1;
        }
        const int incl = wave_incl_scan(nc);
        int tot = __shfl(incl, 63), before = 0;
        if (MULTI) {
            // every wavefront has read its nodes before any pushes
            if (lane == 0) wtot[w] = tot;
            __syncthreads();
            tot = 0;
            for (int v = 0; v < nw; v++) {
                const int t = wtot[v];
                before += v < w ? t : 0;
                tot += t;
            }
        }
        if (top + tot > stack_phys) {   // MULTI: the same decision in every wavefront
            overflow = true;
            break;
        }
        if (open) {
            int pos = top + before + incl - nc;
#pragma unroll
            for (int s = 7; s >= 0; s--)
                if (ch[s] != -1) stack[pos++] = ch[s];
        }
        top += tot;
        // list entries: particles, and cells (with quadrupole: a list of their own)
        const uint64_t mP = wave_ballot(isPart), mA = wave_ballot(accept);
        const uint64_t mL = QUAD ? mP : (mP | mA);
        const bool toP = isPart || (!QUAD && accept);
        if (toP) {
            const int pos = pl_n + popc64(mL & lt);
            const double ex = isPart ? prec.x : ccx, ey = isPart ? prec.y : ccy, ez = isPart ? prec.z : ccz;
            const double em = isPart ? prec.w : cmass;
            if constexpr (FP64) L.p[pos] = make_double4(ex, ey, ez, em);
            else L.p[pos] = make_float4((float)(ex - refx), (float)(ey - refy), (float)(ez - refz), (float)em);
            if (POT) L.id[pos] = isPart ? node : -1;
        }
        if constexpr (QUAD) {
            if (accept) {
                const int pos = cl_n + popc64(mA & lt);
                if constexpr (FP64) L.c[pos] = make_double4(ccx, ccy, ccz, cmass);
                else
                    L.c[pos] = make_float4((float)(ccx - refx), (float)(ccy - refy), (float)(ccz - refz),
                                           (float)cmass);
                L.q0[pos] = qa;
                L.q1[pos] = make_float2(qb.x, qb.y);
            }
            cl_n += popc64(mA);
        }
        pl_n += popc64(mL);
        n_parts += popc64(mP);
        n_cells += popc64(mA);
        wave_sync();
        if (pl_n >= 64) {
            flush_p(64, acc);
            wave_sync();
            const int rest = pl_n - 64;
            if (lane < rest) {
                const auto a = L.p[64 + lane];
                L.p[lane] = a;
                if (POT) {
                    const int id = L.id[64 + lane];
                    L.id[lane] = id;
                }
            }
            pl_n = rest;
            wave_sync();
        }
        if constexpr (QUAD) {
            if (cl_n >= 64) {
                flush_c(64, acc);
                wave_sync();
                const int rest = cl_n - 64;
                if (lane < rest) {
                    const auto a = L.c[64 + lane];
                    const float4 q0 = L.q0[64 + lane];
                    const float2 q1 = L.q1[64 + lane];
                    L.c[lane] = a;
                    L.q0[lane] = q0;
                    L.q1[lane] = q1;
                }
                cl_n = rest;
                wave_sync();
            }
        }
        if (MULTI) __syncthreads();   // the pushed children are on the stack
    }
    if (overflow) {
        if (lane == 0) set_err(A.err, ERRF_STACK);
        return;
    }
    if (pl_n > 0) flush_p(pl_n, acc);
    if constexpr (QUAD) {
        if (cl_n > 0) flush_c(cl_n, acc);
    }
    double ax = acc.x.value(), ay = acc.y.value(), az = acc.z.value(), ph = POT ? acc.phi.value() : 0.0;
    if (MULTI) {
        // the wavefronts' partial sums, added in wavefront order (their lists are done with)
        __syncthreads();
        double *const part = reinterpret_cast<double *>(lds);
        static_assert(sizeof(Lists) >= 4 * 64 * sizeof(double), "the lists hold the partial sums");
        part[(w * 4 + 0) * 64 + lane] = ax;
        part[(w * 4 + 1) * 64 + lane] = ay;
        part[(w * 4 + 2) * 64 + lane] = az;
        part[(w * 4 + 3) * 64 + lane] = ph;
        __syncthreads();
        if (w == 0) {
            for (int v = 1; v < nw; v++) {
                ax += part[(v * 4 + 0) * 64 + lane];
                ay += part[(v * 4 + 1) * 64 + lane];
                az += part[(v * 4 + 2) * 64 + lane];
                ph += part[(v * 4 + 3) * 64 + lane];
            }
        }
    }
    if (valid && (!MULTI || w == 0)) {
        const int32_t i = A.perm[k];
        A.gax[i] = A.G * ax;
        A.gay[i] = A.G * ay;
        A.gaz[i] = A.G * az;
        if (POT) A.u[i] = 0.5 * own.w * A.G * ph;
    }
    if (lane == 0) {
        atomicAdd(&cnt_slot(A.counters)[CNT_CELL_INT], (unsigned long long)(n_cells * nvalid));
        atomicAdd(&cnt_slot(A.counters)[CNT_PART_INT], (unsigned long long)(n_parts * nvalid));
    }
}

// Wavefronts per group: enough groups fill the chip (256 CUs, 4 SIMDs each) by themselves; with
// fewer, each group is shared by up to 4 wavefronts, and by up to 8 where even that leaves the
// chip half empty (not with quadrupoles, whose lists take more LDS).  RHS times with 1 wavefront
// per group and with this rule: 65,536 FP64 monopole 735 / 514 us (8 wavefronts: 528), 300,007
// FP32 quadrupole 1018 / 955 us (2 wavefronts: 978), a leapfrog step of 2048 385 / 293 us; 1M FP32
// monopole (16,384 groups, so one either way) is no faster with two (6.13 / 6.22 ms with SPH).
static int bh_waves_per_group(int64_t groups, bool quad) {
    const int most = !quad && groups < BH_FILL_WAVES / 32 ? BH_MULTI_MAX : 4;
    int w = 1;
    while (w < most && groups * w < BH_FILL_WAVES) w *= 2;
    return w;
}

template <bool FP64, bool POT, bool QUAD>
static void launch_bh(mhpc_ctx *c, const BHArgs &a) {
    typedef BHBlock<FP64, QUAD> Blk;
    const int64_t groups = ceil_div(c->n, 64);
    const bool vote = c->p.bh_accept == MHPC_BH_VOTE;
    const int waves = bh_waves_per_group(groups, QUAD);
    if (waves == 1) {
        const dim3 grid((unsigned)ceil_div(groups, BH_WAVES)), block(64 * BH_WAVES);
        const size_t bytes = Blk::bytes(false, BH_WAVES);
        if (vote) hipLaunchKernelGGL((k_bh_walk<FP64, POT, QUAD, true, false>), grid, block, bytes, c->stream, a);
        else hipLaunchKernelGGL((k_bh_walk<FP64, POT, QUAD, false, false>), grid, block, bytes, c->stream, a);
        return;
    }
    static_assert(Blk::bytes(true, QUAD ? 4 : BH_MULTI_MAX) <= 65536, "LDS of a block");
    const dim3 grid((unsigned)groups), block(64 * waves);
    const size_t bytes = Blk::bytes(true, waves);
    if (vote) hipLaunchKernelGGL((k_bh_walk<FP64, POT, QUAD, true, true>), grid, block, bytes, c->stream, a);
    else hipLaunchKernelGGL((k_bh_walk<FP64, POT, QUAD, false, true>), grid, block, bytes, c->stream, a);
}

// ------------------------------------------------------------------------------------
// a7' computeForces_v1 (gravity.cu:252-396) as the reference runs it: one thread per particle
// walks the tree depth first from the root, resuming each level at its next child slot
// (curNode / curChild per depth), skipping itself; a child is taken if it is a particle or
// (d^2 + eps^2) theta^2 > cellSize[depth], cellSize[d] = 4 R^2 / 4^d, else descended into.
// Monopole, FP64, in the reference's order and expressions (f = m / d^3 with d the square
// root of the softened distance; u -= 1/2 m_c m_i / d).  The per-depth resume state lives in
// LDS; the tree has at most MHPC_LEVELS + 1 levels below the root.
#define BH1_THREADS 64
#define BH1_DEPTH (MHPC_LEVELS + 3)

template <bool POT>
__global__ __launch_bounds__(BH1_THREADS) void k_bh_v1(BHArgs A) {
    __shared__ int cur_node[BH1_DEPTH][BH1_THREADS];
    __shared__ unsigned char cur_child[BH1_DEPTH][BH1_THREADS];
    const int t = threadIdx.x;
    const int64_t k = blockIdx.x * (int64_t)BH1_THREADS + t;
    const int64_t n = A.n;
    // lanes past the last particle walk nothing but take part in the wave's counter sums
    const bool valid = k < n;
    const double4 own = valid ? A.sxm[k] : make_double4(0.0, 0.0, 0.0, 0.0);
    const double px = own.x, py = own.y, pz = own.z;
    const double R = 0.5 * (A.box[1] - A.box[0]);
    const double cs0 = 4.0 * R * R;
    const double thetasq = A.theta * A.theta;
    double axi = 0.0, ayi = 0.0, azi = 0.0, ui = 0.0;
    long long n_cells = 0, n_parts = 0;
    int depth = valid ? 1 : 0;
    cur_node[1][t] = (int)n;   // root
    cur_child[1][t] = 0;
    bool overflow = false;
    while (depth > 0) {
        int child_number = cur_child[depth][t];
        int node = cur_node[depth][t];
        // cellSize[depth] of the reference's table: 4 R^2 / 4^depth, exact powers of 4
        double cell_size = cs0 * ldexp(1.0, -2 * depth);
        while (child_number < 8) {
            int c;
            do {
                c = node >= n ? A.cchild[8 * (int64_t)(node - n) + child_number] : -1;
                child_number++;
            } while (c == -1 && child_number < 8);
            if (c != -1 && c != (int)k) {
                double cx, cy, cz, cm;
                if (c < n) {
                    const double4 r = A.sxm[c];
                    cx = r.x; cy = r.y; cz = r.z; cm = r.w;
                } else {
                    const int64_t q = c - n;
                    cx = A.cx[q]; cy = A.cy[q]; cz = A.cz[q]; cm = A.cmass[q];
                }
                const double dx = cx - px;
                double dist = dx * dx + A.eps2;
                const double dy = cy - py;
                dist += dy * dy;
                const double dz = cz - pz;
                dist += dz * dz;
                if (c < n || dist * thetasq > cell_size) {
                    dist = sqrt(dist);
                    const double f = cm / (dist * dist * dist);
                    axi += f * dx;
                    ayi += f * dy;
                    azi += f * dz;
                    if (POT) ui -= 0.5 * (cm * own.w) / dist;
                    if (c < n) n_parts++; else n_cells++;
                } else {
                    cur_child[depth][t] = (unsigned char)child_number;
                    cur_node[depth][t] = node;
                    depth++;
                    if (depth >= BH1_DEPTH) {
                        overflow = true;
                        depth = 0;
                        break;
                    }
                    child_number = 0;
                    node = c;
                    cell_size = cs0 * ldexp(1.0, -2 * depth);
                }
            }
        }
        depth--;
    }
    if (overflow) set_err(A.err, ERRF_STACK);
    if (valid) {
        const int32_t i = A.perm[k];
        A.gax[i] = A.G * axi;
        A.gay[i] = A.G * ayi;
        A.gaz[i] = A.G * azi;
        if (POT) A.u[i] = A.G * ui;
    }
    const unsigned long long sc = (unsigned long long)wave_sum(n_cells);
    const unsigned long long sp = (unsigned long long)wave_sum(n_parts);
    if (wave_lane() == 0) {
        atomicAdd(&cnt_slot(A.counters)[CNT_CELL_INT], sc);
        atomicAdd(&cnt_slot(A.counters)[CNT_PART_INT], sp);
    }
}

void launch_gravity(mhpc_ctx *c, bool potential) {
    if (c->n <= 0) return;
    BHArgs a;
    a.n = c->n;
    a.perm = c->perm;
    a.sxm = c->sxm;
    a.clevel = c->clevel;
    a.cchild = c->cchild;
    a.cmass = c->cmass; a.cx = c->cx; a.cy = c->cy; a.cz = c->cz;
    a.cquadf = c->cquadf;
    a.box = c->box;
    a.theta = c->p.theta;
    a.eps2 = c->p.smoothing;
    a.G = c->p.G;
    a.mac = c->p.mac;
    a.gax = c->f[MHPC_F_G_AX]; a.gay = c->f[MHPC_F_G_AY]; a.gaz = c->f[MHPC_F_G_AZ];
    a.u = c->f[MHPC_F_U];
    a.err = c->err;
    a.counters = c->counters;
    if (c->p.bh_accept == MHPC_BH_PER_PARTICLE) {
        const dim3 grid((unsigned)ceil_div(c->n, BH1_THREADS)), block(BH1_THREADS);
        if (potential) hipLaunchKernelGGL(k_bh_v1<true>, grid, block, 0, c->stream, a);
        else hipLaunchKernelGGL(k_bh_v1<false>, grid, block, 0, c->stream, a);
        return;
    }
    const bool fp64 = c->p.precision == MHPC_PREC_FP64;
    const bool quad = c->p.quadrupole != 0;
    if (fp64) {
        if (potential) {
            if (quad) launch_bh<true, true, true>(c, a); else launch_bh<true, true, false>(c, a);
        } else {
            if (quad) launch_bh<true, false, true>(c, a); else launch_bh<true, false, false>(c, a);
        }
    } else {
        if (potential) {
            if (quad) launch_bh<false, true, true>(c, a); else launch_bh<false, true, false>(c, a);
        } else {
            if (quad) launch_bh<false, false, true>(c, a); else launch_bh<false, false, false>(c, a);
        }
    }
}
