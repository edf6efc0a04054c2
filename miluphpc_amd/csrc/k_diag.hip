// k_diag.hip -- global sums (Miluphpc::energy / angularMomentum, miluphpc.cpp:577-677;
// Physics::Kernel::kineticEnergy and calculateAngularMomentumBlockwise, subdomain.cu:
// 2428-2619).  FP64 with Neumaier compensation in every partial and in the combine, and a
// fixed two-stage order (per-block partials, then one block folds them in block order),
// so the result is deterministic.  The reference's blockwise reduction reads past n and
// reduces the input array instead of its shared buffer (subdomain.cu:2324-2393); this
// one does not inherit that.
#include "mhpc_internal.h"

#define DIAG_Q 13          // quantities
#define DIAG_BLOCKS 1024
#define DIAG_PARTIAL (DIAG_BLOCKS * 2 * DIAG_Q)   // doubles of per-block partials: [q][s, c][block]

struct Neu {
    double s = 0.0, c = 0.0;
    // the rounding error of s + x without a comparison of the two (Knuth's two-sum): the value
    // Neumaier's branch computes, in fewer instructions
    __device__ __forceinline__ void add(double x) {
        const double t = s + x, b = t - s;
        c += (s - (t - b)) + (x - b);
        s = t;
    }
    __device__ __forceinline__ void add(const Neu &o) {
        add(o.s);
        add(o.c);
    }
    __device__ __forceinline__ double value() const { return s + c; }
    // merges over each row of 16 lanes, the row's sum in its first lane (the other lanes hold it
    // with its terms in another order)
    template <int CTRL>
    __device__ __forceinline__ void merge_dpp() {
        auto moved = [](double v) {
            const uint64_t u = __builtin_bit_cast(uint64_t, v);
            const uint32_t lo = (uint32_t)dpp_mov<CTRL>((int)u), hi = (uint32_t)dpp_mov<CTRL>((int)(u >> 32));
            return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
        };
        Neu o;
        o.s = moved(s);
        o.c = moved(c);
        add(o);
    }
    __device__ __forceinline__ void row_fold() {
        merge_dpp<DPP_XOR1>();
        merge_dpp<DPP_XOR2>();
        merge_dpp<DPP_HALF_MIRROR>();
        merge_dpp<DPP_MIRROR>();
    }
    // a merged over the wave's halves (ROWS 2) or over its rows pairwise (ROWS 1) in the lower half /
    // the even rows, b in the upper half / the odd rows: one merge for two quantities
    template <int ROWS>
    static __device__ __forceinline__ Neu merge_rows(const Neu &a, const Neu &b) {
        Neu r, o;
        auto swap = [](double x, double y, double &first, double &second) {
            const uint64_t u = __builtin_bit_cast(uint64_t, x), v = __builtin_bit_cast(uint64_t, y);
            const auto lo = ROWS == 2 ? __builtin_amdgcn_permlane32_swap((uint32_t)u, (uint32_t)v, false, false)
                                      : __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)v, false, false);
            const auto hi = ROWS == 2
                                ? __builtin_amdgcn_permlane32_swap((uint32_t)(u >> 32), (uint32_t)(v >> 32), false, false)
                                : __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(v >> 32), false, false);
            first = __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]);
            second = __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
        };
        swap(a.s, b.s, r.s, o.s);
        swap(a.c, b.c, r.c, o.c);
        r.add(o);
        return r;
    }
    // the wave's sum in lane 0
    __device__ __forceinline__ void wave_fold() {
        row_fold();
        *this = merge_rows<1>(*this, *this);
        *this = merge_rows<2>(*this, *this);
    }
};

// quantities: 0 kinetic, 1 potential (sum u), 2 internal (sum m e), 3-5 momentum,
// 6-8 angular momentum sum m x cross v, 9 mass, 10-12 sum m x
//
// Bound by the nine field reads (72 B per particle).  One thread per quantity adding a block's 256
// partial sums in turn was a chain of 512 dependent compensated additions (68 us for 2,097,152
// particles); a butterfly per quantity through LDS 40 us, with the next particle's fields requested
// ahead; lane-row swaps that merge two quantities at once 28.7 us = 5.3 TB/s, a large copy's rate.
__global__ __launch_bounds__(256) void k_diag_partial(int64_t n, const double *__restrict__ x,
                                                      const double *__restrict__ y,
                                                      const double *__restrict__ z,
                                                      const double *__restrict__ vx,
                                                      const double *__restrict__ vy,
                                                      const double *__restrict__ vz,
                                                      const double *__restrict__ m,
                                                      const double *__restrict__ u,
                                                      const double *__restrict__ e,
                                                      double *__restrict__ partial) {
    Neu q[DIAG_Q];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    // the next particle's fields are requested before this one's sums
    double nx = 0.0, ny = 0.0, nz = 0.0, na = 0.0, nb = 0.0, nc = 0.0, nm = 0.0, nu = 0.0, ne = 0.0;
    auto request = [&]() {
        nx = x[i]; ny = y[i]; nz = z[i];
        na = vx[i]; nb = vy[i]; nc = vz[i];
        nm = m[i]; nu = u[i]; ne = e[i];
    };
    if (i < n) request();
    while (i < n) {
        const double mi = nm, xi = nx, yi = ny, zi = nz, a = na, b = nb, cz = nc, ui = nu, ei = ne;
        i += stride;
        if (i < n) request();
        q[0].add(0.5 * mi * (a * a + b * b + cz * cz));
        q[1].add(ui);
        q[2].add(mi * ei);
        q[3].add(mi * a);
        q[4].add(mi * b);
        q[5].add(mi * cz);
        q[6].add(mi * (yi * cz - zi * b));
        q[7].add(mi * (zi * a - xi * cz));
        q[8].add(mi * (xi * b - yi * a));
        q[9].add(mi);
        q[10].add(mi * xi);
        q[11].add(mi * yi);
        q[12].add(mi * zi);
    }
    __shared__ double ws[DIAG_Q][4], wc[DIAG_Q][4];
    // sixteen quantities to eight per half wave, four per row, then over the rows: 28 merges where
    // a butterfly per quantity is 78.  Row r's first lane ends with quantities 4 r .. 4 r + 3.
#pragma unroll
    for (int k = 0; k < 8; k++) q[k] = Neu::merge_rows<2>(q[k], k + 8 < DIAG_Q ? q[k + 8 < DIAG_Q ? k + 8 : 0] : Neu());
#pragma unroll
    for (int k = 0; k < 4; k++) {
        q[k] = Neu::merge_rows<1>(q[k], q[k + 4]);
        q[k].row_fold();
        const int at = 4 * (wave_lane() >> 4) + k;
        if ((wave_lane() & 15) == 0 && at < DIAG_Q) {
            ws[at][threadIdx.x / 64] = q[k].s;
            wc[at][threadIdx.x / 64] = q[k].c;
        }
    }
    __syncthreads();
    if (threadIdx.x < DIAG_Q) {
        const int k = threadIdx.x;
        Neu acc;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            acc.add(ws[k][w]);
            acc.add(wc[k][w]);
        }
        partial[(2 * k) * DIAG_BLOCKS + blockIdx.x] = acc.s;
        partial[(2 * k + 1) * DIAG_BLOCKS + blockIdx.x] = acc.c;
    }
}

// folds the block partials in a fixed order -- one wavefront per quantity, each lane a strided
// share of the blocks, then the butterfly -- and writes the diagnostics record (the derived
// quantities -- total, |L|, centre of mass -- with the same expressions for every caller).  One
// thread per quantity reading the partials in turn waited for 2048 dependent loads and additions
// (276 us at 1024 blocks; 6 us).  `out` may be host memory.
__global__ __launch_bounds__(64 * DIAG_Q) void k_diag_final(const double *__restrict__ partial, int nb,
                                                            mhpc_diagnostics *__restrict__ out) {
    __shared__ double q[DIAG_Q];
    const int k = threadIdx.x / 64;
    Neu acc;
#pragma unroll 4
    for (int b = wave_lane(); b < nb; b += 64) {
        acc.add(partial[(2 * k) * DIAG_BLOCKS + b]);
        acc.add(partial[(2 * k + 1) * DIAG_BLOCKS + b]);
    }
    acc.wave_fold();
    if (wave_lane() == 0) q[k] = acc.value();
    __syncthreads();
    if (threadIdx.x != 0) return;
    mhpc_diagnostics d;
    d.kinetic = q[0];
    d.potential = q[1];
    d.internal = q[2];
    d.total = q[0] + q[1] + q[2];
    for (int a = 0; a < 3; a++) {
        d.momentum[a] = q[3 + a];
        d.angular_momentum[a] = q[6 + a];
        d.com[a] = q[9] > 0.0 ? q[10 + a] / q[9] : 0.0;
    }
    d.angular_momentum_norm = sqrt(q[6] * q[6] + q[7] * q[7] + q[8] * q[8]);
    d.mass = q[9];
    *out = d;
}

static int diag_blocks(int64_t n) {
    int nb = (int)ceil_div(n, 256 * 4);
    if (nb < 1) nb = 1;
    if (nb > DIAG_BLOCKS) nb = DIAG_BLOCKS;
    return nb;
}

// device doubles the context keeps for the record (at least the five time-step terms)
int diag_num_quantities() { return (int)(sizeof(mhpc_diagnostics) / sizeof(double)) > 5
                                       ? (int)(sizeof(mhpc_diagnostics) / sizeof(double)) : 5; }
int diag_partial_size() { return DIAG_PARTIAL; }

static void diag_launch(hipStream_t stream, int64_t n, const double *x, const double *y, const double *z,
                        const double *vx, const double *vy, const double *vz, const double *m,
                        const double *u, const double *e, double *partial, mhpc_diagnostics *out) {
    const int nb = diag_blocks(n);
    hipLaunchKernelGGL(k_diag_partial, dim3(nb), dim3(256), 0, stream, n, x, y, z, vx, vy, vz, m, u, e, partial);
    hipLaunchKernelGGL(k_diag_final, dim3(1), dim3(64 * DIAG_Q), 0, stream, partial, nb, out);
}

void launch_diagnostics(mhpc_ctx *c, double *partial, mhpc_diagnostics *out) {
    double **f = c->f;
    diag_launch(c->stream, c->n, f[MHPC_F_X], f[MHPC_F_Y], f[MHPC_F_Z], f[MHPC_F_VX], f[MHPC_F_VY],
                f[MHPC_F_VZ], f[MHPC_F_MASS], f[MHPC_F_U], f[MHPC_F_E], partial, out);
}
