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
    // the wave's sum in every lane: a butterfly of compensated merges (each step adds a lane's
    // sum and correction into its partner's, lower lane first, so both hold the same bits)
    __device__ __forceinline__ void wave_fold() {
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            Neu a, b;
            const double ps = __shfl_xor(s, o), pc = __shfl_xor(c, o);
            const bool upper = wave_lane() & o;
            a.s = upper ? ps : s;
            a.c = upper ? pc : c;
            b.s = upper ? s : ps;
            b.c = upper ? c : pc;
            a.add(b);
            *this = a;
        }
    }
};

// quantities: 0 kinetic, 1 potential (sum u), 2 internal (sum m e), 3-5 momentum,
// 6-8 angular momentum sum m x cross v, 9 mass, 10-12 sum m x
//
// Bound by the nine field reads (72 B per particle).  A block's 256 partial sums are merged by
// wavefront butterflies: one thread per quantity adding them in turn was a chain of 512 dependent
// compensated additions (68 us for 2,097,152 particles; 42 us as butterflies, 40 us = 3.8 TB/s with
// the next particle's fields requested ahead).
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
#pragma unroll
    for (int k = 0; k < DIAG_Q; k++) {
        q[k].wave_fold();
        if (wave_lane() == 0) {
            ws[k][threadIdx.x / 64] = q[k].s;
            wc[k][threadIdx.x / 64] = q[k].c;
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
