// k_mlp.hip -- learned smoothing length: a 7 -> 64 -> 64 -> 1 tanh MLP with BF16 weights
// and activations on the matrix cores (v_mfma_f32_16x16x16_bf16, FP32 accumulation),
// FP32 master weights and Adam.  It predicts log(h_converged / h_previous) from a
// particle's state; the plain h-iteration starts from the prediction and has the last word.
// No counterpart in the reference.
//
// Inference and training both take 16 samples per step with the activations and, in training,
// the gradients' accumulators in registers (mlp_forward_16, k_mlp_train_grad).  Training writes
// one gradient partial per block; one kernel folds them in a fixed order (deterministic) and
// updates the weights (Adam).
#include <math.h>

#include "mhpc_internal.h"

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float f) {
    unsigned u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);   // round to nearest even (inputs are finite)
    return (unsigned short)(u >> 16);
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bfl2 __attribute__((ext_vector_type(2)));
// the same rounding by the hardware's packed conversion (v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bfl2));
}
__device__ __forceinline__ bf16x4 pack_bf16x4(float a, float b, float c, float d) {
    const uint2 v = make_uint2(pack_bf16(a, b), pack_bf16(c, d));
    return __builtin_bit_cast(bf16x4, v);
}
__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float(((unsigned)b) << 16); }

// D(16x16) += A(16x16) B(16x16).  Fragments: lane l holds A[l%16][4(l/16)..+3],
// B[4(l/16)..+3][l%16] and D[4(l/16)+r][l%16], r = 0..3.
__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

#define MLP_IN 8      // 7 features + 1 zero pad
#define MLP_H 64
#define MLP_NPARAM (MLP_H * MLP_IN + MLP_H + MLP_H * MLP_H + MLP_H + MLP_H + 1)   // 4801

// parameter offsets in the flat FP32 vector
#define P_W1 0
#define P_B1 (P_W1 + MLP_H * MLP_IN)
#define P_W2 (P_B1 + MLP_H)
#define P_B2 (P_W2 + MLP_H * MLP_H)
#define P_W3 (P_B2 + MLP_H)
#define P_B3 (P_W3 + MLP_H)

static_assert(MLP_NPARAM == MHPC_MLP_NPARAM, "parameter layout of include/mhpc.h");

int mlp_num_params() { return MLP_NPARAM; }

// tanh(x) = 1 - 2 / (exp(2x) + 1) from the hardware exp2 and reciprocal estimates: absolute
// error ~1e-7, far below the BF16 rounding the activations are stored with; saturates to
// +-1 for large |x|
__device__ __forceinline__ float tanh_fast(float x) {
    const float e = __builtin_amdgcn_exp2f(x * 2.8853900817779268f);   // exp(2x) = 2^(2x log2 e)
    return 1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f);
}

// ------------------------------------------------------------------------------------
// features, caller order: 0 log10 h, 1 neighbour count / target, 2 log10 rho, 3 div v h/c
// (div v = -drho/dt / rho), 4 |curl v| h / c, 5 |grad rho| h / rho, 6 dt c / h;
// c = cs + (tiny) so cold gas gives finite values.  Normalised with the stored mean / std.
__global__ __launch_bounds__(256) void k_mlp_features(int64_t n, const double *__restrict__ h,
                                                      const int32_t *__restrict__ noi,
                                                      const double *__restrict__ rho,
                                                      const double *__restrict__ drhodt,
                                                      const double *__restrict__ curl,
                                                      const double *__restrict__ gradrho,
                                                      const double *__restrict__ cs, double dt,
                                                      int n_target, const float *__restrict__ norm,
                                                      float clip, float *__restrict__ X,
                                                      double *__restrict__ hprev) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double hi = h[i];
    const double r = rho[i] > 0.0 ? rho[i] : 1e-300;
    const double c = cs[i] + 1e-12;
    float f[7];
    f[0] = (float)log10(hi);
    f[1] = (float)((double)noi[i] / (double)n_target);
    f[2] = (float)log10(r);
    f[3] = (float)(-drhodt[i] / r * hi / c);
    f[4] = (float)(curl[i] * hi / c);
    f[5] = (float)(gradrho[i] * hi / r);
    f[6] = (float)(dt * c / hi);
#pragma unroll
    for (int k = 0; k < 7; k++) {
        float v = (f[k] - norm[k]) / norm[8 + k];
        v = fminf(fmaxf(v, -clip), clip);
        X[i * MLP_IN + k] = v;
    }
    X[i * MLP_IN + 7] = 0.f;
    hprev[i] = hi;
}

// normalised features are clipped to +-MLP_CLIP standard deviations
#define MLP_CLIP 8.f

// normalise raw features in place (after the statistics have been taken from them)
__global__ __launch_bounds__(256) void k_mlp_renorm(int64_t n, const float *__restrict__ norm, float *__restrict__ X) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= n * MLP_IN) return;
    const int k = (int)(t % MLP_IN);
    if (k >= 7) return;
    const float v = (X[t] - norm[k]) / norm[8 + k];
    X[t] = fminf(fmaxf(v, -MLP_CLIP), MLP_CLIP);
}

void launch_mlp_renorm(mhpc_ctx *c) {
    if (c->n <= 0) return;
    hipLaunchKernelGGL(k_mlp_renorm, dim3((unsigned)ceil_div(c->n * MLP_IN, 256)), dim3(256), 0, c->stream, c->n,
                       c->mlp_norm, c->mlp_x);
}

// Inference with the activations kept in registers.  The layers are computed transposed --
// hidden units as rows, samples as columns -- so the fragment a lane holds after one layer,
// D[4q + r][c] (q = lane / 16, c = lane % 16, r = 0..3), is exactly its B operand of the next
// layer, B[k = 4q + r][c]: no LDS round trip and no layout change between the layers.  The
// weights are the A operands and stay in registers for the whole kernel.  One step takes 16
// samples (one column block): layer 1 is 4 MFMAs (K = 16, features 8..15 zero), layer 2 is 16
// (4 row blocks x 4 K steps), and the output a per-lane partial over the lane's 16 hidden
// units plus two cross-lane sums.  Same BF16 roundings as the training kernel's forward
// (inputs, weights and both layers' activations), FP32 accumulation.
struct MlpRegs {
    bf16x4 w1[4];                         // W1[mt*16 + c][4q .. 4q+3]
    bf16x4 w2[4][4];                      // W2[mt*16 + c][kt*16 + 4q .. +3]
    float b1[4][4], b2[4][4], w3[4][4];   // [mt][r]: hidden unit mt*16 + 4q + r
    float b3;
};

__device__ __forceinline__ void load_regs(MlpRegs &R, const float *__restrict__ p) {
    const int lane = wave_lane(), c = lane & 15, q = lane >> 4;
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = 4 * q + j;
            R.w1[mt][j] = (short)(k < MLP_IN ? f2bf(p[P_W1 + (mt * 16 + c) * MLP_IN + k]) : 0);
        }
#pragma unroll
        for (int kt = 0; kt < 4; kt++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                R.w2[mt][kt][j] = (short)f2bf(p[P_W2 + (mt * 16 + c) * MLP_H + kt * 16 + 4 * q + j]);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int hu = mt * 16 + 4 * q + r;
            R.b1[mt][r] = p[P_B1 + hu];
            R.b2[mt][r] = p[P_B2 + hu];
            R.w3[mt][r] = p[P_W3 + hu];
        }
    }
    R.b3 = p[P_B3];
}

// the network's output for samples s0 .. s0 + 15 (lane c and its copies c + 16, c + 32, c + 48
// return the value of sample s0 + c; samples at or beyond n read zero features)
__device__ __forceinline__ float mlp_forward_16(const MlpRegs &R, const float *__restrict__ X, int64_t s0,
                                                int64_t n) {
    const int lane = wave_lane(), c = lane & 15, q = lane >> 4;
    bf16x4 xb = {0, 0, 0, 0};
    const int64_t s = s0 + c;
    if (q < 2 && s < n) {
        const float4 v = *reinterpret_cast<const float4 *>(X + s * MLP_IN + 4 * q);
        xb[0] = (short)f2bf(v.x);
        xb[1] = (short)f2bf(v.y);
        xb[2] = (short)f2bf(v.z);
        xb[3] = (short)f2bf(v.w);
    }
    bf16x4 a1[4];
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        const f32x4 d = mfma16(R.w1[mt], xb, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int r = 0; r < 4; r++) a1[mt][r] = (short)f2bf(tanh_fast(d[r] + R.b1[mt][r]));
    }
    float part = 0.f;
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < 4; kt++) d = mfma16(R.w2[mt][kt], a1[kt], d);
#pragma unroll
        for (int r = 0; r < 4; r++) part += bf2f(f2bf(tanh_fast(d[r] + R.b2[mt][r]))) * R.w3[mt][r];
    }
    part += __shfl_xor(part, 16);
    part += __shfl_xor(part, 32);
    return part + R.b3;
}

// inference: h = h_prev * exp(y * sigma_t + mu_t), clamped to [1/4, 4] x h_prev.  A bounded
// grid of wavefronts looping over 16-sample steps; each wave converts its weight fragments once.
#define MLP_INF_WAVES 4
#define MLP_INF_BLOCKS 1024
__global__ __launch_bounds__(64 * MLP_INF_WAVES) void k_mlp_predict(int64_t n, const float *__restrict__ X,
                                                                   const float *__restrict__ params,
                                                                   const float *__restrict__ norm,
                                                                   const double *__restrict__ hprev,
                                                                   double *__restrict__ h_out) {
    MlpRegs R;
    load_regs(R, params);
    const int w = threadIdx.x / 64, lane = wave_lane();
    const double mu = norm[16], sd = norm[16 + 1];
    for (int64_t s0 = ((int64_t)blockIdx.x * MLP_INF_WAVES + w) * 16; s0 < n;
         s0 += (int64_t)gridDim.x * MLP_INF_WAVES * 16) {
        const float y = mlp_forward_16(R, X, s0, n);
        const int64_t i = s0 + lane;
        if (lane < 16 && i < n) {
            double t = (double)y * sd + mu;
            t = fmin(fmax(t, -1.3862943611198906), 1.3862943611198906);   // ln 4
            h_out[i] = hprev[i] * exp(t);
        }
    }
}

// forward only on given inputs (test hook): Y[i] = y
__global__ __launch_bounds__(64 * MLP_INF_WAVES) void k_mlp_forward_raw(int64_t n, const float *__restrict__ X,
                                                                       const float *__restrict__ params,
                                                                       float *__restrict__ Y) {
    MlpRegs R;
    load_regs(R, params);
    const int w = threadIdx.x / 64, lane = wave_lane();
    for (int64_t s0 = ((int64_t)blockIdx.x * MLP_INF_WAVES + w) * 16; s0 < n;
         s0 += (int64_t)gridDim.x * MLP_INF_WAVES * 16) {
        const float y = mlp_forward_16(R, X, s0, n);
        const int64_t i = s0 + lane;
        if (lane < 16 && i < n) Y[i] = y;
    }
}

// ------------------------------------------------------------------------------------
// random sample of a training step: a hash of the seed and the slot
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Training gradient: each wavefront takes 16 samples per step -> forward, loss, backward -- and
// keeps the gradient in registers over all its steps (MFMA accumulators of dW2 and dW1, per-lane
// sums of the rest).
//
// Two layouts, "T" (lane (q, c) holds hidden units 4q + r of sample c) and "N" (samples 4q + r
// of hidden unit c).  An MFMA result in one is an operand of the next product without any
// exchange between lanes, and swapping the two operands of a product gives its result in the
// other layout, with the same value for every element; so the forward pass is computed in both:
//   T feeds the products over hidden units (layer 2, dA1 = dz2 W2);
//   N feeds the products over samples (dW2 = dz2^T a1, dW1 = dz1^T x).
// No activation goes through LDS.  Bound by latency and the 64 tanh per lane and step: one wave
// per 64 samples with the activations in LDS (two wavefronts per CU, transposed 2-byte reads)
// took 52 us for 65,536 samples, this 20 us
// (30 us with the weights converted by every block instead of by the Adam update).
#define MLP_TR_WAVES 4
#define MLP_TR_BLOCKS 256                // gradient partials at most
// A partial is laid out as the lanes hold it, four floats (r) per lane: dW2 blocks, dW1 blocks,
// then dW3, db2, db1 per hidden unit, db3 and the loss.
#define G_W1 (MLP_H * MLP_H)
#define G_W3 (G_W1 + 4 * 64 * 4)
#define G_B2 (G_W3 + MLP_H)
#define G_B1 (G_B2 + MLP_H)
#define G_B3 (G_B1 + MLP_H)
#define G_LOSS (G_B3 + 1)
#define MLP_ROW 5376
static_assert(MLP_ROW > G_LOSS && MLP_ROW % 64 == 0, "a partial holds the gradient and the loss");

// the parameter that element i of a partial is the gradient of (-1: none)
__device__ __forceinline__ int mlp_param_of(int i) {
    const int r = i & 3, lane = (i >> 2) & 63, c = lane & 15, q = lane >> 4;
    if (i < G_W1) {
        const int t = i >> 8, mt = t >> 2, nt = t & 3;
        return P_W2 + (mt * 16 + 4 * q + r) * MLP_H + nt * 16 + c;
    }
    if (i < G_W3) return c < MLP_IN ? P_W1 + (((i - G_W1) >> 8) * 16 + 4 * q + r) * MLP_IN + c : -1;
    if (i < G_B2) return P_W3 + (i - G_W3);
    if (i < G_B1) return P_B2 + (i - G_B2);
    if (i < G_B3) return P_B1 + (i - G_B1);
    return i == G_B3 ? P_B3 : -1;
}

// Weight fragments in BF16 as the training kernel's lanes hold them (lane-contiguous 8-byte
// loads): W1 and W2 with K = inputs (fragments 0..3 and 4 + 4 mt + kt), W2 with K = its outputs
// (20 + 4 mt + kt).  Written once per call by k_mlp_frag and kept up to date by the Adam update.
#define MLP_NFRAG 36
__device__ __forceinline__ void put_frag(unsigned short *__restrict__ frag, int p, float v) {
    const unsigned short b = f2bf(v);
    if (p < P_B1) {
        const int o = p / MLP_IN, k = p % MLP_IN;
        frag[(((o >> 4) * 64) + (k >> 2) * 16 + (o & 15)) * 4 + (k & 3)] = b;
    } else if (p >= P_W2 && p < P_B2) {
        const int j = (p - P_W2) / MLP_H, k = (p - P_W2) % MLP_H, t = (j >> 4) * 4 + (k >> 4);
        frag[((4 + t) * 64 + ((k >> 2) & 3) * 16 + (j & 15)) * 4 + (k & 3)] = b;
        frag[((20 + t) * 64 + ((j >> 2) & 3) * 16 + (k & 15)) * 4 + (j & 3)] = b;
    }
}

__global__ __launch_bounds__(256) void k_mlp_frag(const float *__restrict__ params, unsigned short *__restrict__ frag) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < 4 * 32 * 4) frag[((p >> 7) * 64 + 32) * 4 + (p & 127)] = 0;   // W1: inputs 8..15
    if (p < MLP_NPARAM) put_frag(frag, p, params[p]);
}

int64_t mlp_frag_size() { return (int64_t)MLP_NFRAG * 64 * 4; }

int64_t mlp_partial_size() { return (int64_t)MLP_TR_BLOCKS * MLP_ROW; }

// SAMPLED: training slot i reads pair mix64(...) mod n of (X, T); otherwise pair i
template <bool SAMPLED>
__global__ __launch_bounds__(64 * MLP_TR_WAVES, 1) void k_mlp_train_grad(int64_t nb, int64_t n, uint64_t seed,
                                                                        const float *__restrict__ X,
                                                                        const float *__restrict__ T,
                                                                        const float *__restrict__ params,
                                                                        const bf16x4 *__restrict__ frag,
                                                                        float *__restrict__ partial) {
    __shared__ __align__(16) float sb1[MLP_H], sb2[MLP_H], sw3[MLP_H];
    __shared__ __align__(16) float buf[2][MLP_ROW];
    const int w = threadIdx.x / 64, lane = wave_lane(), c = lane & 15, q = lane >> 4;
    const int64_t stride = (int64_t)gridDim.x * (16 * MLP_TR_WAVES);
    int64_t s = ((int64_t)blockIdx.x * MLP_TR_WAVES + w) * 16 + c;
    // sample c's features 4q .. 4q + 3 and target, requested a step ahead
    float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
    float tv = 0.f;
    auto request = [&]() {
        xv = make_float4(0.f, 0.f, 0.f, 0.f);
        tv = 0.f;
        if (s < nb) {
            const int64_t src = SAMPLED ? (int64_t)(mix64(seed * 0x9E3779B97F4A7C15ull + (uint64_t)s) % (uint64_t)n) : s;
            if (q < 2) xv = *reinterpret_cast<const float4 *>(X + src * MLP_IN + 4 * q);
            tv = T[src];
        }
    };
    // weight fragments: W1 and W2 with K = inputs (either operand), W2 with K = its outputs
    bf16x4 w1[4], w2[4][4], w2t[4][4];
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        w1[mt] = frag[mt * 64 + lane];
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
            w2[mt][kt] = frag[(4 + 4 * mt + kt) * 64 + lane];
            w2t[mt][kt] = frag[(20 + 4 * mt + kt) * 64 + lane];
        }
    }
    request();
    if (threadIdx.x < MLP_H) {
        sb1[threadIdx.x] = params[P_B1 + threadIdx.x];
        sb2[threadIdx.x] = params[P_B2 + threadIdx.x];
        sw3[threadIdx.x] = params[P_W3 + threadIdx.x];
    }
    __syncthreads();
    float b1n[4], b2n[4], w3n[4];
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        b1n[mt] = sb1[mt * 16 + c];
        b2n[mt] = sb2[mt * 16 + c];
        w3n[mt] = sw3[mt * 16 + c];
    }
    const float b3 = params[P_B3];
    f32x4 gw2[4][4] = {}, gw1[4] = {};
    float gw3[4] = {}, gb2[4] = {}, gb1[4] = {}, gb3 = 0.f, loss = 0.f;
    const float fnb = (float)nb, inv_nb = 1.f / fnb;

    while (wave_ballot(s < nb) != 0) {
        const bool valid = s < nb;
        const float t = tv;
        const bf16x4 xb = pack_bf16x4(xv.x, xv.y, xv.z, xv.w);
        s += stride;
        request();
        // x with K = samples: lane (q, c) takes feature c of samples 4q + r (c < 8; the other
        // columns of dW1 are not used)
        bf16x4 xn;
        {
            const uint2 xp = __builtin_bit_cast(uint2, xb);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int from = 4 * q + r + ((c >> 2) & 1) * 16;
                const unsigned lo = __shfl(xp.x, from), hi = __shfl(xp.y, from);
                const unsigned v = (c & 2) ? hi : lo;
                xn[r] = (short)((c & 1) ? (v >> 16) : v);
            }
        }
        // layer 1
        bf16x4 a1t[4], a1n[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            const float4 b = *reinterpret_cast<const float4 *>(&sb1[mt * 16 + 4 * q]);
            const f32x4 dt = mfma16(w1[mt], xb, f32x4{0.f, 0.f, 0.f, 0.f});
            const f32x4 dn = mfma16(xb, w1[mt], f32x4{0.f, 0.f, 0.f, 0.f});
            const float bt[4] = {b.x, b.y, b.z, b.w};
            a1t[mt] = pack_bf16x4(tanh_fast(dt[0] + bt[0]), tanh_fast(dt[1] + bt[1]), tanh_fast(dt[2] + bt[2]),
                                  tanh_fast(dt[3] + bt[3]));
            a1n[mt] = pack_bf16x4(tanh_fast(dn[0] + b1n[mt]), tanh_fast(dn[1] + b1n[mt]), tanh_fast(dn[2] + b1n[mt]),
                                  tanh_fast(dn[3] + b1n[mt]));
        }
        // layer 2 (T): the output, then dz2 = dy w3 (1 - a2^2)
        float a2t[4][4], w3t[4][4];
        float y = 0.f;
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < 4; kt++) d = mfma16(w2[mt][kt], a1t[kt], d);
            const float4 b = *reinterpret_cast<const float4 *>(&sb2[mt * 16 + 4 * q]);
            const float4 v = *reinterpret_cast<const float4 *>(&sw3[mt * 16 + 4 * q]);
            const float bt[4] = {b.x, b.y, b.z, b.w}, vt[4] = {v.x, v.y, v.z, v.w};
            const bf16x4 a2 = pack_bf16x4(tanh_fast(d[0] + bt[0]), tanh_fast(d[1] + bt[1]), tanh_fast(d[2] + bt[2]),
                                          tanh_fast(d[3] + bt[3]));
#pragma unroll
            for (int r = 0; r < 4; r++) {
                a2t[mt][r] = bf2f((unsigned short)a2[r]);
                w3t[mt][r] = vt[r];
                y += a2t[mt][r] * vt[r];
            }
        }
        y += __shfl_xor(y, 16);
        y += __shfl_xor(y, 32);
        y += b3;
        const float e = valid ? y - t : 0.f;
        // e / nb, the product corrected by its exact residual: the rounding of 1/nb alone would be the
        // same error in every gradient
        float dy = e * inv_nb;
        dy = __builtin_fmaf(__builtin_fmaf(-fnb, dy, e), inv_nb, dy);
        if (q == 0) {
            loss += 0.5f * e * e;
            gb3 += dy;
        }
        bf16x4 dz2t[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            float z[4];
#pragma unroll
            for (int r = 0; r < 4; r++) z[r] = dy * w3t[mt][r] * (1.f - a2t[mt][r] * a2t[mt][r]);
            dz2t[mt] = pack_bf16x4(z[0], z[1], z[2], z[3]);
        }
        float dyn[4];
#pragma unroll
        for (int r = 0; r < 4; r++) dyn[r] = __shfl(dy, 4 * q + r);
        // layer 2 (N): dW3, db2, dW2
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < 4; kt++) d = mfma16(a1t[kt], w2[mt][kt], d);
            const bf16x4 a2 = pack_bf16x4(tanh_fast(d[0] + b2n[mt]), tanh_fast(d[1] + b2n[mt]),
                                          tanh_fast(d[2] + b2n[mt]), tanh_fast(d[3] + b2n[mt]));
            float z[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float a = bf2f((unsigned short)a2[r]);
                gw3[mt] += dyn[r] * a;
                z[r] = dyn[r] * w3n[mt] * (1.f - a * a);
            }
            const bf16x4 dz = pack_bf16x4(z[0], z[1], z[2], z[3]);
#pragma unroll
            for (int r = 0; r < 4; r++) gb2[mt] += bf2f((unsigned short)dz[r]);
#pragma unroll
            for (int nt = 0; nt < 4; nt++) gw2[mt][nt] = mfma16(dz, a1n[nt], gw2[mt][nt]);
        }
        // dA1 = dz2 W2 (N), dz1 = dA1 (1 - a1^2): db1, dW1
#pragma unroll
        for (int nt = 0; nt < 4; nt++) {
            f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < 4; kt++) d = mfma16(dz2t[kt], w2t[kt][nt], d);
            float z[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float a = bf2f((unsigned short)a1n[nt][r]);
                z[r] = d[r] * (1.f - a * a);
            }
            const bf16x4 dz = pack_bf16x4(z[0], z[1], z[2], z[3]);
#pragma unroll
            for (int r = 0; r < 4; r++) gb1[nt] += bf2f((unsigned short)dz[r]);
            gw1[nt] = mfma16(dz, xn, gw1[nt]);
        }
    }
    // the per-lane sums over the wave
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        gw3[mt] += __shfl_xor(gw3[mt], 16);
        gw3[mt] += __shfl_xor(gw3[mt], 32);
        gb2[mt] += __shfl_xor(gb2[mt], 16);
        gb2[mt] += __shfl_xor(gb2[mt], 32);
        gb1[mt] += __shfl_xor(gb1[mt], 16);
        gb1[mt] += __shfl_xor(gb1[mt], 32);
    }
    gb3 = wave_sum(gb3);
    loss = wave_sum(loss);
    // the block's sum (w0 + w2) + (w1 + w3), through LDS: waves 2 and 3 put their sums, waves 0
    // and 1 add theirs (each only touches its own lanes' places)
    auto put4 = [&](int i, const f32x4 &v) {
        f32x4 &b = *reinterpret_cast<f32x4 *>(&buf[w & 1][i]);
        b = w >= 2 ? v : v + b;
    };
    auto put1 = [&](int i, float v) { buf[w & 1][i] = w >= 2 ? v : v + buf[w & 1][i]; };
    auto put_all = [&]() {
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
#pragma unroll
            for (int nt = 0; nt < 4; nt++) put4(((mt * 4 + nt) * 64 + lane) * 4, gw2[mt][nt]);
            put4(G_W1 + (mt * 64 + lane) * 4, gw1[mt]);
            if (q == 0) {
                put1(G_W3 + mt * 16 + c, gw3[mt]);
                put1(G_B2 + mt * 16 + c, gb2[mt]);
                put1(G_B1 + mt * 16 + c, gb1[mt]);
            }
        }
        if (lane == 0) {
            put1(G_B3, gb3);
            put1(G_LOSS, loss);
        }
    };
    if (w >= 2) put_all();
    __syncthreads();
    if (w < 2) put_all();
    __syncthreads();
    f32x4 *g = reinterpret_cast<f32x4 *>(partial + (int64_t)blockIdx.x * MLP_ROW);
    for (int i = threadIdx.x; i < (G_LOSS + 4) / 4; i += 64 * MLP_TR_WAVES)
        g[i] = reinterpret_cast<const f32x4 *>(buf[0])[i] + reinterpret_cast<const f32x4 *>(buf[1])[i];
}

// Folds the blocks' partials in a fixed order (deterministic) -- 16 wavefronts take every 16th
// partial, then their sums in wavefront order -- and, with ADAM, updates the FP32 master weights
// (beta1 0.9, beta2 0.999, eps 1e-8) in the same launch; loss = mean of 0.5 (y - t)^2.
#define MLP_RED_WAVES 16
template <bool ADAM>
__global__ __launch_bounds__(64 * MLP_RED_WAVES) void k_mlp_reduce(int nblk, int64_t nb,
                                                                  const float *__restrict__ partial,
                                                                  float *__restrict__ grad, float *__restrict__ loss,
                                                                  float *__restrict__ params, float *__restrict__ m1,
                                                                  float *__restrict__ m2,
                                                                  unsigned short *__restrict__ frag, float lr,
                                                                  float bc1, float bc2) {
    __shared__ float sum[MLP_RED_WAVES][64];
    const int w = threadIdx.x / 64, lane = wave_lane();
    const int i = blockIdx.x * 64 + lane;   // < MLP_ROW
    float s = 0.f;
#pragma unroll 8
    for (int b = w; b < nblk; b += MLP_RED_WAVES) s += partial[(int64_t)b * MLP_ROW + i];
    sum[w][lane] = s;
    __syncthreads();
    if (w != 0) return;
    s = sum[0][lane];
#pragma unroll
    for (int v = 1; v < MLP_RED_WAVES; v++) s += sum[v][lane];
    if (i == G_LOSS) *loss = s / (float)nb;
    const int p = mlp_param_of(i);
    if (p < 0) return;
    grad[p] = s;
    if (ADAM) {
        const float a = 0.9f * m1[p] + 0.1f * s;
        const float b = 0.999f * m2[p] + 0.001f * s * s;
        m1[p] = a;
        m2[p] = b;
        const float v = params[p] - lr * (a / bc1) / (sqrtf(b / bc2) + 1e-8f);
        params[p] = v;
        put_frag(frag, p, v);
    }
}

// ------------------------------------------------------------------------------------
void launch_mlp_features(mhpc_ctx *c, double dt) {
    if (c->n <= 0) return;
    double **f = c->f;
    hipLaunchKernelGGL(k_mlp_features, dim3((unsigned)ceil_div(c->n, 256)), dim3(256), 0, c->stream, c->n,
                       f[MHPC_F_SML], c->noi, f[MHPC_F_RHO], f[MHPC_F_DRHODT], f[MHPC_F_CURLV],
                       f[MHPC_F_GRADRHO], f[MHPC_F_CS], dt, c->p.n_target, c->mlp_norm,
                       c->mlp_norm_set ? MLP_CLIP : 3.0e38f, c->mlp_x, c->mlp_hprev);
}

void launch_mlp_predict(mhpc_ctx *c) {
    if (c->n <= 0) return;
    const unsigned g = (unsigned)std::min<int64_t>(ceil_div(c->n, 16 * MLP_INF_WAVES), MLP_INF_BLOCKS);
    hipLaunchKernelGGL(k_mlp_predict, dim3(g), dim3(64 * MLP_INF_WAVES), 0, c->stream, c->n, c->mlp_x,
                       c->mlp_params, c->mlp_norm, c->mlp_hprev, c->f[MHPC_F_SML]);
}

void launch_mlp_forward_raw(mhpc_ctx *c, int64_t n, const float *X, float *Y) {
    const unsigned g = (unsigned)std::min<int64_t>(ceil_div(n, 16 * MLP_INF_WAVES), MLP_INF_BLOCKS);
    hipLaunchKernelGGL(k_mlp_forward_raw, dim3(g), dim3(64 * MLP_INF_WAVES), 0, c->stream, n, X,
                       c->mlp_params, Y);
}

static unsigned mlp_train_blocks(int64_t nb) {
    return (unsigned)std::min<int64_t>(ceil_div(nb, 16 * MLP_TR_WAVES), MLP_TR_BLOCKS);
}

// the training kernel's weight fragments from the master weights
void launch_mlp_frag(mhpc_ctx *c) {
    hipLaunchKernelGGL(k_mlp_frag, dim3((unsigned)ceil_div(MLP_NPARAM, 256)), dim3(256), 0, c->stream,
                       c->mlp_params, c->mlp_frag);
}

// one gradient evaluation over the nb pairs (X, T); grad and loss on the device
void launch_mlp_gradient(mhpc_ctx *c, int64_t nb, const float *X, const float *T, float *grad, float *loss) {
    const unsigned blocks = mlp_train_blocks(nb);
    hipLaunchKernelGGL(k_mlp_train_grad<false>, dim3(blocks), dim3(64 * MLP_TR_WAVES), 0, c->stream, nb, nb,
                       (uint64_t)0, X, T, c->mlp_params, reinterpret_cast<const bf16x4 *>(c->mlp_frag), c->mlp_partial);
    hipLaunchKernelGGL(k_mlp_reduce<false>, dim3(MLP_ROW / 64), dim3(64 * MLP_RED_WAVES), 0, c->stream, (int)blocks,
                       nb, c->mlp_partial, grad, loss, nullptr, nullptr, nullptr, nullptr, 0.f, 1.f, 1.f);
}

// one Adam step on nsamples random pairs of the context's features and targets
void launch_mlp_train_step(mhpc_ctx *c, int64_t nsamples, uint64_t seed, float lr, int step) {
    const unsigned blocks = mlp_train_blocks(nsamples);
    const float bc1 = 1.f - powf(0.9f, (float)step), bc2 = 1.f - powf(0.999f, (float)step);
    hipLaunchKernelGGL(k_mlp_train_grad<true>, dim3(blocks), dim3(64 * MLP_TR_WAVES), 0, c->stream, nsamples, c->n,
                       seed, c->mlp_x, c->mlp_t, c->mlp_params, reinterpret_cast<const bf16x4 *>(c->mlp_frag),
                       c->mlp_partial);
    hipLaunchKernelGGL(k_mlp_reduce<true>, dim3(MLP_ROW / 64), dim3(64 * MLP_RED_WAVES), 0, c->stream, (int)blocks,
                       nsamples, c->mlp_partial, c->mlp_grad, c->mlp_loss, c->mlp_params, c->mlp_m1, c->mlp_m2,
                       c->mlp_frag, lr, bc1, bc2);
}

// training targets: T = (log(sml / h_previous) - mu_t) / sigma_t for every particle
__global__ __launch_bounds__(256) void k_mlp_targets(int64_t n, const double *__restrict__ h,
                                                     const double *__restrict__ hprev,
                                                     const float *__restrict__ norm, float *__restrict__ T) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) T[i] = (float)((log(h[i] / hprev[i]) - norm[16]) / norm[17]);
}

void launch_mlp_targets(mhpc_ctx *c) {
    if (c->n <= 0) return;
    hipLaunchKernelGGL(k_mlp_targets, dim3((unsigned)ceil_div(c->n, 256)), dim3(256), 0, c->stream, c->n,
                       c->f[MHPC_F_SML], c->mlp_hprev, c->mlp_norm, c->mlp_t);
}
