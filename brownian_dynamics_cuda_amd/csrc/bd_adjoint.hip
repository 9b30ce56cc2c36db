// bd_adjoint.hip -- the core-core charge term of the force pass and its
// adjoint, for the differentiable trajectory (torch.autograd.Function in
// brownian_dynamics_cuda_amd/diff.py).
//
// Term (func.cpp:1489-1566): for two cores i, j within the 25 nm bead
// rule and every pair of their point charges k (on i) and l (on j), with
// z = Q_k - Q_l, d = |z|,
//   E  = ke q_k q_l exp(-kappa d) / d  +  [d <= 8] kex ((s/d)^12 - (s/d)^6)
//   f_k = g(d) z/d = -f_l,   g = -dE/dd
//       = ke q_k q_l exp(-kappa d) (kappa d + 1) / d^2
//         + [d <= 8] kex (12 (s/d)^12 - 6 (s/d)^6) / d.
// Here the output is the force on every charge site (the caller turns it
// into core forces and body-frame torques, whose derivatives torch takes)
// and each core's half of its pairs' energy.
//
// Adjoint: with lambda_k = dLoss/df_k and eps_i = dLoss/de_i, a pair adds
//   phi = (lambda_k - lambda_l) . g z/d + (eps_i + eps_j)/2 E
// to the loss; with u = lambda_k - lambda_l and uz = u . z/d,
//   dphi/dQ_k = g'(d) uz z/d + g(d) (u - uz z/d) / d - eps g z/d = -dphi/dQ_l,
//   g'_DH = -ke q_k q_l exp(-kappa d) (kappa^2 d^2 + 2 kappa d + 2) / d^3,
//   g'_EV = kex (-156 (s/d)^12 + 42 (s/d)^6) / d^2,
// and dphi/dq_k = q_l (uz gh + eps eh) with gh = g_DH / (q_k q_l),
// eh = E_DH / (q_k q_l) (the excluded volume does not depend on charge).
//
// Layout: a workgroup of NT threads owns a block of KB charges of a core i
// (blockIdx.y), one per lane; the partner charges of the core (CSR list, both directions)
// pass through LDS as one stream of records, NT at a time, dealt over the workgroup's
// wavefronts (and, for KB < 64, over the lanes' groups of KB), and their
// partial sums are added in a fixed order at the end.  Every pair is
// evaluated from both sides, so each site's output has one owner and there
// are no atomics: the results are deterministic.  A core's energy needs its
// blocks' parts: with a work buffer each of several blocks leaves its part there
// and k_cc_esum adds them, without one a single workgroup takes all the core's
// blocks in turn (bd_cc_forward).
//
// What bounds it: FP32 (FP64) VALU issue, ~40 instructions a pair forward and
// ~55 backward.  With one 256-thread workgroup per core (300 charges: three
// rounds, the last with 44 lanes) 50 cores kept 50 of 256 CUs at 4 wavefronts
// each, and the IEEE root, quotient and expf of a pair were most of its
// instructions.  50 cores of 300 charges, forward and backward: 3692 -> 135 us
// in FP32, 4734 -> 301 us in FP64; 300 cores 3982 -> 672 and 6277 -> 1581 us.
// Templated on the arithmetic (float for the FP32 force passes of the
// differentiable trajectory, double for its FP64 checks).
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>

#include "../../include/bd_hip.h"
#include "bd_kernels.h"

namespace bd {
namespace {

constexpr int kMaxSites = 640;  // charges per core

struct CCParams {
    double ke, kappa, kex, sigma;
};

// The distance terms of a pair in the two arithmetics: 1/d and d from d2,
// exp(-kappa d), and the reference's d <= 8 as a test of d2 (the largest
// number whose correctly rounded root is 8).
template <typename T> struct Arith;
template <> struct Arith<float> {
    static constexpr float kD8 = 0x1.000002p+6f;
    static __device__ __forceinline__ float rsqrt(float f) {  // v_rsq_f32 and one Newton step
        const float y = __builtin_amdgcn_rsqf(f);
        return __builtin_fmaf(0.5f * y, __builtin_fmaf(-f * y, y, 1.0f), y);
    }
    // e^x = 2^(x log2 e), the product's rounding error carried into a factor
    static __device__ __forceinline__ float exp(float x) {
        const float p = x * 0x1.715476p+0f;
        const float e = __builtin_fmaf(x, 0x1.4ae0cp-26f, __builtin_fmaf(x, 0x1.715476p+0f, -p));
        const float y = __builtin_amdgcn_exp2f(p);
        return __builtin_fmaf(y, e * 0x1.62e43p-1f, y);
    }
};
template <> struct Arith<double> {
    static constexpr double kD8 = 0x1.0000000000001p+6;
    static __device__ __forceinline__ double rsqrt(double f) { return rsqrt_f64(f); }
    // below -745 the result is 0; exp_neg takes arguments above -800
    static __device__ __forceinline__ double exp(double x) { return exp_neg(fmax(x, -800.0)); }
};

template <typename T>
struct PairTerms {
    T id, g, gp, e, gh, eh;  // 1/d, g, g', energy, g_DH/(q_k q_l), E_DH/(q_k q_l)
};

template <typename T, bool GP>
__device__ __forceinline__ PairTerms<T> pair_terms(T d2, T qkql, const CCParams &p) {
    const T kap = (T)p.kappa, ke = (T)p.ke;
    const T id = Arith<T>::rsqrt(d2), kd = kap * (d2 * id);
    PairTerms<T> r;
    r.id = id;
    r.eh = ke * Arith<T>::exp(-kd) * id;
    r.gh = r.eh * (kd + T(1)) * id;
    r.e = qkql * r.eh;
    r.g = qkql * r.gh;
    if (GP) r.gp = -qkql * r.eh * (kd * (kd + T(2)) + T(2)) * (id * id);
    if (d2 <= Arith<T>::kD8) {
        const T sd = (T)p.sigma * id, s2 = sd * sd, s6 = s2 * s2 * s2, s12 = s6 * s6, kex = (T)p.kex;
        r.e += kex * (s12 - s6);
        r.g += kex * (T(12) * s12 - T(6) * s6) * id;
        if (GP) r.gp += kex * (T(-156) * s12 + T(42) * s6) * (id * id);
    }
    return r;
}

template <typename T> struct alignas(4 * sizeof(T)) Rec4 {
    T x, y, z, w;
};

// The sums v of the workgroup's slots (SL slots of KB lanes), added in slot
// order by the first KB NV threads: result of value u of lane k on thread
// u KB + k.
template <typename T, int KB, int NT, int NV>
__device__ __forceinline__ T slot_sum(const T (&v)[NV], T *buf) {
    constexpr int SL = NT / KB;
    const int k = threadIdx.x % KB, s = threadIdx.x / KB;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NV; u++) buf[(s * NV + u) * KB + k] = v[u];
    __syncthreads();
    T t = T(0);
    if (threadIdx.x < KB * NV)
        for (int i = 0; i < SL; i++) t += buf[i * NV * KB + threadIdx.x];
    return t;
}

// f[i][k][3] of the block's charges, and half the energy of its pairs into
// eo: e[i] where the workgroup takes every block (gridDim.y = 1), else the
// block's part work[i gridDim.y + block]
template <typename T, int KB, int NT>
__global__ void __launch_bounds__(NT) k_cc_fwd(int Nq, const T *__restrict__ Q, const T *__restrict__ q,
                                                     const int *__restrict__ off, const int *__restrict__ nbr,
                                                     CCParams p, T *__restrict__ f, T *__restrict__ eo) {
    constexpr int SL = NT / KB;
    __shared__ Rec4<T> S[NT];
    const int i = blockIdx.x, slot = threadIdx.x / KB, s0 = off[i], M = (off[i + 1] - s0) * Nq;
    static_assert(sizeof(S) >= NT * 4 * sizeof(T), "the slots' sums take the records' place");
    T en = T(0);
    for (int k0 = blockIdx.y * KB; k0 < Nq; k0 += gridDim.y * KB) {
        const int k = min(k0 + (int)threadIdx.x % KB, Nq - 1);
        const T *src = Q + ((size_t)i * Nq + k) * 3;
        const T px = src[0], py = src[1], pz = src[2], qk = q[k];
        T v[4] = {T(0), T(0), T(0), T(0)};
        for (int t0 = 0; t0 < M; t0 += NT) {
            const int R = min(M - t0, NT);
            __syncthreads();
            for (int r = threadIdx.x; r < R; r += NT) {
                const int m = t0 + r, l = m % Nq;
                const T *o = Q + ((size_t)nbr[s0 + m / Nq] * Nq + l) * 3;
                S[r] = Rec4<T>{o[0], o[1], o[2], q[l]};
            }
            __syncthreads();
#pragma unroll 2
            for (int r = slot; r < R; r += SL) {
                const Rec4<T> o = S[r];
                const T zx = px - o.x, zy = py - o.y, zz = pz - o.z;
                const PairTerms<T> t = pair_terms<T, false>(zx * zx + zy * zy + zz * zz, qk * o.w, p);
                const T gi = t.g * t.id;
                v[0] += gi * zx;
                v[1] += gi * zy;
                v[2] += gi * zz;
                v[3] += t.e;
            }
        }
        const T sum = slot_sum<T, KB, NT, 4>(v, reinterpret_cast<T *>(S));
        const int u = threadIdx.x / KB, kk = k0 + threadIdx.x % KB;
        if (threadIdx.x < 3 * KB && kk < Nq) f[((size_t)i * Nq + kk) * 3 + u] = sum;
        if (u == 3 && kk < Nq) en += T(0.5) * sum;
    }
    // the energy sits in the KB lanes of value 3
    if (threadIdx.x >= 3 * KB && threadIdx.x < 4 * KB) {
        for (int o = KB / 2; o > 0; o >>= 1) en += __shfl_down(en, o, KB);
        if (threadIdx.x == 3 * KB) eo[(size_t)i * gridDim.y + blockIdx.y] = en;
    }
}

// e[i] = the parts of core i in order
template <typename T>
__global__ void k_cc_esum(int n_c, int parts, const T *__restrict__ work, T *__restrict__ e) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_c) return;
    T t = T(0);
    for (int b = 0; b < parts; b++) t += work[(size_t)i * parts + b];
    e[i] = t;
}

// gQ[i][k][3] and gq[i][k] (per-site charge gradient; the template
// gradient is its sum over cores), both written
template <typename T, int KB, int NT>
__global__ void __launch_bounds__(NT) k_cc_bwd(int Nq, const T *__restrict__ Q, const T *__restrict__ q,
                                                     const int *__restrict__ off, const int *__restrict__ nbr,
                                                     CCParams p, const T *__restrict__ gf, const T *__restrict__ ge,
                                                     T *__restrict__ gQ, T *__restrict__ gqs) {
    constexpr int SL = NT / KB;
    __shared__ Rec4<T> S[2 * NT];
    const int i = blockIdx.x, slot = threadIdx.x / KB, s0 = off[i], M = (off[i + 1] - s0) * Nq;
    const int k0 = blockIdx.y * KB, k = min(k0 + (int)threadIdx.x % KB, Nq - 1);
    const size_t ok = ((size_t)i * Nq + k) * 3;
    const T px = Q[ok], py = Q[ok + 1], pz = Q[ok + 2], lx = gf[ok], ly = gf[ok + 1], lz = gf[ok + 2], qk = q[k];
    const T ei = ge[i];
    T v[4] = {T(0), T(0), T(0), T(0)};
    for (int t0 = 0; t0 < M; t0 += NT) {
        const int R = min(M - t0, NT);
        __syncthreads();
        for (int r = threadIdx.x; r < R; r += NT) {
            const int m = t0 + r, l = m % Nq, j = nbr[s0 + m / Nq];
            const size_t o = ((size_t)j * Nq + l) * 3;
            S[2 * r] = Rec4<T>{Q[o], Q[o + 1], Q[o + 2], q[l]};
            S[2 * r + 1] = Rec4<T>{gf[o], gf[o + 1], gf[o + 2], T(0.5) * (ei + ge[j])};
        }
        __syncthreads();
        for (int r = slot; r < R; r += SL) {
            const Rec4<T> o = S[2 * r], w = S[2 * r + 1];
            const T zx = px - o.x, zy = py - o.y, zz = pz - o.z;
            const PairTerms<T> t = pair_terms<T, true>(zx * zx + zy * zy + zz * zz, qk * o.w, p);
            const T ux = lx - w.x, uy = ly - w.y, uz_ = lz - w.z;
            const T hx = zx * t.id, hy = zy * t.id, hz = zz * t.id;
            const T uz = ux * hx + uy * hy + uz_ * hz;
            const T b = t.g * t.id, a = t.gp * uz - w.w * t.g - b * uz;
            v[0] += a * hx + b * ux;
            v[1] += a * hy + b * uy;
            v[2] += a * hz + b * uz_;
            v[3] += o.w * (uz * t.gh + w.w * t.eh);
        }
    }
    const T sum = slot_sum<T, KB, NT, 4>(v, reinterpret_cast<T *>(S));
    const int u = threadIdx.x / KB, kk = k0 + threadIdx.x % KB;
    if (kk < Nq) {
        if (u < 3) gQ[((size_t)i * Nq + kk) * 3 + u] = sum;
        else if (u == 3) gqs[(size_t)i * Nq + kk] = sum;
    }
}

// Charges and threads of a block.  16 charges, with fewer idle lanes in the last
// block (300 charges: 304 lanes against 320) and more workgroups, until the
// blocks of 64 alone are several rounds of workgroups, which then read half the
// records from LDS; 64 only if their lanes are hardly more (5 charges: 64 lanes
// against 16).  Forward and backward with 64 / 16 in turn, us: 20 cores of 300
// FP32 142 / 110, FP64 270 / 158; 50 cores 158 / 152, 306 / 334; 120 cores 382 /
// 332, 826 / 731; 300 cores 741 / 760, 1629 / 1726.  1024 threads share a core's
// records, but for cores of one block and many of them, where the launch of the
// wavefronts counts: forward with 1024 / 256 threads, 16 charges, us: 1000 cores
// with 2 partners FP32 6.4 / 5.2, FP64 9.5 / 5.5, with 80 partners 21.0 / 22.8 and
// 46.1 / 40.7; 2048 cores 10.4 / 5.0, 16.4 / 7.1, 37.4 / 37.1, 92.1 / 74.5.
struct Shape {
    int KB, NT;
};
template <typename T>
Shape block_shape(int n_c, int Nq) {
    const int b64 = (Nq + 63) / 64, b16 = (Nq + 15) / 16;
    if (b16 == 1 && n_c >= (sizeof(T) == 8 ? 1000 : 2048)) return {16, 256};
    if ((long long)n_c * b64 >= 1000 && 10 * 64 * b64 <= 11 * 16 * b16) return {64, 1024};
    return {16, 1024};
}

template <typename T>
void cc_fwd(int n_c, int Nq, const void *Q, const void *q, const int *off, const int *nbr, const CCParams &p, void *f,
            void *e, void *work, hipStream_t s) {
    const Shape b = work || Nq <= 16 ? block_shape<T>(n_c, Nq) : Shape{64, 1024};
    const int nb = work ? (Nq + b.KB - 1) / b.KB : 1;
    // a core of one block has its energy from that
    auto *eo = static_cast<T *>(nb > 1 ? work : e);
    auto launch = [&](auto kernel) {
        kernel<<<dim3(n_c, nb), b.NT, 0, s>>>(Nq, (const T *)Q, (const T *)q, off, nbr, p, (T *)f, eo);
    };
    if (b.KB == 64) launch(k_cc_fwd<T, 64, 1024>);
    else if (b.NT == 1024) launch(k_cc_fwd<T, 16, 1024>);
    else launch(k_cc_fwd<T, 16, 256>);
    if (nb > 1) k_cc_esum<T><<<(n_c + 255) / 256, 256, 0, s>>>(n_c, nb, eo, (T *)e);
}

template <typename T>
void cc_bwd(int n_c, int Nq, const void *Q, const void *q, const int *off, const int *nbr, const CCParams &p,
            const void *gf, const void *ge, void *gQ, void *gqs, hipStream_t s) {
    const Shape b = block_shape<T>(n_c, Nq);
    auto launch = [&](auto kernel) {
        kernel<<<dim3(n_c, (Nq + b.KB - 1) / b.KB), b.NT, 0, s>>>(Nq, (const T *)Q, (const T *)q, off, nbr, p, (const T *)gf,
                                                                  (const T *)ge, (T *)gQ, (T *)gqs);
    };
    if (b.KB == 64) launch(k_cc_bwd<T, 64, 1024>);
    else if (b.NT == 1024) launch(k_cc_bwd<T, 16, 1024>);
    else launch(k_cc_bwd<T, 16, 256>);
}

int cc_fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    set_last_error(buf);
    return code;
}

int cc_check(int n_c, int Nq, const void *Q, const void *q, const int *off, const int *nbr) {
    if (n_c < 1 || Nq < 1 || Nq > kMaxSites)
        return cc_fail(BD_E_ARG, "need n_c >= 1 and 1 <= Nq <= %d (n_c=%d, Nq=%d)", kMaxSites, n_c, Nq);
    if (!Q || !q || !off || !nbr) return cc_fail(BD_E_ARG, "null argument");
    return BD_OK;
}

}  // namespace
}  // namespace bd

using namespace bd;

extern "C" {

int bd_cc_forward_work(int fp64, int n_c, int Nq, const void *Q, const void *q, const int *nbr_off, const int *nbr,
                       double ke, double kappa, double kex, double sigma, void *f, void *e, void *work,
                       void *stream) {
    int r = cc_check(n_c, Nq, Q, q, nbr_off, nbr);
    if (r) return r;
    if (!f || !e) return cc_fail(BD_E_ARG, "null output");
    const CCParams p{ke, kappa, kex, sigma};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (fp64) cc_fwd<double>(n_c, Nq, Q, q, nbr_off, nbr, p, f, e, work, s);
    else cc_fwd<float>(n_c, Nq, Q, q, nbr_off, nbr, p, f, e, work, s);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return cc_fail(BD_E_HIP, "k_cc_fwd: %s", hipGetErrorString(err));
    return BD_OK;
}

int bd_cc_forward(int fp64, int n_c, int Nq, const void *Q, const void *q, const int *nbr_off, const int *nbr,
                  double ke, double kappa, double kex, double sigma, void *f, void *e, void *stream) {
    return bd_cc_forward_work(fp64, n_c, Nq, Q, q, nbr_off, nbr, ke, kappa, kex, sigma, f, e, nullptr, stream);
}

int bd_cc_backward(int fp64, int n_c, int Nq, const void *Q, const void *q, const int *nbr_off, const int *nbr,
                   double ke, double kappa, double kex, double sigma, const void *gf, const void *ge, void *gQ,
                   void *gq_sites, void *stream) {
    int r = cc_check(n_c, Nq, Q, q, nbr_off, nbr);
    if (r) return r;
    if (!gf || !ge || !gQ || !gq_sites) return cc_fail(BD_E_ARG, "null argument");
    const CCParams p{ke, kappa, kex, sigma};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (fp64) cc_bwd<double>(n_c, Nq, Q, q, nbr_off, nbr, p, gf, ge, gQ, gq_sites, s);
    else cc_bwd<float>(n_c, Nq, Q, q, nbr_off, nbr, p, gf, ge, gQ, gq_sites, s);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return cc_fail(BD_E_HIP, "k_cc_bwd: %s", hipGetErrorString(err));
    return BD_OK;
}

}  // extern "C"
