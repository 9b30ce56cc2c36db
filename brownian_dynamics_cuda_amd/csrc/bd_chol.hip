// bd_chol.hip -- RPY diffusion tensor, blocked Cholesky and the noise
// displacement rd = s2dt * L * p on gfx950.
//
// Replaces Diffusion_Tensor_CUDA + cusolverDnDpotrf + Cholesky_Decomposition_mod
// + rd_cal (func_cuda.cu:500-647, 3504-3552).  The factor follows the CPU
// Cholesky of func.cpp:806-836, including |f| for a negative pivot.
//
// Matrix: row-major, lower triangle, padded to a multiple of 64 with an
// identity block (so the padded factor is [[L,0],[0,I]] and no kernel needs
// a bounds test).  Right-looking blocked algorithm with 64x64 tiles, one
// launch per block column kb (k_step, k_step2): every workgroup forms the two panel
// tiles it needs as A_ib,kb inv(L_kb,kb)^T (FP64 matrix cores), updates its
// trailing tile A_ib,jb -= L_ib,kb L_jb,kb^T (FP64, FP32 or three-slice
// BF16 matrix-core products), and the workgroup owning tile (kb+1,kb+1)
// then factors it and inverts the factor (four wavefronts, FP64, one
// elimination of the tile and the identity).  The solved off-diagonal tile L_ib,kb
// stays parked in the upper block (kb, ib) of the same storage.
//
// Large matrices take super-panels of NB block columns instead: the panel
// columns are factored as above with their updates restricted to the panel,
// and the trailing matrix then receives the whole panel at once (each tile
// accumulates K = 64 NB in registers before its one read-modify-write), so the trailing matrix streams through HBM once per
// NB block columns rather than once per block column.  The panel tiles lie
// once more in the operand order of the matrix cores for it (k_trail_pk; in
// BF16 split into slices, k_trail_bf).  Panels of eight in FP64 and FP32
// (chol_panels) factor only their diagonal block column by column, beside
// tiles of the trailing update before it (k_block_step), and solve the rows
// below in one launch (k_panel_rows).  In the FP32 and BF16 modes only the
// trailing update takes the reduced precision; the panel's own columns stay
// FP64.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "bd_dev.h"
#include "bd_kernels.h"

namespace bd {

constexpr int TB = 64;        // tile edge
constexpr int LDP = TB + 1;   // LDS row pitch (doubles)
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef float flt4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

static inline int nblk(long long n, int t) { return (int)((n + t - 1) / t); }

// ---------------------------------------------------------------------------
// RPY tensor assembly (func.cpp:737-804): one workgroup per lower 64x64
// tile, a thread per bead pair whose 3x3 block meets the tile (the pair's
// distance terms evaluated once, each entry by the reference's expression),
// staged in LDS and stored row by row; zeros above the diagonal and the
// identity padding.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double3 hi_pos(const Stat &s, const Geo &g, int b) {
    if (b < s.n) return ld3(g.r + 3 * b);
    b -= s.n;
    if (b < s.n_tail) return ld3(g.r_t + 3 * b);
    return ld3(g.r_lh + 3 * (b - s.n_tail));
}

// M[k][l] for beads i != j at ri, rj (func.cpp:754-796)
__device__ __forceinline__ void rpy_block(double3 ri, double3 rj, double radi, double radj, double a1, double a2,
                                          double (&M)[3][3]) {
    const double sij[3] = {ri.x - rj.x, ri.y - rj.y, ri.z - rj.z};
    const double ssq = rpy_ssq(ri - rj);
    const double s = sqrt(ssq);
    if (rpy_far(ssq, radi + radj)) {
        const double f = (radi * radi + radj * radj) / ssq;
        const double f1 = 1.0 + f / 3, f2 = 1.0 - f, c = a2 / s;
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int l = 0; l < 3; l++)
                M[k][l] = (k == l) ? c * (f1 + f2 * sij[k] * sij[k] / ssq) : c * (f2 * sij[k] * sij[l] / ssq);
    } else {
        const double se = pow((radi * radi * radi + radj * radj * radj) / 2.0, 1.0 / 3);
        const double sq = sqrt(ssq), c = a1 / se;
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int l = 0; l < 3; l++)
                M[k][l] = (k == l) ? c * (1.0 - 9.0 * sq / (32 * se) + 3.0 * sij[k] * sij[k] / (32.0 * se * sq))
                                   : c * (3.0 * sij[k] * sij[l] / (32.0 * se * sq));
    }
}

__device__ __forceinline__ void tri_index(int idx, int &i, int &j) {
    // idx -> (i, j), 0 <= j <= i, row-major over the lower triangle
    int r = (int)((sqrt(8.0 * idx + 1.0) - 1.0) * 0.5);
    while ((r + 1) * (r + 2) / 2 <= idx) r++;
    while (r * (r + 1) / 2 > idx) r--;
    i = r;
    j = idx - r * (r + 1) / 2;
}

constexpr int kDiagLds = 5408;  // LDS of diag_factor_inv, doubles
__device__ __forceinline__ void diag_factor_inv(double *lds, double *T, double *A, int ld, int d0, double *Linv,
                                                int *neg);

// FACTOR: workgroup 0 (tile (0,0)) then factors and inverts its tile in
// place of a separate first-tile launch, beside the other tiles' assembly
// (every workgroup then carries the factor's LDS).
template <bool FACTOR>
__global__ void __launch_bounds__(256) k_rpy(Stat s, Geo g, const double *rad_all, double *A, int m, int ld,
                                             double a1, double a2, int *neg, double *Linv) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *neg = 0;  // negative-pivot count of the factor that follows
    __shared__ double T[FACTOR ? kDiagLds : TB * LDP];
    int ti, tj;
    tri_index(blockIdx.x, ti, tj);
    const int r0 = ti * TB, c0 = tj * TB, nhi = m / 3;
    // beads whose rows / columns meet the tile
    const int bi0 = r0 / 3, bj0 = c0 / 3;
    const int nbi = max(0, min((r0 + TB - 1) / 3, nhi - 1) - bi0 + 1);
    const int nbj = max(0, min((c0 + TB - 1) / 3, nhi - 1) - bj0 + 1);
    for (int p = threadIdx.x; p < nbi * nbj; p += blockDim.x) {
        const int i = bi0 + p / nbj, j = bj0 + p % nbj;
        if (j > i) continue;
        double M[3][3];
        if (i == j) {
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int l = 0; l < 3; l++) M[k][l] = (k == l) ? a1 / rad_all[i] : 0.0;
        } else {
            rpy_block(hi_pos(s, g, i), hi_pos(s, g, j), rad_all[i], rad_all[j], a1, a2, M);
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int row = 3 * i + k - r0;
            if (row < 0 || row >= TB) continue;
#pragma unroll
            for (int l = 0; l < 3; l++) {
                const int col = 3 * j + l - c0;
                if (col >= 0 && col < TB) T[row * LDP + col] = M[k][l];
            }
        }
    }
    __syncthreads();
    const bool fac = FACTOR && blockIdx.x == 0;
    for (int e = threadIdx.x; e < TB * TB; e += blockDim.x) {
        const int row = r0 + e / TB, col = c0 + e % TB;
        double v;
        if (col > row) v = 0.0;
        else if (row >= m || col >= m) v = (row == col) ? 1.0 : 0.0;
        else v = T[(e / TB) * LDP + e % TB];
        if (fac) T[(e / TB) * LDP + e % TB] = v;  // the factor writes L here instead
        else A[(size_t)row * ld + col] = v;
    }
    if constexpr (FACTOR) {
        if (fac) {
            __syncthreads();
            diag_factor_inv(T, T, A, ld, 0, Linv, neg);
        }
    }
}

// ---------------------------------------------------------------------------
// tile helpers
// ---------------------------------------------------------------------------
// Tile copies between global memory and LDS (pitch LDP) by the 256 threads
// of a workgroup, 16-byte accesses, fully unrolled: all eight global loads
// of a thread are in flight before the first LDS store waits on them.
constexpr int NTHR = 256;
// thread of the team of 256 that works on a tile (k_step2 has two teams in a
// workgroup)
__device__ __forceinline__ int tid() { return threadIdx.x & (NTHR - 1); }
__device__ __forceinline__ void load_tile(const double *A, int ld, int r0, int c0, double *S) {
    dbl2 v[TB * TB / 2 / NTHR];
#pragma unroll
    for (int i = 0; i < TB * TB / 2 / NTHR; i++) {
        const int e = tid() + i * NTHR, r = e / (TB / 2), c = 2 * (e % (TB / 2));
        v[i] = *reinterpret_cast<const dbl2 *>(A + (size_t)(r0 + r) * ld + c0 + c);
    }
#pragma unroll
    for (int i = 0; i < TB * TB / 2 / NTHR; i++) {
        const int e = tid() + i * NTHR, r = e / (TB / 2), c = 2 * (e % (TB / 2));
        S[r * LDP + c] = v[i].x;
        S[r * LDP + c + 1] = v[i].y;
    }
}
__device__ __forceinline__ void store_tile(double *A, int ld, int r0, int c0, const double *S, bool lower_only) {
#pragma unroll
    for (int i = 0; i < TB * TB / 2 / NTHR; i++) {
        const int e = tid() + i * NTHR, r = e / (TB / 2), c = 2 * (e % (TB / 2));
        dbl2 v;
        v.x = (lower_only && c > r) ? 0.0 : S[r * LDP + c];
        v.y = (lower_only && c + 1 > r) ? 0.0 : S[r * LDP + c + 1];
        if (!lower_only || c <= r) *reinterpret_cast<dbl2 *>(A + (size_t)(r0 + r) * ld + c0 + c) = v;
    }
}

// acc += As * Bs^T for a 64x64 tile; 4 waves, each a 32x32 quarter as 2x2
// tiles of v_mfma_f64_16x16x4f64.  Lane l supplies A[l%16][l/16] and
// B^T[l/16][l%16]; result register v of lane l is C[l/16 + 4v][l%16]
// (measured on gfx950; the FP32 16x16x4 form places it at C[4(l/16)+v]).
__device__ __forceinline__ void mma_f64(const double *As, const double *Bs, dbl4 acc[2][2]) {
    const int lane = tid() & 63, w = tid() >> 6;
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32, i16 = lane & 15, k4 = lane >> 4;
    // the operands of K step kk + 4 are read while the products of step kk run
    const double *pa0 = As + (wr + i16) * LDP + k4, *pa1 = pa0 + 16 * LDP;
    const double *pb0 = Bs + (wc + i16) * LDP + k4, *pb1 = pb0 + 16 * LDP;
    double na0 = pa0[0], na1 = pa1[0], nb0 = pb0[0], nb1 = pb1[0];
#pragma unroll
    for (int kk = 0; kk < TB; kk += 4) {
        const double a0 = na0, a1 = na1, b0 = nb0, b1 = nb1;
        if (kk + 4 < TB) {
            na0 = pa0[kk + 4];
            na1 = pa1[kk + 4];
            nb0 = pb0[kk + 4];
            nb1 = pb1[kk + 4];
        }
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
}

// Same product with FP32 operands and FP32 accumulation
// (v_mfma_f32_16x16x4f32, identical lane layout).
__device__ __forceinline__ void mma_f32(const double *As, const double *Bs, flt4 acc[2][2]) {
    const int lane = tid() & 63, w = tid() >> 6;
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32, i16 = lane & 15, k4 = lane >> 4;
    const double *pa0 = As + (wr + i16) * LDP + k4, *pa1 = pa0 + 16 * LDP;
    const double *pb0 = Bs + (wc + i16) * LDP + k4, *pb1 = pb0 + 16 * LDP;
    double na0 = pa0[0], na1 = pa1[0], nb0 = pb0[0], nb1 = pb1[0];
#pragma unroll
    for (int kk = 0; kk < TB; kk += 4) {
        const float a0 = (float)na0, a1 = (float)na1, b0 = (float)nb0, b1 = (float)nb1;
        if (kk + 4 < TB) {
            na0 = pa0[kk + 4];
            na1 = pa1[kk + 4];
            nb0 = pb0[kk + 4];
            nb1 = pb1[kk + 4];
        }
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1, acc[1][1], 0, 0, 0);
    }
}

// Three-slice BF16 form of the same product.  Each operand x is rounded to
// FP32 and split exactly into three BF16 numbers, x_f32 = h + m + l
// (h = bf16(x), m = bf16(x - h), l = x - h - m, which has at most 8
// significant bits and is exact); the six products whose weight reaches
// 2^-24 -- hh, hm, mh, hl, mm, lh -- are accumulated in FP32 on
// v_mfma_f32_16x16x32_bf16, smallest first.  The result carries FP32-class
// accuracy from BF16 matrix-core products.  Lane l supplies row l%16 and
// the eight K entries 8(l/16)..8(l/16)+7 of a 32-wide K step (the same K
// mapping for both operands, so the sum is the same whatever the hardware's
// K order); results as in the FP32 form (row 4(l/16) + v).
__device__ __forceinline__ void split3(const double *src, bf8 &h, bf8 &m, bf8 &l) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float f = (float)src[e];
        const __bf16 hh = (__bf16)f;
        const float r1 = f - (float)hh;
        const __bf16 mm = (__bf16)r1;
        h[e] = hh;
        m[e] = mm;
        l[e] = (__bf16)(r1 - (float)mm);
    }
}
__device__ __forceinline__ void mma_bf16x3(const double *As, const double *Bs, flt4 acc[2][2]) {
    const int lane = tid() & 63, w = tid() >> 6;
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32, i16 = lane & 15, k8 = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < TB; kk += 32) {
        bf8 ah[2], am[2], al[2], bh[2], bm[2], bl[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            split3(As + (wr + 16 * q + i16) * LDP + kk + 8 * k8, ah[q], am[q], al[q]);
            split3(Bs + (wc + 16 * q + i16) * LDP + kk + 8 * k8, bh[q], bm[q], bl[q]);
        }
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++) {
                flt4 c = acc[mi][ni];
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[mi], bh[ni], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am[mi], bm[ni], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[mi], bl[ni], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am[mi], bh[ni], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[mi], bm[ni], c, 0, 0, 0);
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[mi], bh[ni], c, 0, 0, 0);
            }
    }
}

// acc (-)= As Bs^T for one 64x64 tile in the arithmetic of MODE
// (BD_CHOL_FP64 / FP32 / BF16); Acc is dbl4 for FP64, flt4 otherwise.
template <int MODE, typename Acc>
__device__ __forceinline__ void tile_mma(const double *As, const double *Bs, Acc acc[2][2]) {
    if constexpr (MODE == 0) mma_f64(As, Bs, acc);
    else if constexpr (MODE == 1) mma_f32(As, Bs, acc);
    else mma_bf16x3(As, Bs, acc);
}
template <int MODE> struct AccOf { typedef flt4 T; };
template <> struct AccOf<0> { typedef dbl4 T; };

// C (LDS) += sign * acc, element mapping of mma_* (row of register v of
// lane l: l/16 + 4v for the FP64 MFMA, 4(l/16) + v for the FP32 one)
template <typename V>
__device__ __forceinline__ void acc_to_lds(double *C, V acc[2][2], double sign, bool overwrite) {
    const int lane = tid() & 63, w = tid() >> 6;
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32, i16 = lane & 15, k4 = lane >> 4;
    constexpr bool f64 = sizeof(acc[0][0][0]) == 8;
    for (int mi = 0; mi < 2; mi++)
        for (int ni = 0; ni < 2; ni++)
            for (int v = 0; v < 4; v++) {
                int r = wr + 16 * mi + (f64 ? k4 + 4 * v : 4 * k4 + v), c = wc + 16 * ni + i16;
                double x = sign * (double)acc[mi][ni][v];
                if (overwrite) C[r * LDP + c] = x;
                else C[r * LDP + c] += x;
            }
}

// A 16x16 output block of the FP64 matrix cores (mapping of mma_f64:
// register v of lane l is element (l/16 + 4v, l%16) of the block) into C.
__device__ __forceinline__ void blk_to_lds(double *C, int I, int J, dbl4 acc, double sign, bool overwrite) {
    const int lane = tid() & 63, i16 = lane & 15, k4 = lane >> 4;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        double *c = C + (16 * I + k4 + 4 * v) * LDP + 16 * J + i16;
        if (overwrite) *c = sign * acc[v];
        else *c += sign * acc[v];
    }
}

// Panel product P = A inv(L)^T with inv(L) lower triangular (zero above
// its diagonal 16x16 blocks): output block column J needs k < 16 (J + 1)
// only, and wavefront w takes the 16-row stripe w of P, so every
// wavefront issues the same 40 products.  Skipping the zero blocks adds
// nothing to any sum, so P is the full product bit for bit.
__device__ __forceinline__ void mma_panel(const double *As, const double *Li, dbl4 (&acc)[4]) {
    const int lane = tid() & 63, w = tid() >> 6, i16 = lane & 15, k4 = lane >> 4;
    const double *pa = As + (16 * w + i16) * LDP + k4, *pl = Li + i16 * LDP + k4;
    double na = pa[0], nb[4];
#pragma unroll
    for (int J = 0; J < 4; J++) nb[J] = pl[16 * J * LDP];
#pragma unroll
    for (int kk = 0; kk < TB; kk += 4) {
        const double a = na;
        double b[4];
#pragma unroll
        for (int J = 0; J < 4; J++) b[J] = nb[J];
        if (kk + 4 < TB) {  // next K step's operands beside this step's products
            na = pa[kk + 4];
#pragma unroll
            for (int J = 0; J < 4; J++)
                if (kk + 4 < 16 * (J + 1)) nb[J] = pl[16 * J * LDP + kk + 4];
        }
#pragma unroll
        for (int J = 0; J < 4; J++)
            if (kk < 16 * (J + 1)) acc[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[J], acc[J], 0, 0, 0);
    }
}
__device__ __forceinline__ void panel_to_lds(double *C, const dbl4 (&acc)[4]) {
    const int w = tid() >> 6;
#pragma unroll
    for (int J = 0; J < 4; J++) blk_to_lds(C, w, J, acc[J], 1.0, true);
}

// Diagonal tile update C -= P P^T on its ten lower 16x16 blocks only (the
// factor never reads above the diagonal), three or two per wavefront, their
// products interleaved (independent accumulators) with the next K step's
// operands read beside them; each block sums K in increasing order from
// zero and is then subtracted from C.
template <int N, int I0, int J0, int I1, int J1, int I2, int J2>
__device__ __forceinline__ void syrk_blocks(const double *P, double *C) {
    constexpr int I[3] = {I0, I1, I2}, J[3] = {J0, J1, J2};
    const int lane = tid() & 63, i16 = lane & 15, k4 = lane >> 4;
    const double *p = P + i16 * LDP + k4;
    dbl4 acc[N];
    double na[N], nb[N];
#pragma unroll
    for (int b = 0; b < N; b++) {
        acc[b] = dbl4{0.0, 0.0, 0.0, 0.0};
        na[b] = p[16 * I[b] * LDP];
        nb[b] = p[16 * J[b] * LDP];
    }
#pragma unroll
    for (int kk = 0; kk < TB; kk += 4) {
        double a[N], bv[N];
#pragma unroll
        for (int b = 0; b < N; b++) {
            a[b] = na[b];
            bv[b] = nb[b];
        }
        if (kk + 4 < TB)
#pragma unroll
            for (int b = 0; b < N; b++) {
                na[b] = p[16 * I[b] * LDP + kk + 4];
                nb[b] = p[16 * J[b] * LDP + kk + 4];
            }
#pragma unroll
        for (int b = 0; b < N; b++) acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[b], bv[b], acc[b], 0, 0, 0);
    }
#pragma unroll
    for (int b = 0; b < N; b++) blk_to_lds(C, I[b], J[b], acc[b], -1.0, false);
}
__device__ __forceinline__ void syrk_lower(const double *P, double *C) {
    const int w = __builtin_amdgcn_readfirstlane(tid() >> 6);
    // (I, J) blocks of wavefront w: {00 10 11} {20 21 22} {30 31} {32 33}
    if (w == 0) syrk_blocks<3, 0, 0, 1, 0, 1, 1>(P, C);
    else if (w == 1) syrk_blocks<3, 2, 0, 2, 1, 2, 2>(P, C);
    else if (w == 2) syrk_blocks<2, 3, 0, 3, 1, 0, 0>(P, C);
    else syrk_blocks<2, 3, 2, 3, 3, 0, 0>(P, C);
}

// ---------------------------------------------------------------------------
// Diagonal tile: factor L and inverse inv(L) by the four wavefronts of a
// workgroup, as one forward elimination of [C | I].
//
// What bounds it is the chain of 64 pivots, so the tile is cut into 16x16
// blocks, a block row's pivots stay in the registers of one wavefront, and
// everything off the chain goes to the other three.  Roles are fixed:
//
//   wavefront 0 holds the diagonal block of block row b, one column per lane
//     (the four groups of 16 lanes alike), its 16 rows in registers.  A
//     pivot's row times -1/|f| is added to the rows below with the factor of
//     row k taken from the lane of column k inside the FMA (DPP row
//     broadcast).  1/|f| is v_rcp_f64 with one third-order step; no square
//     root is on the chain: L and inv(L) are scaled by 1/sqrt(|f|) when they
//     are stored.  |f| where f < 0 (func.cpp:825-835), counted.
//   wavefront 1 eliminates the four other blocks of the block row side by
//     side, one per lane group: C_bj for j > b and the blocks of I for
//     j <= b; it follows wavefront 0 by a panel of four rows.
//   wavefronts 2 and 3 hold the blocks below (matrix-core result registers)
//     and subtract the panels' rank-4 products as they come; after the last
//     panel the blocks of row b + 1 go to wavefronts 0 and 1 through LDS.
//     In the last block row, where nothing is below, they store the rows
//     before it.
//
// Rows and columns of a 16x16 block are permuted alike, index i at position
// pos(i) = i/4 + 4 (i%4): register v of lane (g, c) of a matrix-core result
// is then row 4g + v, and a panel's rows serve as either operand.
// Panel buffers: W(b, j) and E(b, j), 16x16 each, element [64 p + 4 c + k] =
// row 4p + k, column position c.
//
// Measured alone, warm: 15.0k cycles (6.2 us) against 25.1k for one wavefront
// owning panels of 8 columns with rank-8 updates through LDS; of a block
// column's launch 16.0 -> 13.4 us.  What was in the way on gfx950: an FP64 FMA
// issues every 5 cycles from one wavefront, dependent or not, v_rcp_f64 and
// v_rsq_f64 take 16, a dependent 16x16x4 FP64 product 69 (and no FP64 FMA
// beside it), a store to LDS and the read back 135-165, so the pivots' updates
// stay in registers and the matrix cores do what is off the chain.
// ---------------------------------------------------------------------------
__device__ __forceinline__ constexpr int pos16(int i) { return i / 4 + 4 * (i % 4); }

// Rows in registers: the factor of row k times a scaled pivot row is one FMA
// whose first operand comes from the lane of column k of the same 16 lanes
// (v_fmac_f64_dpp row_newbcast).  The compiler does not form it, so these
// steps are inline code, in an order that keeps two instructions between a
// VALU write and the DPP read of the register (what the hardware needs, and
// the compiler does not add around inline code) with as few s_nop as possible:
// an s_nop 1 costs 8 cycles of the chain, an FMA 5, v_rcp_f64 16.
#define BD_POS_0 "0"
#define BD_POS_1 "4"
#define BD_POS_2 "8"
#define BD_POS_3 "12"
#define BD_POS_4 "1"
#define BD_POS_5 "5"
#define BD_POS_6 "9"
#define BD_POS_7 "13"
#define BD_POS_8 "2"
#define BD_POS_9 "6"
#define BD_POS_10 "10"
#define BD_POS_11 "14"
#define BD_POS_12 "3"
#define BD_POS_13 "7"
#define BD_POS_14 "11"
#define BD_POS_15 "15"
#define BD_DPP " row_mask:0xf bank_mask:0xf\n\t"
// row k += (column k of row j) m
#define BD_FM(k, j, m) "v_fmac_f64_dpp %[w" #k "], %[w" #j "], %[" #m "] row_newbcast:" BD_POS_##k BD_DPP
// 1/|f_j| (third-order step from its seed y = v_rcp_f64(|f|): y (1 + e + e^2),
// e = 1 - |f| y) and m = -w_j / |f_j|
#define BD_RM(j)                                                                          \
    "v_fma_f64 %[e], -|%[f]|, %[y], 1.0\n\tv_fma_f64 %[e], %[e], %[e], %[e]\n\t"          \
    "v_fma_f64 %[r], %[y], %[e], %[y]\n\tv_mul_f64 %[m], %[w" #j "], -%[r]\n\t"
// the next pivot (column j of row j) and its seed
#define BD_NEXT(j) "v_mov_b64_dpp %[f], %[w" #j "] row_newbcast:" BD_POS_##j BD_DPP
#define BD_SEED "v_rcp_f64 %[y], |%[f]|\n\t"
#define BD_PIVOT(J, TEXT)                                                                                           \
    {                                                                                                               \
    asm volatile(TEXT                                                                                               \
                 : [w0] "+v"(w[0]), [w1] "+v"(w[1]), [w2] "+v"(w[2]), [w3] "+v"(w[3]), [w4] "+v"(w[4]),             \
                   [w5] "+v"(w[5]), [w6] "+v"(w[6]), [w7] "+v"(w[7]), [w8] "+v"(w[8]), [w9] "+v"(w[9]),             \
                   [w10] "+v"(w[10]), [w11] "+v"(w[11]), [w12] "+v"(w[12]), [w13] "+v"(w[13]), [w14] "+v"(w[14]),   \
                   [w15] "+v"(w[15]), [r] "=&v"(r[J]), [m] "=&v"(m), [e] "=&v"(e), [y] "+v"(y), [f] "+v"(f)         \
                 : [n] "v"(n));                                                                                     \
    n = m;                                                                                                          \
    }
// Pivots J of wavefront 0: y, f the seed and the pivot; the products of the
// two last rows are left to the next pivot (n: its m) while there are enough.
template <int J>
__device__ __forceinline__ void pivot(double (&w)[16], double (&r)[16], double &y, double &f, double &n) {
    double m, e;
    if constexpr (J == 0)
        BD_PIVOT(0, "s_nop 1\n\t" BD_NEXT(0) BD_SEED "s_nop 0\n\t" BD_RM(0) "s_nop 1\n\t" BD_FM(1, 0, m) BD_FM(2, 0, m) BD_FM(3, 0, m)
                 BD_NEXT(1) BD_FM(4, 0, m) BD_SEED BD_FM(5, 0, m) BD_FM(6, 0, m) BD_FM(7, 0, m) BD_FM(8, 0, m)
                 BD_FM(9, 0, m) BD_FM(10, 0, m) BD_FM(11, 0, m) BD_FM(12, 0, m) BD_FM(13, 0, m));
    if constexpr (J == 1)
        BD_PIVOT(1, BD_RM(1) BD_FM(14, 0, n) BD_FM(15, 0, n) BD_FM(2, 1, m) BD_FM(3, 1, m) BD_FM(4, 1, m)
                 BD_NEXT(2) BD_FM(5, 1, m) BD_SEED BD_FM(6, 1, m) BD_FM(7, 1, m) BD_FM(8, 1, m) BD_FM(9, 1, m)
                 BD_FM(10, 1, m) BD_FM(11, 1, m) BD_FM(12, 1, m) BD_FM(13, 1, m));
    if constexpr (J == 2)
        BD_PIVOT(2, BD_RM(2) BD_FM(14, 1, n) BD_FM(15, 1, n) BD_FM(3, 2, m) BD_FM(4, 2, m) BD_FM(5, 2, m)
                 BD_NEXT(3) BD_FM(6, 2, m) BD_SEED BD_FM(7, 2, m) BD_FM(8, 2, m) BD_FM(9, 2, m) BD_FM(10, 2, m)
                 BD_FM(11, 2, m) BD_FM(12, 2, m) BD_FM(13, 2, m));
    if constexpr (J == 3)
        BD_PIVOT(3, BD_RM(3) BD_FM(14, 2, n) BD_FM(15, 2, n) BD_FM(4, 3, m) BD_FM(5, 3, m) BD_FM(6, 3, m)
                 BD_NEXT(4) BD_FM(7, 3, m) BD_SEED BD_FM(8, 3, m) BD_FM(9, 3, m) BD_FM(10, 3, m) BD_FM(11, 3, m)
                 BD_FM(12, 3, m) BD_FM(13, 3, m));
    if constexpr (J == 4)
        BD_PIVOT(4, BD_RM(4) BD_FM(14, 3, n) BD_FM(15, 3, n) BD_FM(5, 4, m) BD_FM(6, 4, m) BD_FM(7, 4, m)
                 BD_NEXT(5) BD_FM(8, 4, m) BD_SEED BD_FM(9, 4, m) BD_FM(10, 4, m) BD_FM(11, 4, m) BD_FM(12, 4, m)
                 BD_FM(13, 4, m));
    if constexpr (J == 5)
        BD_PIVOT(5, BD_RM(5) BD_FM(14, 4, n) BD_FM(15, 4, n) BD_FM(6, 5, m) BD_FM(7, 5, m) BD_FM(8, 5, m)
                 BD_NEXT(6) BD_FM(9, 5, m) BD_SEED BD_FM(10, 5, m) BD_FM(11, 5, m) BD_FM(12, 5, m) BD_FM(13, 5, m));
    if constexpr (J == 6)
        BD_PIVOT(6, BD_RM(6) BD_FM(14, 5, n) BD_FM(15, 5, n) BD_FM(7, 6, m) BD_FM(8, 6, m) BD_FM(9, 6, m)
                 BD_NEXT(7) BD_FM(10, 6, m) BD_SEED BD_FM(11, 6, m) BD_FM(12, 6, m) BD_FM(13, 6, m));
    if constexpr (J == 7)
        BD_PIVOT(7, BD_RM(7) BD_FM(14, 6, n) BD_FM(15, 6, n) BD_FM(8, 7, m) BD_FM(9, 7, m) BD_FM(10, 7, m)
                 BD_NEXT(8) BD_FM(11, 7, m) BD_SEED BD_FM(12, 7, m) BD_FM(13, 7, m));
    if constexpr (J == 8)
        BD_PIVOT(8, BD_RM(8) BD_FM(14, 7, n) BD_FM(15, 7, n) BD_FM(9, 8, m) BD_FM(10, 8, m) BD_FM(11, 8, m)
                 BD_NEXT(9) BD_FM(12, 8, m) BD_SEED BD_FM(13, 8, m));
    if constexpr (J == 9)
        BD_PIVOT(9, BD_RM(9) BD_FM(14, 8, n) BD_FM(15, 8, n) BD_FM(10, 9, m) BD_FM(11, 9, m) BD_FM(12, 9, m)
                 BD_NEXT(10) BD_FM(13, 9, m) BD_SEED BD_FM(14, 9, m) BD_FM(15, 9, m));
    if constexpr (J == 10)
        BD_PIVOT(10, BD_RM(10) "s_nop 1\n\t" BD_FM(11, 10, m) BD_FM(12, 10, m) BD_FM(13, 10, m) BD_NEXT(11)
                 BD_FM(14, 10, m) BD_SEED BD_FM(15, 10, m));
    if constexpr (J == 11)
        BD_PIVOT(11, BD_RM(11) "s_nop 1\n\t" BD_FM(12, 11, m) BD_FM(13, 11, m) BD_FM(14, 11, m) BD_NEXT(12)
                 BD_SEED BD_FM(15, 11, m));
    if constexpr (J == 12)
        BD_PIVOT(12, BD_RM(12) "s_nop 1\n\t" BD_FM(13, 12, m) BD_FM(14, 12, m) BD_FM(15, 12, m) BD_NEXT(13)
                 BD_SEED "s_nop 0\n\t");
    if constexpr (J == 13)
        BD_PIVOT(13, BD_RM(13) "s_nop 1\n\t" BD_FM(14, 13, m) BD_FM(15, 13, m) "s_nop 0\n\t" BD_NEXT(14)
                 BD_SEED "s_nop 0\n\t");
    if constexpr (J == 14)
        BD_PIVOT(14, BD_RM(14) "s_nop 1\n\t" BD_FM(15, 14, m) "s_nop 1\n\t" BD_NEXT(15) BD_SEED "s_nop 0\n\t");
    if constexpr (J == 15) BD_PIVOT(15, BD_RM(15));
}

// Rows of another block column: the panel's own rows x[K..K+3] by the pivot
// rows u before them, m_j = -x_j / |f_j| ...
template <int K>
__device__ __forceinline__ void follow_rows(double (&x)[16], const double (&u)[4], const double (&r)[4],
                                            double (&m)[4]) {
#define BD_FX(d, s, q, c) "v_fmac_f64_dpp %[" d "], %[" s "], %[" q "] row_newbcast:%[" c "]" BD_DPP
#define BD_MX(q, d, s) "v_mul_f64 %[" q "], %[" d "], -%[" s "]\n\ts_nop 1\n\t"
    asm volatile(BD_MX("m0", "x0", "r0") BD_FX("x1", "u0", "m0", "c1") BD_FX("x2", "u0", "m0", "c2")
                     BD_FX("x3", "u0", "m0", "c3") BD_MX("m1", "x1", "r1") BD_FX("x2", "u1", "m1", "c2")
                         BD_FX("x3", "u1", "m1", "c3") BD_MX("m2", "x2", "r2") BD_FX("x3", "u2", "m2", "c3")
                 : [x1] "+v"(x[K + 1]), [x2] "+v"(x[K + 2]), [x3] "+v"(x[K + 3]), [m0] "=&v"(m[0]), [m1] "=&v"(m[1]),
                   [m2] "=&v"(m[2])
                 : [x0] "v"(x[K]), [u0] "v"(u[0]), [u1] "v"(u[1]), [u2] "v"(u[2]), [r0] "v"(r[0]), [r1] "v"(r[1]),
                   [r2] "v"(r[2]), [c1] "n"(pos16(K + 1)), [c2] "n"(pos16(K + 2)), [c3] "n"(pos16(K + 3)));
    m[3] = x[K + 3] * -r[3];
}
// ... and four rows x[K..K+3] below by all four
template <int K>
__device__ __forceinline__ void below_rows(double (&x)[16], const double (&u)[4], const double (&m)[4]) {
    asm volatile("s_nop 1\n\t" BD_FX("x0", "u0", "m0", "c0") BD_FX("x1", "u0", "m0", "c1") BD_FX("x2", "u0", "m0", "c2")
                     BD_FX("x3", "u0", "m0", "c3") BD_FX("x0", "u1", "m1", "c0") BD_FX("x1", "u1", "m1", "c1")
                         BD_FX("x2", "u1", "m1", "c2") BD_FX("x3", "u1", "m1", "c3") BD_FX("x0", "u2", "m2", "c0")
                             BD_FX("x1", "u2", "m2", "c1") BD_FX("x2", "u2", "m2", "c2") BD_FX("x3", "u2", "m2", "c3")
                                 BD_FX("x0", "u3", "m3", "c0") BD_FX("x1", "u3", "m3", "c1")
                                     BD_FX("x2", "u3", "m3", "c2") BD_FX("x3", "u3", "m3", "c3")
                 : [x0] "+v"(x[K]), [x1] "+v"(x[K + 1]), [x2] "+v"(x[K + 2]), [x3] "+v"(x[K + 3])
                 : [u0] "v"(u[0]), [u1] "v"(u[1]), [u2] "v"(u[2]), [u3] "v"(u[3]), [m0] "v"(m[0]), [m1] "v"(m[1]),
                   [m2] "v"(m[2]), [m3] "v"(m[3]), [c0] "n"(pos16(K)), [c1] "n"(pos16(K + 1)), [c2] "n"(pos16(K + 2)),
                   [c3] "n"(pos16(K + 3)));
}

// LDS of the elimination; the tile itself may lie anywhere in it until it is
// in registers
struct DiagLds {
    double *base;
    // panel buffers W(b, j), j >= b, and E(b, j), j <= b, 256 each; the last
    // block row's E takes the place of the blocks handed to it
    __device__ __forceinline__ double *W(int b, int j) const { return base + (b * (9 - b) / 2 + j - b) * 256; }
    __device__ __forceinline__ double *E(int b, int j) const { return base + (10 + b * (b + 1) / 2 + j) * 256; }
    // blocks of the next block row, element [18 c + row]: lane group q of
    // wavefront 1, q = 3 wavefront 0
    __device__ __forceinline__ double *next(int q) const { return base + 4096 + 288 * q; }
    __device__ __forceinline__ double *R() const { return base + 5248; }  // 1/|f|, 64
    __device__ __forceinline__ double *S() const { return base + 5312; }  // 1/sqrt(|f|), 64
    // exponents the rows are scaled by (rescale_tile), 64; the tile does not reach here
    __device__ __forceinline__ int *K() const { return reinterpret_cast<int *>(base + 5376); }
};
static_assert(TB * LDP <= 5376, "tile and exponents");
constexpr int kNextPitch = 18;

// the operand register of a panel: lane (k, c) holds row k, column c
__device__ __forceinline__ double panel_op(const double *S, int p) {
    const int lane = tid() & 63;
    return S[64 * p + 4 * (lane & 15) + (lane >> 4)];
}
__device__ __forceinline__ dbl4 rank4(double a, double b, dbl4 acc) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
}
// rows 4P..4P+3 of w to a panel buffer (this lane's column)
template <int P>
__device__ __forceinline__ void put_rows(double *S, const double (&w)[16]) {
    double2 *d = reinterpret_cast<double2 *>(S + 64 * P + 4 * (tid() & 15));
    d[0] = make_double2(w[4 * P], w[4 * P + 1]);
    d[1] = make_double2(w[4 * P + 2], w[4 * P + 3]);
}
__device__ __forceinline__ void load_rows(double (&w)[16], const double *src) {
    const double2 *s = reinterpret_cast<const double2 *>(src);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const double2 v = s[i];
        w[2 * i] = v.x;
        w[2 * i + 1] = v.y;
    }
}

// Panel P of wavefront 0.  Its rows and 1/|f| are published with the next
// panel's first pivot between their LDS stores and the barrier.
template <int P>
__device__ __forceinline__ void pivot_panel(double (&w)[16], double (&r)[16], double &y, double &f, double &n,
                                            const DiagLds &l, int b) {
    if constexpr (P == 0) pivot<0>(w, r, y, f, n);
    pivot<4 * P + 1>(w, r, y, f, n);
    pivot<4 * P + 2>(w, r, y, f, n);
    pivot<4 * P + 3>(w, r, y, f, n);
    const int lane = tid() & 63;
    if (lane < 16) put_rows<P>(l.W(b, b), w);
    if (lane == 16) {
        double2 *d = reinterpret_cast<double2 *>(l.R() + 16 * b + 4 * P);
        d[0] = make_double2(r[4 * P], r[4 * P + 1]);
        d[1] = make_double2(r[4 * P + 2], r[4 * P + 3]);
    }
    if constexpr (P < 3) pivot<4 * P + 4>(w, r, y, f, n);
    __syncthreads();
}

// Panel P of wavefront 1: rows 4P..4P+3 of its four blocks by the pivot rows
// of wavefront 0, published, and the rows below them.
template <int P>
__device__ __forceinline__ void follow_panel(double (&x)[16], const DiagLds &l, double *Y, int b) {
    __syncthreads();
    const double2 *u2 = reinterpret_cast<const double2 *>(l.W(b, b) + 64 * P + 4 * (tid() & 15));
    const double2 *r2 = reinterpret_cast<const double2 *>(l.R() + 16 * b + 4 * P);
    const double2 ua = u2[0], ub = u2[1], ra = r2[0], rb = r2[1];
    const double u[4] = {ua.x, ua.y, ub.x, ub.y}, r[4] = {ra.x, ra.y, rb.x, rb.y};
    double m[4];
    follow_rows<4 * P>(x, u, r, m);
    put_rows<P>(Y, x);
    if constexpr (P < 3) below_rows<4 * P + 4>(x, u, m);
    if constexpr (P < 2) below_rows<4 * P + 8>(x, u, m);
    if constexpr (P < 1) below_rows<4 * P + 12>(x, u, m);
}

// L(b + q, b) for q < 4 - b, inv(L)(b, q - (4 - b)) after them: block q of
// the five that block row b leaves, scaled by 1/sqrt(|f|) and stored.
__device__ __forceinline__ void store_block(const DiagLds &l, int b, int q, double *A, int ld, int d0, double *Linv) {
    const int lane = tid() & 63, g = lane >> 4, c = lane & 15, ci = 4 * (c & 3) + (c >> 2);
    const bool isl = q < 4 - b;
    const int j = isl ? b + q : q - (4 - b);
    const double2 *s = reinterpret_cast<const double2 *>((isl ? l.W(b, j) : l.E(b, j)) + 64 * g + 4 * c);
    const double2 *i2 = reinterpret_cast<const double2 *>(l.S() + 16 * b + 4 * g);
    const double2 x0 = s[0], x1 = s[1], i0 = i2[0], i1 = i2[1];
    double x[4] = {x0.x * i0.x, x0.y * i0.y, x1.x * i1.x, x1.y * i1.y};
    if (isl) {
        if (j == b) {  // lower triangle of the diagonal block, L_jj = |f| / sqrt(|f|)
#pragma unroll
            for (int v = 0; v < 4; v++) x[v] = 4 * g + v > ci ? 0.0 : 4 * g + v == ci ? fabs(x[v]) : x[v];
        }
        double *row = A + (size_t)(d0 + 16 * j + ci) * ld + d0 + 16 * b + 4 * g;
        *reinterpret_cast<dbl2 *>(row) = dbl2{x[0], x[1]};
        *reinterpret_cast<dbl2 *>(row + 2) = dbl2{x[2], x[3]};
    } else {
#pragma unroll
        for (int v = 0; v < 4; v++) Linv[(16 * b + 4 * g + v) * TB + 16 * j + ci] = x[v];
    }
}

// Block (i, j) of the tile, i <= j, in matrix-core result registers
__device__ __forceinline__ dbl4 tile_block(const double *T, int i, int j) {
    const int lane = tid() & 63, g = lane >> 4, c = lane & 15, ci = 4 * (c & 3) + (c >> 2);
    dbl4 x;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int r = 16 * i + 4 * g + v, k = 16 * j + ci;
        x[v] = T[max(r, k) * LDP + min(r, k)];
    }
    return x;
}
// a finished block of block row b + 1 to its reader
__device__ __forceinline__ void put_next(const DiagLds &l, int q, dbl4 x) {
    const int lane = tid() & 63;
    double2 *d = reinterpret_cast<double2 *>(l.next(q) + kNextPitch * (lane & 15) + 4 * (lane >> 4));
    d[0] = make_double2(x[0], x[1]);
    d[1] = make_double2(x[2], x[3]);
}

// Panel p of block row B on the blocks that wavefront 2 + U holds, rows from
// I0 to I1: U = 0 has C11 C12 C22 C23 C33 E31, U = 1 has C13 E10 E20 E21 E30 E32.
template <int B, int U, int I0, int I1>
__device__ __forceinline__ void below_panel(dbl4 (&Z)[6], const DiagLds &l, int p) {
    const int g = (tid() & 63) >> 4;
    const double rn = -l.R()[16 * B + 4 * p + g];
    double a[4], e[3];
#pragma unroll
    for (int i = B + 1; i < 4; i++) a[i] = panel_op(l.W(B, i), p);
#pragma unroll
    for (int j = 0; j <= B; j++)
        if (U == 0 ? j == 1 : j != 1 || B == 1) e[j] = panel_op(l.E(B, j), p) * rn;
    auto in = [](int i) { return i > B && i >= I0 && i <= I1; };
    if constexpr (U == 0) {
        if (in(1)) Z[0] = rank4(a[1], a[1] * rn, Z[0]);
        if (in(1)) Z[1] = rank4(a[1], a[2] * rn, Z[1]);
        if (in(2)) Z[2] = rank4(a[2], a[2] * rn, Z[2]);
        if (in(2)) Z[3] = rank4(a[2], a[3] * rn, Z[3]);
        if (in(3)) Z[4] = rank4(a[3], a[3] * rn, Z[4]);
        if constexpr (B >= 1)
            if (in(3)) Z[5] = rank4(a[3], e[1], Z[5]);
    } else {
        if (in(1)) Z[0] = rank4(a[1], a[3] * rn, Z[0]);
        if (in(1)) Z[1] = rank4(a[1], e[0], Z[1]);
        if (in(2)) Z[2] = rank4(a[2], e[0], Z[2]);
        if constexpr (B >= 1)
            if (in(2)) Z[3] = rank4(a[2], e[1], Z[3]);
        if (in(3)) Z[4] = rank4(a[3], e[0], Z[4]);
        if constexpr (B >= 2)
            if (in(3)) Z[5] = rank4(a[3], e[2], Z[5]);
    }
}
template <int B, int U>
__device__ __forceinline__ void below_row(dbl4 (&Z)[6], const DiagLds &l) {
    __syncthreads();
#pragma unroll 1
    for (int p = 0; p < 3; p++) {
        __syncthreads();
        below_panel<B, U, B + 1, 3>(Z, l, p);
    }
    __syncthreads();
    below_panel<B, U, B + 1, B + 1>(Z, l, 3);
    if constexpr (U == 0) {
        put_next(l, 3, Z[B == 0 ? 0 : B == 1 ? 2 : 4]);
        put_next(l, B == 2 ? 1 : 0, Z[B == 0 ? 1 : B == 1 ? 3 : 5]);
    } else {
        put_next(l, B == 2 ? 0 : 1, Z[B == 0 ? 0 : B == 1 ? 2 : 4]);
        put_next(l, 2, Z[B == 0 ? 1 : B == 1 ? 3 : 5]);
    }
    __syncthreads();
    if constexpr (B < 2) below_panel<B, U, B + 2, 3>(Z, l, 3);
}

// The elimination divides by |f| and forms inv(L) from rows over |f|, which
// overflow where a pivot is below 2^-1024, though its root and 1/sqrt(|f|) do
// not.  A tile with diagonal entries outside [2^-960, 2^960] is therefore
// factored as S C S with S = 2^-k, k half the exponent of a row's diagonal
// entry, and L = inv(S) L', inv(L) = inv(L') S on its way out: the scaling is
// exact.  Inside the bounds the pivots keep clear of 2^-1022 (cancellation
// takes 53 bits at most) and nothing is scaled.  The test is one LDS read and
// one comparison ahead of the tile's own reads (33 block columns 500.2 -> 501.3
// us a factor, 49 847.0 -> 848.8); beside them, a copy of the
// scaling to each wavefront's role, it cost three times that.
__device__ __forceinline__ bool tile_out_of_range(const double *T) {
    const double d = fabs(T[(tid() & 63) * (LDP + 1)]);
    return __ballot(!(d >= 0x1p-960 && d <= 0x1p+960)) != 0;
}
// By all four wavefronts, before they read T.
__device__ __forceinline__ void rescale_tile(const DiagLds &l, double *T) {
    __syncthreads();
    if (tid() < TB) {
        const double d = fabs(T[tid() * (LDP + 1)]);
        // zero, infinity and NaN have the exponent 0
        l.K()[tid()] = d >= 0x1p-960 && d <= 0x1p+960 ? 0 : __builtin_amdgcn_frexp_exp(d) / 2;
    }
    __syncthreads();
#pragma unroll 1
    for (int e = tid(); e < TB * TB; e += NTHR) {
        const int r = e / TB, c = e % TB;
        if (c <= r) T[r * LDP + c] = __builtin_ldexp(T[r * LDP + c], -l.K()[r] - l.K()[c]);
    }
    __syncthreads();
}
__device__ __forceinline__ void unscale_tile(const DiagLds &l, double *A, int ld, int d0, double *Linv) {
    __syncthreads();
#pragma unroll 1
    for (int e = tid(); e < TB * TB; e += NTHR) {
        const int r = e / TB, c = e % TB;
        if (c > r) continue;
        double *a = A + (size_t)(d0 + r) * ld + d0 + c, *i = Linv + r * TB + c;
        *a = __builtin_ldexp(*a, l.K()[r]);
        *i = __builtin_ldexp(*i, -l.K()[c]);
    }
}

// A pivot of exactly 0, which rows that depend on each other leave where the
// column-wise form had a rounding error (a reciprocal times its pivot is mostly
// exactly 1, a root squared is not), makes all that follows NaN.  The
// elimination therefore keeps a copy of its tile (save, row-major, the lower
// triangle), and a tile with a pivot that has no reciprocal root is factored
// again from it column by column: L's column and inv(L)'s row of a zero pivot
// are 0, so that L L^T is D for dependent rows.
__device__ __forceinline__ void save_block(double *save, int i, int j, dbl4 x) {
    const int lane = tid() & 63, g = lane >> 4, c = lane & 15, ci = 4 * (c & 3) + (c >> 2);
    dbl2 *d = reinterpret_cast<dbl2 *>(save + (16 * j + ci) * TB + 16 * i + 4 * g);
    d[0] = dbl2{x[0], x[1]};
    d[1] = dbl2{x[2], x[3]};
}
__device__ __forceinline__ bool pivot_without_root(const DiagLds &l) {
    return __ballot(!(l.S()[tid() & 63] < HUGE_VAL)) != 0;
}
__device__ __forceinline__ void refactor_tile(const DiagLds &l, const double *save, double *A, int ld, int d0, double *Linv,
                                              int *neg) {
    double *T = l.base, *I = l.base + TB * LDP;  // inv(L) above T's diagonal, transposed, and its diagonal in I
    static_assert(TB * LDP + TB <= 5376, "below the exponents");
    __syncthreads();
#pragma unroll 1
    for (int e = tid(); e < TB * TB; e += NTHR)
        if (e % TB <= e / TB) T[(e / TB) * LDP + e % TB] = save[e];
    __syncthreads();
    int n = 0;
#pragma unroll 1
    for (int j = 0; j < TB; j++) {
        const double f = T[j * (LDP + 1)], a = fabs(f), inv = a == 0.0 ? 0.0 : rsqrt_f64(a);
        n += f < 0;
        __syncthreads();
        if (tid() < TB && tid() >= j) T[tid() * LDP + j] = tid() == j ? a * inv : T[tid() * LDP + j] * inv;
        if (tid() == j) I[j] = inv;
        __syncthreads();
#pragma unroll 1
        for (int e = tid(); e < TB * TB; e += NTHR) {
            const int r = e / TB, c = e % TB;
            if (c > j && c <= r) T[r * LDP + c] -= T[r * LDP + j] * T[c * LDP + j];
        }
        __syncthreads();
    }
    if (tid() == 0 && n) atomicAdd(neg, n);
#pragma unroll 1
    for (int e = tid(); e < TB * TB; e += NTHR) {
        const int r = e / TB, c = e % TB;
        if (c <= r) A[(size_t)(d0 + r) * ld + d0 + c] = T[r * LDP + c];
    }
    if (tid() < TB) {
        const int c = tid();
#pragma unroll 1
        for (int i = 0; i < TB; i++) {
            double x = i == c ? I[c] : 0.0;
            if (i > c) {
                x = -T[i * LDP + c] * I[c];
                for (int k = c + 1; k < i; k++) x -= T[i * LDP + k] * T[c * LDP + k];
                x *= I[i];
                T[c * LDP + i] = x;
            }
            Linv[i * TB + c] = x;
        }
    }
}

// Called by all four wavefronts.  lds: kDiagLds doubles; T, LDS that may
// overlap its first 5376 doubles, holds the tile (pitch LDP) at (d0, d0), of
// which the lower triangle is read.  L goes
// to A (lower triangle), inv(L), row-major 64x64 with zeros above its
// diagonal, to Linv; the tile behind it there, the next column's, is scratch.
__device__ __forceinline__ void diag_factor_inv(double *lds, double *T, double *A, int ld, int d0, double *Linv,
                                                int *neg) {
    const int lane = tid() & 63, wv = __builtin_amdgcn_readfirstlane(tid() >> 6);
    const int g = lane >> 4, c = lane & 15, ci = 4 * (c & 3) + (c >> 2);
    const DiagLds l = {lds};
    const bool scaled = tile_out_of_range(T);
    if (__builtin_expect(scaled, false)) rescale_tile(l, T);
    double *save = Linv + TB * TB;
    int nneg = 0;  // of wavefront 0
    if (wv == 0) {
        double w[16], r[16];
#pragma unroll
        for (int k = 0; k < 16; k++) w[k] = T[max(k, ci) * LDP + min(k, ci)];
        __syncthreads();
#pragma unroll 1
        for (int b = 0; b < 4; b++) {
            if (b) load_rows(w, l.next(3) + kNextPitch * c);
            double y = 0.0, f = 0.0, n = 0.0;
            pivot_panel<0>(w, r, y, f, n, l, b);
            pivot_panel<1>(w, r, y, f, n, l, b);
            pivot_panel<2>(w, r, y, f, n, l, b);
            pivot_panel<3>(w, r, y, f, n, l, b);
            // the scale factors of the block row and its negative pivots
            const double fd = l.W(b, b)[64 * (c >> 2) + 4 * pos16(c) + (c & 3)];
            if (lane < 16) l.S()[16 * b + c] = rsqrt_f64(fabs(fd));
            nneg += __popcll(__ballot(lane < 16 && fd < 0));
            __syncthreads();
            if (b < 3) __syncthreads();
        }
    } else if (wv == 1) {
        double x[16];
#pragma unroll
        for (int k = 0; k < 16; k++) x[k] = g < 3 ? T[(16 * (g + 1) + ci) * LDP + k] : k == ci ? 1.0 : 0.0;
        __syncthreads();
        if (g < 3)
#pragma unroll
            for (int k = 0; k < 16; k += 2)
                *reinterpret_cast<dbl2 *>(save + (16 * (g + 1) + ci) * TB + k) = dbl2{x[k], x[k + 1]};
#pragma unroll 1
        for (int b = 0; b < 4; b++) {
            if (b) {
                load_rows(x, l.next(min(g, 2)) + kNextPitch * c);
#pragma unroll
                for (int k = 0; k < 16; k++) x[k] = g < 3 ? x[k] : k == ci ? 1.0 : 0.0;
            }
            double *Y = g < 3 - b ? l.W(b, b + 1 + g) : l.E(b, b + g - 3);
            follow_panel<0>(x, l, Y, b);
            follow_panel<1>(x, l, Y, b);
            follow_panel<2>(x, l, Y, b);
            follow_panel<3>(x, l, Y, b);
            __syncthreads();
            if (b < 3) __syncthreads();
        }
    } else {
        const dbl4 z = {0.0, 0.0, 0.0, 0.0};
        // the blocks of inv(L) above its diagonal
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const int k = 3 * (wv - 2) + t, bi = k < 3 ? 0 : k < 5 ? 1 : 2, bj = k < 3 ? k + 1 : k < 5 ? k - 1 : 3;
            dbl2 *o = reinterpret_cast<dbl2 *>(Linv + (16 * bi + (lane >> 2)) * TB + 16 * bj + 4 * (lane & 3));
            o[0] = o[1] = dbl2{0.0, 0.0};
        }
        if (wv == 2) {
            dbl4 Z[6] = {tile_block(T, 1, 1), tile_block(T, 1, 2), tile_block(T, 2, 2), tile_block(T, 2, 3),
                         tile_block(T, 3, 3), z};
            __syncthreads();
            save_block(save, 1, 1, Z[0]);
            save_block(save, 1, 2, Z[1]);
            save_block(save, 2, 2, Z[2]);
            save_block(save, 2, 3, Z[3]);
            save_block(save, 3, 3, Z[4]);
            below_row<0, 0>(Z, l);
            below_row<1, 0>(Z, l);
            below_row<2, 0>(Z, l);
        } else {
            dbl4 Z[6] = {tile_block(T, 1, 3), z, z, z, z, z};
            const dbl4 first = tile_block(T, 0, 0);
            __syncthreads();
            save_block(save, 0, 0, first);
            save_block(save, 1, 3, Z[0]);
            below_row<0, 1>(Z, l);
            below_row<1, 1>(Z, l);
            below_row<2, 1>(Z, l);
        }
        // block rows 0 to 2 are complete: 15 blocks, beside the last pivots
#pragma unroll 1
        for (int p = 0; p < 5; p++) {
            __syncthreads();
            if (p < 4)
                for (int t = 4 * p + wv - 2; t < min(4 * p + 4, 15); t += 2) store_block(l, t / 5, t % 5, A, ld, d0, Linv);
        }
    }
    const bool broken = pivot_without_root(l);
    store_block(l, 3, wv, A, ld, d0, Linv);
    if (wv == 0) store_block(l, 3, 4, A, ld, d0, Linv);
    if (__builtin_expect(broken, false)) refactor_tile(l, save, A, ld, d0, Linv, neg);
    else if (wv == 0 && lane == 0 && nneg) atomicAdd(neg, nneg);
    if (__builtin_expect(scaled, false)) unscale_tile(l, A, ld, d0, Linv);
}

// a tile between global memory, registers and LDS (pitch LDP), 16-byte
// accesses, every load of a thread in flight at once
constexpr int PERT = TB * TB / 2 / NTHR;
__device__ __forceinline__ void tile_to_regs(const double *src, int ld, dbl2 (&v)[PERT]) {
#pragma unroll
    for (int i = 0; i < PERT; i++) {
        const int e = tid() + i * NTHR, r = e / (TB / 2), c = 2 * (e % (TB / 2));
        v[i] = *reinterpret_cast<const dbl2 *>(src + (size_t)r * ld + c);
    }
}
__device__ __forceinline__ void regs_to_lds(const dbl2 (&v)[PERT], double *S) {
#pragma unroll
    for (int i = 0; i < PERT; i++) {
        const int e = tid() + i * NTHR, r = e / (TB / 2), c = 2 * (e % (TB / 2));
        S[r * LDP + c] = v[i].x;
        S[r * LDP + c + 1] = v[i].y;
    }
}
// C -= Pi Pj^T for an off-diagonal tile C in global memory, from registers
// (element mapping of mma_*)
template <int MODE>
__device__ __forceinline__ void tile_update(const double *Pi, const double *Pj, double *C, int ld) {
    typename AccOf<MODE>::T acc[2][2];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) acc[a][b] = {};
    tile_mma<MODE>(Pi, Pj, acc);
    const int lane = tid() & 63, w = tid() >> 6;
    const int wr = (w >> 1) * 32, wc = (w & 1) * 32, i16 = lane & 15, k4 = lane >> 4;
    constexpr bool f64 = MODE == 0;
    double cv[2][2][4];
#pragma unroll
    for (int mi = 0; mi < 2; mi++)
#pragma unroll
        for (int ni = 0; ni < 2; ni++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = wr + 16 * mi + (f64 ? k4 + 4 * v : 4 * k4 + v), c = wc + 16 * ni + i16;
                cv[mi][ni][v] = C[(size_t)r * ld + c];
            }
#pragma unroll
    for (int mi = 0; mi < 2; mi++)
#pragma unroll
        for (int ni = 0; ni < 2; ni++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = wr + 16 * mi + (f64 ? k4 + 4 * v : 4 * k4 + v), c = wc + 16 * ni + i16;
                C[(size_t)r * ld + c] = cv[mi][ni][v] + -1.0 * (double)acc[mi][ni][v];
            }
}
// C -= P P^T for a diagonal tile in LDS
template <int MODE>
__device__ __forceinline__ void diag_tile_update(const double *P, double *C) {
    if (MODE == 0) {
        syrk_lower(P, C);
    } else {
        typename AccOf<MODE>::T acc[2][2];
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++) acc[a][b] = {};
        tile_mma<MODE>(P, P, acc);
        acc_to_lds(C, acc, -1.0, false);
    }
}
// A tile from LDS by wavefronts 2 and 3, which have two of syrk_lower's
// blocks where 0 and 1 have three
__device__ __forceinline__ void store_tile_half(double *dst, int ld, const double *S) {
    if (tid() < NTHR / 2) return;
#pragma unroll
    for (int i = 0; i < 2 * PERT; i++) {
        const int e = tid() - NTHR / 2 + i * (NTHR / 2), r = e / (TB / 2), c = 2 * (e % (TB / 2));
        *reinterpret_cast<dbl2 *>(dst + (size_t)r * ld + c) = dbl2{S[r * LDP + c], S[r * LDP + c + 1]};
    }
}

// A panel tile from LDS, negated, in the operand order of k_panel_rows: 16
// bytes of lane l of unit u = 2 b + h of wavefront w are row 16 w +
// row_pi(l % 16), K = 16 b + 4 (l / 16) + 2 h and the next
__device__ __forceinline__ int row_pi(int i16) { return 4 * (i16 & 3) + (i16 >> 2); }
__device__ __forceinline__ void store_operand(double *dst, const double *S) {
    const int lane = tid() & 63, w = tid() >> 6;
    const double *src = S + (16 * w + row_pi(lane & 15)) * LDP + 4 * (lane >> 4);
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int c = 16 * (u >> 1) + 2 * (u & 1);
        *reinterpret_cast<dbl2 *>(dst + (w * 8 + u) * 128 + 2 * lane) = dbl2{-src[c], -src[c + 1]};
    }
}

// Trailing tiles of block column kb restricted to the first jcols trailing
// block columns, row-major: rows ii = 0..M-1, columns jj <= min(ii, jcols-1)
// (jcols = M: the whole trailing triangle, in tri_index order).
__device__ __forceinline__ void trap_index(int idx, int jcols, int &i, int &j) {
    const int tri = jcols * (jcols + 1) / 2;
    if (idx < tri) {
        tri_index(idx, i, j);
        return;
    }
    idx -= tri;
    i = jcols + idx / jcols;
    j = idx % jcols;
}

// One block column kb of the factorisation in one launch, one workgroup per
// trailing lower tile (ib, jb), kb < jb <= ib, jb - kb <= jcols:
//   1. the panel tiles L_ib,kb = A_ib,kb inv(L_kb,kb)^T and L_jb,kb on the
//      FP64 matrix cores, from the inverse the previous launch left in
//      Linv; the workgroup of the first column (jb = kb + 1) stores L_ib,kb,
//      so every panel tile is written exactly once, into the upper block
//      (kb, ib), because other workgroups of this launch still read
//      A_ib,kb; the tiles stay there (k_noise, k_trail and the host copy
//      of the factor read them from there);
//   2. A_ib,jb -= L_ib,kb L_jb,kb^T on the matrix cores (FP64, or FP32 /
//      three-slice BF16 with FP32 accumulation for MODE 1 / 2);
//   3. the workgroup of tile (kb+1, kb+1) factors and inverts it, which the
//      next launch needs.
// The panel products are repeated by the workgroups of a block row, in
// exchange for one launch (and one kernel boundary) per block column.
// jcols < M restricts the update to the columns of a super-panel.
constexpr int kStepLds = 2 * TB * LDP;
template <int MODE>
__device__ __forceinline__ void step_tile(double *S, double *A, int ld, int kb, int jcols, int lb, double *Linv, int *neg,
                                          double *Lp) {
    // two tiles of LDS: first inv(L_kb,kb) and the row's panel block, then the
    // column's panel block in place of the row's, then the two panel tiles;
    // the target tile stays in registers
    double *S0 = S, *S1 = S + TB * LDP;
    int ii, jj;
    trap_index(lb, jcols, ii, jj);
    const int ib = kb + 1 + ii, jb = kb + 1 + jj;
    const bool diag = ib == jb;
    // ahead of force kernels on its CU (100 nucleosomes 864 us a step, 875 without)
    if (lb == 0) __builtin_amdgcn_s_setprio(3);
    dbl2 vi[PERT], vj[PERT];
    {
        dbl2 vw[PERT];
        tile_to_regs(Linv + (size_t)kb * TB * TB, TB, vw);
        tile_to_regs(A + (size_t)ib * TB * ld + kb * TB, ld, vi);
        // the column's panel block, or the diagonal target tile
        tile_to_regs(diag ? A + (size_t)ib * TB * ld + jb * TB : A + (size_t)jb * TB * ld + kb * TB, ld, vj);
        regs_to_lds(vw, S0);
        regs_to_lds(vi, S1);
    }
    __syncthreads();
    dbl4 pi[4];
    for (int J = 0; J < 4; J++) pi[J] = dbl4{0.0, 0.0, 0.0, 0.0};
    mma_panel(S1, S0, pi);
    __syncthreads();
    if (diag) {
        panel_to_lds(S1, pi);
        regs_to_lds(vj, S0);
        __syncthreads();
        diag_tile_update<MODE>(S1, S0);
        if (jj == 0) store_tile_half(A + (size_t)kb * TB * ld + ib * TB, ld, S1);
        if (Lp && jcols == 1) store_operand(Lp, S1);
        __syncthreads();
        if (ii == 0)
            diag_factor_inv(S, S0, A, ld, ib * TB, Linv + (size_t)ib * TB * TB, neg);
        else
            store_tile(A, ld, ib * TB, jb * TB, S0, true);
        return;
    }
    regs_to_lds(vj, S1);
    __syncthreads();
    {
        dbl4 pj[4];
        for (int J = 0; J < 4; J++) pj[J] = dbl4{0.0, 0.0, 0.0, 0.0};
        mma_panel(S1, S0, pj);
        __syncthreads();
        panel_to_lds(S0, pi);
        panel_to_lds(S1, pj);
    }
    __syncthreads();
    if (jj == 0) {
        store_tile(A, ld, kb * TB, ib * TB, S0, false);
        if (Lp) {
            store_operand(Lp + ii * TB * TB, S0);
            if (ii == 1) store_operand(Lp, S1);  // L_kb+1,kb, which workgroup 0 has no time for
        }
    }
    tile_update<MODE>(S0, S1, A + (size_t)ib * TB * ld + jb * TB, ld);
}
template <int MODE>
__global__ void __launch_bounds__(256, 2) k_step(double *A, int ld, int kb, int jcols, double *Linv, int *neg) {
    __shared__ double S[kStepLds];  // two workgroups per CU
    // workgroups go round-robin over the eight XCDs (b % 8); XCD x takes a
    // contiguous run of tiles, so the tiles of a block row, which read the
    // same panel tile, share an L2 (workgroup 0, the diagonal tile, stays 0)
    int lb = blockIdx.x;
    const int G8 = gridDim.x / 8;
    if (lb < 8 * G8) lb = (lb % 8) * G8 + lb / 8;
    step_tile<MODE>(S, A, ld, kb, jcols, lb, Linv, neg, nullptr);
}

// The same with one workgroup of two teams per CU, for 257 to 485 tiles on 256
// CUs (from 486, split_tiles, k_panel and k_update are the shorter way): tile
// 0 has workgroup 0, and with it a CU, to itself, so that its factor, a chain
// of FP64 vector arithmetic, does not stand still beside another workgroup's
// matrix products; the others go in contiguous runs to the XCDs (workgroups go
// round-robin over the eight), each XCD's as many as it has teams for.  The
// teams share their barriers, which a team that has left no longer takes part
// in.  17.0 us against 18.4 (253 tiles in k_step: 15.5); what is left are two
// tiles' products on a CU, 10.2 us.  k_update in this form, its teams going
// from tile to tile, took 18 to 28 us against 15 to 20.
constexpr int kStep2Tiles(int grid) { return 2 * (grid - 1) + 1; }
template <int MODE>
__global__ void __launch_bounds__(512, 2) k_step2(double *A, int ld, int kb, int jcols, int n, double *Linv, int *neg) {
    __shared__ double S[2 * kStepLds];
    const int team = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int per = gridDim.x / 8, x = blockIdx.x & 7, all = 2 * ((int)gridDim.x - 1);
    const int before = x ? 2 * (per - 1) + 2 * per * (x - 1) : 0, own = x ? 2 * per : 2 * (per - 1);
    const int t0 = (n - 1) * before / all, t1 = (n - 1) * (before + own) / all;
    int lb = t0 + 2 * ((blockIdx.x >> 3) - (x == 0)) + team, end = t1;
    if (blockIdx.x == 0) {
        lb = team - 1;
        end = 0;
    }
    if (lb >= end) return;
    step_tile<MODE>(S + team * kStepLds, A, ld, kb, jcols, lb + 1, Linv, neg, nullptr);
}

// The same block column in two launches, for wide trailing matrices (many
// tiles per launch): k_panel forms every panel tile L_ib,kb once and parks
// it in the upper block (kb, ib); k_update then updates each trailing tile
// from two parked panel tiles, and its workgroup of tile (kb+1, kb+1)
// factors and inverts it.  This trades one launch for the panel products
// that k_step repeats in every workgroup of a block row (and for a smaller
// LDS footprint: two panel workgroups fit on a CU).
__global__ void __launch_bounds__(256) k_panel(double *A, int ld, int kb, const double *Linv) {
    __shared__ double W[TB * LDP], As[TB * LDP];
    const int ib = kb + 1 + blockIdx.x;
    {
        dbl2 vw[PERT], va[PERT];
        tile_to_regs(Linv + (size_t)kb * TB * TB, TB, vw);
        tile_to_regs(A + (size_t)ib * TB * ld + kb * TB, ld, va);
        regs_to_lds(vw, W);
        regs_to_lds(va, As);
    }
    __syncthreads();
    dbl4 pi[4];
    for (int J = 0; J < 4; J++) pi[J] = dbl4{0.0, 0.0, 0.0, 0.0};
    mma_panel(As, W, pi);
    __syncthreads();
    panel_to_lds(As, pi);
    __syncthreads();
    store_tile(A, ld, kb * TB, ib * TB, As, false);
}

template <int MODE>
__global__ void __launch_bounds__(256, 2) k_update(double *A, int ld, int kb, int jcols, double *Linv, int *neg) {
    __shared__ double S[2 * TB * LDP];
    double *S0 = S, *S1 = S + TB * LDP;
    int lb = blockIdx.x;  // XCD-contiguous runs of tiles, as in k_step
    const int G8 = gridDim.x / 8;
    if (lb < 8 * G8) lb = (lb % 8) * G8 + lb / 8;
    int ii, jj;
    trap_index(lb, jcols, ii, jj);
    const int ib = kb + 1 + ii, jb = kb + 1 + jj;
    const bool diag = ib == jb;
    if (lb == 0) __builtin_amdgcn_s_setprio(3);
    {
        // the parked panel tiles L_ib,kb and L_jb,kb
        // (the target tile in place of the second on the diagonal)
        dbl2 vi[PERT], vj[PERT];
        tile_to_regs(A + (size_t)kb * TB * ld + ib * TB, ld, vi);
        tile_to_regs(diag ? A + (size_t)ib * TB * ld + jb * TB : A + (size_t)kb * TB * ld + jb * TB, ld, vj);
        regs_to_lds(vi, S1);
        regs_to_lds(vj, S0);
    }
    __syncthreads();
    if (!diag) {
        tile_update<MODE>(S1, S0, A + (size_t)ib * TB * ld + jb * TB, ld);
        return;
    }
    diag_tile_update<MODE>(S1, S0);
    __syncthreads();
    if (ii == 0)
        diag_factor_inv(S, S0, A, ld, ib * TB, Linv + (size_t)ib * TB * TB, neg);
    else
        store_tile(A, ld, ib * TB, jb * TB, S0, true);
}

// Trailing update of a super-panel: block columns k0 .. k0+nb-1 are
// factored and their panel tiles parked; every lower tile (ib, jb) of the
// trailing matrix (rows and columns from j0 = k0 + nb) takes
//   A_ib,jb -= sum_k L_ib,k L_jb,k^T   (K = 64 nb)
// with the sum held in registers across the nb panel tiles and the tile
// read and written once.  The next panel tiles are loaded into registers
// while the current ones are multiplied (the target tile during the last).
// Workgroups are grouped in 8x8 blocks of tiles, 64 consecutive workgroups
// per block, so the panel tiles of a block's 8 rows and 8 columns are
// shared through the L2; workgroups past the triangle or the edge exit.
// Workgroup 0, dispatched first, goes on to factor and invert its tile
// (j0, j0), which the next panel begins with, beside the others' updates (a
// launch of its own took 21 us per super-panel: 0.39 of 12.1 ms a step at 500
// nucleosomes).  k_trail_pk and k_trail_bf do the same.
template <int MODE>
__global__ void __launch_bounds__(256, 2) k_trail(double *A, int ld, int k0, int nb, int j0, int nt, double *Linv,
                                                  int *neg) {
    __shared__ double S[2 * TB * LDP];
    double *As = S, *Bs = S + TB * LDP;
    int SI, SJ;
    tri_index(blockIdx.x >> 6, SI, SJ);
    const int ib = j0 + 8 * SI + ((blockIdx.x >> 3) & 7), jb = j0 + 8 * SJ + (blockIdx.x & 7);
    if (ib >= nt || jb > ib) return;
    const bool diag = ib == jb;
    dbl2 va[PERT], vb[PERT];
    typename AccOf<MODE>::T acc[2][2];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) acc[a][b] = {};
    // L_ib,k is parked at block (k, ib)
    tile_to_regs(A + (size_t)k0 * TB * ld + ib * TB, ld, va);
    if (!diag) tile_to_regs(A + (size_t)k0 * TB * ld + jb * TB, ld, vb);
    for (int t = 0; t < nb; t++) {
        regs_to_lds(va, As);
        if (!diag) regs_to_lds(vb, Bs);
        __syncthreads();
        if (t + 1 < nb) {
            const size_t row = (size_t)(k0 + t + 1) * TB * ld;
            tile_to_regs(A + row + ib * TB, ld, va);
            if (!diag) tile_to_regs(A + row + jb * TB, ld, vb);
        } else {
            tile_to_regs(A + (size_t)ib * TB * ld + jb * TB, ld, va);
        }
        tile_mma<MODE>(As, diag ? As : Bs, acc);
        __syncthreads();
    }
    regs_to_lds(va, As);
    __syncthreads();
    acc_to_lds(As, acc, -1.0, false);
    __syncthreads();
    if (blockIdx.x == 0) diag_factor_inv(S, As, A, ld, j0 * TB, Linv + (size_t)j0 * TB * TB, neg);
    else store_tile(A, ld, ib * TB, jb * TB, As, diag);
}

constexpr int kPanel = 8;  // super-panel width of chol_panels

// Block lin of a triangle of S x S blocks (tiles, or 2x2 tiles) in the order
// GxG group by GxG group, a group row by row.
template <int G>
__device__ __forceinline__ void group_index(int lin, int S, int &IB, int &JB) {
    int r, c;
    tri_index(lin, r, c);  // r: the block row in row-by-row order, in the same group row
    const int GI = r / G, h = min(G, S - G * GI), o = lin - G * GI * (G * GI + 1) / 2;
    if (o < G * h * GI) {
        const int GJ = o / (G * h), q = o - G * h * GJ;
        IB = G * GI + q / G;
        JB = G * GJ + q % G;
    } else {
        tri_index(o - G * h * GI, r, c);
        IB = G * GI + r;
        JB = G * GI + c;
    }
    IB = __builtin_amdgcn_readfirstlane(IB);
    JB = __builtin_amdgcn_readfirstlane(JB);
}
// Blocks lin0 .. lin0 + n - 1 over the eight XCDs, which workgroups take
// round-robin (b % 8): XCD x takes the x-th eighth of them.  -1 past the end.
__device__ __forceinline__ int xcd_index(int b, int lin0, int n) {
    const int per = (n + 7) / 8, l = (b & 7) * per + (b >> 3);
    return l < n ? lin0 + l : -1;
}
inline int xcd_grid(int n) { return (n + 7) / 8 * 8; }
// Three-slice BF16 trailing update with the panel tiles split once.  Split
// on the fly (k_trail<2>), every workgroup converts every operand fragment it
// multiplies, so each panel tile is split by all the workgroups of its tile
// row and column and the update is bound by that VALU work.  Here k_split3
// writes the three BF16 slices of every parked panel tile of the super-panel
// once, in the operand order of v_mfma_f32_16x16x32_bf16: fragment (rb, ks)
// of a slice (16 rows from 16 rb, 32 K from 32 ks) is 64 lanes x 16 bytes,
// lane l holding row 16 rb + l % 16 and K entries 32 ks + 8 (l / 16) .. +7.
// Slice s of the tile of row block i and panel column t sits at
// sp[((i - j0) nb + t) 3 + s].
constexpr size_t kSplitTile = (size_t)TB * TB;
__device__ __forceinline__ size_t frag_off(int rb, int ks, int lane) { return (size_t)((rb * 2 + ks) * 64 + lane) * 8; }

// one workgroup per (row block, panel column) tile; wavefront w writes the
// fragments of row block w
__global__ void __launch_bounds__(256) k_split3(const double *A, int ld, int k0, int nb, int j0, __bf16 *sp) {
    const int i = j0 + blockIdx.x / nb, t = blockIdx.x % nb;
    const double *src = A + (size_t)(k0 + t) * TB * ld + (size_t)i * TB;
    __bf16 *dst = sp + (size_t)blockIdx.x * 3 * kSplitTile;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        const int r = 16 * w + (lane & 15), c = 32 * ks + 8 * (lane >> 4);
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; q += 2) {
            const dbl2 x = *reinterpret_cast<const dbl2 *>(src + (size_t)r * ld + c + q);
            v[q] = x.x;
            v[q + 1] = x.y;
        }
        bf8 h, m, l;
        split3(v, h, m, l);
        const size_t o = frag_off(w, ks, lane);
        *reinterpret_cast<bf8 *>(dst + o) = h;
        *reinterpret_cast<bf8 *>(dst + kSplitTile + o) = m;
        *reinterpret_cast<bf8 *>(dst + 2 * kSplitTile + o) = l;
    }
}

// k_trail_bf: a workgroup takes a 2x2 block of trailing tiles (128x128) and
// wavefront (wr, wc) the whole tile (ib0 + wr, jb0 + wc).  A stage is one K
// step (32) of a panel column: the block's two row tiles' and two column
// tiles' fragments, three slices each, 48 kilobyte slots (op, tile, s, rb),
// copied straight from global memory into LDS (global_load_lds_dwordx4:
// lane l's 16 bytes land at the slot + 16 l, so a fragment lies in LDS as in
// global memory and every wavefront read of it is conflict-free).  The
// copies are what bounds this kernel, so the tile is as large as the
// registers allow (a wavefront reads 24 fragments per stage for 96
// products), and three workgroups share a CU (3 x 48 KB of LDS) to keep
// three stages in flight.  The six products of a 16x16 block, their order
// and the split are those of k_trail<2>: the same factor bit for bit.
typedef __attribute__((address_space(3))) void lds_void;
__device__ __forceinline__ int bf_slot(int op, int tile, int s, int rb) { return ((op * 2 + tile) * 3 + s) * 4 + rb; }
__device__ __forceinline__ const __bf16 *bf_src(const __bf16 *sp, int row, int nb, int t, int s, int rb, int ks,
                                                int lane) {
    return sp + ((size_t)(row * nb + t) * 3 + s) * kSplitTile + frag_off(rb, ks, lane);
}
// Stage st (panel column st / 2, K step st % 2) of tile rows ra, ra + 1 and
// (unless DIAG, where the column tiles are the row tiles) rbw, rbw + 1,
// relative to j0; rows at or past nrow (the odd edge) are not copied.
// Wavefront w copies one tile's 12 fragments (DIAG: half of one tile's).
template <bool DIAG>
__device__ __forceinline__ void bf_issue(const __bf16 *sp, int ra, int rbw, int nb, int nrow, int st, __bf16 *S, int w,
                                         int lane) {
    const int t = st >> 1, ks = st & 1;
    if (DIAG) {
        const int tile = w >> 1, half = w & 1;
        if (ra + tile >= nrow) return;
#pragma unroll
        for (int j = 0; j < 6; j++) {
            const int f = 6 * half + j, sl = f >> 2, rb = f & 3;
            __builtin_amdgcn_global_load_lds(bf_src(sp, ra + tile, nb, t, sl, rb, ks, lane),
                                             (lds_void *)(S + (size_t)bf_slot(0, tile, sl, rb) * 512), 16, 0, 0);
        }
    } else {
        const int op = w >> 1, tile = w & 1, row = (op ? rbw : ra) + tile;
        if (row >= nrow) return;
#pragma unroll
        for (int f = 0; f < 12; f++) {
            const int sl = f >> 2, rb = f & 3;
            __builtin_amdgcn_global_load_lds(bf_src(sp, row, nb, t, sl, rb, ks, lane),
                                             (lds_void *)(S + (size_t)bf_slot(op, tile, sl, rb) * 512), 16, 0, 0);
        }
    }
}
// the six products of column block ni for the four row blocks, each
// block's in the fixed order (smallest first)
__device__ __forceinline__ void bf_mma_col(const bf8 (&fa)[3][4], const bf8 (&fb)[3], flt4 (&acc)[4][4], int ni) {
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int p = 0; p < 6; p++)
#pragma unroll
        for (int mi = 0; mi < 4; mi++)
            acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[PA[p]][mi], fb[PB[p]], acc[mi][ni], 0, 0, 0);
}
__device__ __forceinline__ void bf_read_col(const __bf16 *S, int op, int tile, int q, int lane, bf8 (&fb)[3]) {
#pragma unroll
    for (int sl = 0; sl < 3; sl++)
        fb[sl] = *reinterpret_cast<const bf8 *>(S + (size_t)bf_slot(op, tile, sl, q) * 512 + lane * 8);
}
// Per stage: every wavefront waits for its own copies (vmcnt(0); the LDS
// writes of a copy are done when it retires) and a barrier makes the stage
// whole; the row fragments (12) and two column blocks' (3 each) are read,
// the products of column block 0 run while block 2's fragments are read into
// block 0's registers (1 and 3 likewise); after lgkmcnt(0) a second barrier
// frees the stage, the copy of the next stage is issued, and the products
// of column blocks 2 and 3 run beside it.  The compiler does not order the
// copies against these LDS reads, hence the explicit waits.  Wavefronts
// with no tile (above the diagonal, past the edge) still copy and meet
// every barrier.
template <bool DIAG>
__device__ __forceinline__ void bf_body(const __bf16 *sp, int ra, int rbw, int nb, int nrow, __bf16 *S, int w, int lane,
                                        bool active, flt4 (&acc)[4][4]) {
    constexpr int BOP = DIAG ? 0 : 1;
    const int wr = w >> 1, wc = w & 1;
    bf8 fa[3][4], fb0[3], fb1[3];
    bf_issue<DIAG>(sp, ra, rbw, nb, nrow, 0, S, w, lane);
    for (int st = 0; st < 2 * nb; st++) {
        __builtin_amdgcn_s_waitcnt(0xF70);   // vmcnt(0)
        __builtin_amdgcn_s_barrier();
        if (active) {
#pragma unroll
            for (int sl = 0; sl < 3; sl++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    fa[sl][q] = *reinterpret_cast<const bf8 *>(S + (size_t)bf_slot(0, wr, sl, q) * 512 + lane * 8);
            bf_read_col(S, BOP, wc, 0, lane, fb0);
            bf_read_col(S, BOP, wc, 1, lane, fb1);
            bf_mma_col(fa, fb0, acc, 0);
            bf_read_col(S, BOP, wc, 2, lane, fb0);
            bf_mma_col(fa, fb1, acc, 1);
            bf_read_col(S, BOP, wc, 3, lane, fb1);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        if (st + 1 < 2 * nb) bf_issue<DIAG>(sp, ra, rbw, nb, nrow, st + 1, S, w, lane);
        if (active) {
            bf_mma_col(fa, fb0, acc, 2);
            bf_mma_col(fa, fb1, acc, 3);
        }
    }
}
// The blocks of an XCD follow each other in 4x4 groups (group_index), so a
// group's 8 row and 8 column panel tiles are read into one L2 (8x8 groups, 16
// and 16 tiles: 17.6 ms of trailing updates at 1000 nucleosomes against 16.8).
constexpr int kBfLds = 48 * 512;  // of BF16
__device__ __forceinline__ void trail_bf_block(__bf16 *S, double *A, int ld, const __bf16 *sp, int nb, int j0, int nt, int IB,
                                               int JB, double *Linv, int *neg) {
    const bool first = IB == 0;  // the block of the next panel's first tile
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wr = w >> 1, wc = w & 1;
    const int nrow = nt - j0, ra = 2 * IB, rbw = 2 * JB;  // tile rows relative to j0
    const int ib = j0 + ra + wr, jb = j0 + rbw + wc;
    const bool active = ib < nt && jb <= ib;
    flt4 acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = flt4{0.f, 0.f, 0.f, 0.f};
    if (IB == JB) bf_body<true>(sp, ra, rbw, nb, nrow, S, w, lane, active, acc);
    else bf_body<false>(sp, ra, rbw, nb, nrow, S, w, lane, active, acc);
    if (!active && !first) return;
    const int i16 = lane & 15, k4 = lane >> 4;
    // C -= acc in place, a row of 16x16 blocks at a time: loads, then stores
    // (a diagonal tile keeps its upper triangle; the first tile goes to LDS,
    // for its factor)
    double *T = reinterpret_cast<double *>(S);
    const bool keep = first && w == 0;
    if (active)
#pragma unroll
    for (int mi = 0; mi < 4; mi++) {
        double cv[4][4];
#pragma unroll
        for (int ni = 0; ni < 4; ni++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = 16 * mi + 4 * k4 + v, c = 16 * ni + i16;
                cv[ni][v] = A[(size_t)(ib * TB + r) * ld + jb * TB + c];
            }
#pragma unroll
        for (int ni = 0; ni < 4; ni++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = 16 * mi + 4 * k4 + v, c = 16 * ni + i16;
                if (ib == jb && c > r) continue;
                const double x = cv[ni][v] + -1.0 * (double)acc[mi][ni][v];
                if (keep) T[r * LDP + c] = x;
                else A[(size_t)(ib * TB + r) * ld + jb * TB + c] = x;
            }
    }
    if (first) {
        __syncthreads();
        diag_factor_inv(T, T, A, ld, j0 * TB, Linv + (size_t)j0 * TB * TB, neg);
    }
}
__global__ void __launch_bounds__(256, 3) k_trail_bf(double *A, int ld, const __bf16 *sp, int nb, int j0, int nt, int n,
                                                     double *Linv, int *neg) {
    __shared__ __attribute__((aligned(16))) __bf16 S[kBfLds];
    static_assert(sizeof(S) >= kDiagLds * sizeof(double) && sizeof(S) >= TB * LDP * sizeof(double), "LDS of the factor");
    const int lin = xcd_index(blockIdx.x, 0, n);
    if (lin < 0) return;
    int IB, JB;
    group_index<4>(lin, (nt - j0 + 1) / 2, IB, JB);
    trail_bf_block(S, A, ld, sp, nb, j0, nt, IB, JB, Linv, neg);
}

// FP64 / FP32 trailing update of a super-panel from panel tiles packed once.
// k_pack64 copies each parked panel tile of the super-panel into the operand
// order of v_mfma_f64_16x16x4f64 (v_mfma_f32_16x16x4f32 has the same lane
// layout): unit (u, rb) of a tile is 64 lanes x 16 bytes, lane l holding
// row 16 rb + l % 16 at K = Q u + 4 q + l / 16, q = 0, 1 in doubles (Q = 8)
// or q = 0 .. 3 rounded to floats (Q = 16).  A row block's units follow each
// other through the whole K of the super-panel: unit (u, rb) of the tile of
// row block i and panel column t is the one numbered
// 4 (((i - j0) nb + t) TB / Q + u) + rb.
template <int MODE> struct PackOf { typedef dbl2 T; static constexpr int kUnits = 8; };
template <> struct PackOf<1> { typedef flt4 T; static constexpr int kUnits = 4; };

// one workgroup per (row block, panel column) tile; wavefront w writes the
// units of rows 16 w
template <int MODE>
__global__ void __launch_bounds__(256) k_pack64(const double *A, int ld, int k0, int nb, int j0, void *pk) {
    typedef typename PackOf<MODE>::T T;
    constexpr int U = PackOf<MODE>::kUnits, Q = 16 / U;
    const int i = j0 + blockIdx.x / nb, t = blockIdx.x % nb;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double *src = A + (size_t)((k0 + t) * TB + 16 * w + (lane & 15)) * ld + (size_t)i * TB + (lane >> 4);
    T *dst = static_cast<T *>(pk) + ((size_t)blockIdx.x * U * 4 + w) * 64 + lane;
#pragma unroll
    for (int u = 0; u < U; u++) {
        T v;
#pragma unroll
        for (int q = 0; q < Q; q++) v[q] = src[4 * (Q * u + q)];
        dst[256 * u] = v;
    }
}

// k_trail_pk: a workgroup takes one trailing tile and each wavefront a 32x32
// quarter of it, reading its operands (two row and two column units a step)
// from global memory straight into registers, the next step's while the
// matrix cores work on the current one's.  No LDS, no barrier, and a
// quarter that lies above the diagonal costs nothing.  What bounds it is the
// matrix cores, 85% busy in FP64 and 71% in FP32, where reading and writing the
// tile takes its share: over the launches of a factor 63 TF at 1000 nucleosomes
// (61 to 67 a launch) and 61 at 500, in FP32 110 at 1000, of 78 and 157 that a
// loop of nothing but products reaches.  A CU reads 32 bytes of operands a
// cycle, half of what its L1 gives.  A launch alone, repeated: the form before
// (128x128 blocks staged through LDS by direct copies, two barriers per 16 of K)
// in FP64 60.0 / 54.0 / 48.2 TF at 320 / 156 / 80 trailing block rows, this one
// 64 / 66.9 / 67.5; 64x64 per wavefront in this form 64.4 / 62.0 / 52.8 (as few
// as 3 such blocks per CU) and in FP32 66 against 97 TF.  With the operand
// addresses in vector registers 65 and 100 TF where now 67 and 112.  Three workgroups share a CU (the LDS of the first tile's
// factor); a fourth changed nothing, nor did the tile's own loads before the
// loop (FP32 slower by a fifth: the registers).
//
// Workgroups go round-robin over the eight XCDs (b % 8).  Each XCD takes an
// eighth of the triangle's tiles in the order of group_index, so the tiles in
// flight on it share their 8 row and 8 column panels in its L2 and all eight
// end together (whole groups dealt to XCDs in turn left up to 28% of the chip
// idle at 120 block rows).
//
// Every accumulator takes the MFMAs of k_trail<MODE> in the same order (panel
// column, then K step), so the update is the same bit for bit.
// one step's units from the uniform addresses A and B, which the empty asm
// keeps in scalar registers: an FP64 matrix product and a vector ALU
// instruction do not overlap, so the loop holds no address arithmetic in
// vector registers
template <typename T>
__device__ __forceinline__ void pk_read(const T *A, const T *B, unsigned lane, T (&a)[2], T (&b)[2]) {
    typedef const T __attribute__((address_space(1))) *Global;
    Global pa = (Global)A, pb = (Global)B;
    asm volatile("" : "+s"(pa), "+s"(pb));
#pragma unroll
    for (int q = 0; q < 2; q++) {
        a[q] = pa[lane + 64u * q];
        b[q] = pb[lane + 64u * q];
    }
}
__device__ __forceinline__ dbl4 pk_mfma(double a, double b, dbl4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ flt4 pk_mfma(float a, float b, flt4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <int Q, typename T, typename V>
__device__ __forceinline__ void pk_products(const T (&a)[2], const T (&b)[2], V (&acc)[2][2]) {
    // between the reads before and after it, so that these are in flight
    // beside the products
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++) acc[mi][ni] = pk_mfma(a[mi][q], b[ni][q], acc[mi][ni]);
    __builtin_amdgcn_sched_barrier(0);
}
// D: steps in the operand ring (divides 4 nb)
template <int MODE, int D>
__device__ __forceinline__ void trail_pk_tile(double *S, double *A, int ld, const void *pk, int nb, int j0, int IB, int JB,
                                              double *Linv, int *neg) {
    typedef typename PackOf<MODE>::T T;
    typedef typename AccOf<MODE>::T V;
    constexpr int U = PackOf<MODE>::kUnits;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = w >> 1, wc = w & 1;
    const bool diag = IB == JB && wr == wc, active = IB > JB || wr >= wc;
    const bool first = IB == 0;  // the first tile goes to LDS, for its factor
    if (active) {
        const T *a = static_cast<const T *>(pk) + ((size_t)IB * nb * U * 4 + 2 * wr) * 64;
        const T *b = static_cast<const T *>(pk) + ((size_t)JB * nb * U * 4 + 2 * wc) * 64;
        V acc[2][2];
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++) acc[mi][ni] = V{};
        T ra[D][2], rb[D][2];
#pragma unroll
        for (int d = 0; d < D - 1; d++) pk_read(a + 256 * d, b + 256 * d, lane, ra[d], rb[d]);
        for (int u = U * nb; u > 0; u -= D) {
            pk_read(a + 256 * (D - 1), b + 256 * (D - 1), lane, ra[D - 1], rb[D - 1]);
            const int st = u > D ? 256 * D : 0;  // the last pass reads its own units again
            a += st;
            b += st;
#pragma unroll
            for (int d = 0; d < D; d++) {
                pk_products<16 / U>(ra[d], rb[d], acc);
                if (d + 1 < D) pk_read(a + 256 * d, b + 256 * d, lane, ra[d], rb[d]);
            }
        }
        // C -= acc in place (row of register v: l/16 + 4v for the FP64 MFMA,
        // 4(l/16) + v for the FP32 one), loads before stores
        const int i16 = lane & 15, k4 = lane >> 4;
        double *C = A + (size_t)((j0 + IB) * TB + 32 * wr) * ld + (j0 + JB) * TB + 32 * wc;
        double *T0 = S + 32 * wr * LDP + 32 * wc;
        double cv[2][2][4];
        auto row = [&](int mi, int v) { return 16 * mi + (MODE == 0 ? k4 + 4 * v : 4 * k4 + v); };
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++)
#pragma unroll
                for (int v = 0; v < 4; v++) cv[mi][ni][v] = C[(size_t)row(mi, v) * ld + 16 * ni + i16];
#pragma unroll
        for (int mi = 0; mi < 2; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int r = row(mi, v), c = 16 * ni + i16;
                    if (diag && c > r) continue;
                    const double x = cv[mi][ni][v] + -1.0 * (double)acc[mi][ni][v];
                    if (first) T0[r * LDP + c] = x;
                    else C[(size_t)r * ld + c] = x;
                }
    }
    if (first) {
        __syncthreads();
        diag_factor_inv(S, S, A, ld, j0 * TB, Linv + (size_t)j0 * TB * TB, neg);
    }
}
template <int MODE>
__global__ void __launch_bounds__(256, 3) k_trail_pk(double *A, int ld, const void *pk, int nb, int j0, int nt, int lin0,
                                                     int n, double *Linv, int *neg) {
    __shared__ __attribute__((aligned(16))) double S[kDiagLds];
    static_assert(kDiagLds >= TB * LDP, "the first tile");
    const int lin = xcd_index(blockIdx.x, lin0, n);
    if (lin < 0) return;
    int IB, JB;
    group_index<kPanel>(lin, nt - j0, IB, JB);
    trail_pk_tile<MODE, 2>(S, A, ld, pk, nb, j0, IB, JB, Linv, neg);
}

// One block column inside the diagonal block of a super-panel (step_tile, the
// jcols (jcols + 1) / 2 workgroups before the others) beside n tiles of the
// trailing update that is under way.  The column's launch is a chain of
// latencies (13.0 us, of which 6.2 the next diagonal tile), at most 28
// workgroups of it, so the other CUs take a tile of K = 512 each: 21.5 us with
// 228 of them, where a launch of their own would cost 14.5 us more than the
// chain alone.  jcols = 0: tiles only, the first of them the next panel's
// first, which workgroup 0 goes on to factor.  The FP64 vector arithmetic of a
// diagonal tile stands still beside another workgroup's matrix products, so a
// workgroup asks for more than half of the LDS and has its CU to itself.
constexpr int kOwnCu = 10368;  // doubles, more than half of a CU's LDS
template <int MODE>
__global__ void __launch_bounds__(256, 1) k_block_step(double *A, int ld, int kb, int jcols, const void *pk, int nb, int j0,
                                                       int nt, int lin0, int n, double *Linv, int *neg, double *Lp) {
    __shared__ __attribute__((aligned(16))) double S[kOwnCu];
    static_assert(kOwnCu >= kStepLds && kOwnCu >= kDiagLds, "LDS");
    const int G = jcols * (jcols + 1) / 2;
    if ((int)blockIdx.x < G) {
        step_tile<0>(S, A, ld, kb, jcols, blockIdx.x, Linv, neg, Lp);
        return;
    }
    const int lin = xcd_index(blockIdx.x - G, lin0, n);
    if (lin < 0) return;
    int IB, JB;
    group_index<kPanel>(lin, nt - j0, IB, JB);
    trail_pk_tile<MODE, 4>(S, A, ld, pk, nb, j0, IB, JB, Linv, neg);
}

// The rows below the diagonal block of a super-panel of kPanel columns, once
// the block is factored: X_k = (B_k - sum_{j<k} X_j L_kj^T) inv(L_kk)^T, 16
// rows per workgroup and 16 of a column's 64 rows of L per wavefront, the
// rows' eight column blocks in the accumulators.  The tiles go to their parked
// places and, where the trailing update takes them packed (pk), there too.
// Each wavefront multiplies L (as left operands, negated and in operand order
// from k_block_step) with the transposed rows: a product's result layout is
// then the next one's right operand, and the two exchanges per column, of the
// updated and of the solved block, are two LDS writes and eight reads of a
// wavefront, run between the updates that do not need them.  27 us up to 256
// workgroups (64 block rows; 16 of them the products at the matrix cores'
// rate), 50 up to 512, where column by column beside the block's own steps the
// rows took 3 to 11 us per column, with the trailing update's tiles left
// outside; 80 up to 768, 105 up to 1024, 135 at 1280 (matrix cores 47% busy over
// a factor at 1000 nucleosomes).  Operands in other layouts, with a transposition through LDS on
// either side of each column: 31 and 56 us.
constexpr int kPanelTiles = kPanel * (kPanel + 1) / 2;
// Order of the products of k_panel_rows: the solve of column 0, then for each
// column k its updates of columns k + 1, k + 2, k + 3, the solve of column
// k + 1, and the rest of the updates.
struct PanelTile { int k, t; };  // inv(L_kk) where t == k, else L_tk
constexpr PanelTile panel_tile(int e) {
    if (e == 0) return {0, 0};
    int n = 1;
    for (int k = 0; k + 1 < kPanel; k++) {
        const int before = kPanel - 1 - k < 3 ? kPanel - 1 - k : 3;  // updates before the solve
        const int count = kPanel - k;
        if (e < n + count) {
            const int j = e - n;
            if (j < before) return {k, k + 1 + j};
            if (j == before) return {k + 1, k + 1};
            return {k, k + j};
        }
        n += count;
    }
    return {-1, -2};
}
template <typename F, int... I>
__device__ __forceinline__ void static_steps(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
// Operands of the 16 matrix products of a 64x64 tile, by wavefront w its rows
// 16 w ..: row 16 w + pi(l % 16), K = 16 b + 4 (l / 16) + s, s = 0 .. 3, in
// o[2 b + s / 2]; off: this lane's first element, step: between its pairs
template <int S1, int S2>
__device__ __forceinline__ void read_operand(const double *base, unsigned off, dbl2 (&o)[8]) {
    typedef const double __attribute__((address_space(1))) *Global;
    typedef const dbl2 __attribute__((address_space(1))) *Global2;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        Global p = (Global)base + 2 * S2 * h;
        asm volatile("" : "+s"(p));  // in scalar registers, as in pk_read
#pragma unroll
        for (int u = 0; u < 4; u++) o[4 * h + u] = *(Global2)(p + off + S1 * (u & 1) + S2 * (u >> 1));
    }
    __builtin_amdgcn_sched_barrier(0);
}
template <int MODE>
__global__ void __launch_bounds__(256, 2) k_panel_rows(double *A, int ld, int k0, const double *Linv, const double *Lp,
                                                       void *pk) {
    __shared__ __attribute__((aligned(16))) dbl2 Bs[512], Xs[512];  // [2 b + h][lane]
    const int ri = blockIdx.x / 4, rb = blockIdx.x & 3, i = k0 + kPanel + ri;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
    // column blocks, transposed: lane l holds row l % 16, columns
    // 64 t + 16 w + 4 (l / 16) + v, in the MFMA's result layout with its rows
    // taken by row_pi, which is also the layout of a product's right operand
    dbl4 acc[kPanel];
    dbl2 op[3][8], x[8], y[8];
    const unsigned inv_off = (16 * w + row_pi(i16)) * TB + 4 * k4, tile_off = w * 1024 + 2 * lane;
    auto fetch = [&](auto E) {
        constexpr PanelTile q = panel_tile(E);
        if constexpr (q.t == q.k) read_operand<2, 16>(Linv + (size_t)(k0 + q.k) * TB * TB, inv_off, op[E % 3]);
        else read_operand<128, 256>(Lp + (q.k * kPanel + q.t) * TB * TB, tile_off, op[E % 3]);
    };
    auto products = [&](const dbl2 (&a)[8], const dbl2 (&b)[8], dbl4 c) {
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int q = 0; q < 2; q++) c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][q], b[u][q], c, 0, 0, 0);
        return c;
    };
    auto put = [&](dbl2 *S, const dbl4 &v) {
        S[128 * w + lane] = dbl2{v[0], v[1]};
        S[128 * w + 64 + lane] = dbl2{v[2], v[3]};
    };
    auto get = [&](const dbl2 *S, dbl2 (&v)[8]) {
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = S[64 * u + lane];
    };
    double *row = A + (size_t)(i * TB + 16 * rb + i16) * ld + k0 * TB + 16 * w + 4 * k4;
    double *park = A + (size_t)(k0 * TB + 16 * rb + i16) * ld + i * TB + 16 * w + 4 * k4;
    // column t's block of this wavefront, solved: to the others and to memory
    auto store = [&](int t, const dbl4 &v) {
        put(Xs, v);
        dbl2 *d = reinterpret_cast<dbl2 *>(park + (size_t)t * TB * ld);
        d[0] = dbl2{v[0], v[1]};
        d[1] = dbl2{v[2], v[3]};
    };
    // the packed (split) form of column t, from all four blocks
    auto pack = [&](int t) {
        if (!pk) return;
        const double *X = reinterpret_cast<const double *>(Xs);
        // column c of row i16
        auto at = [&](int c) { return X[((c >> 4) * 128 + ((c >> 1) & 1) * 64 + i16 + 16 * ((c >> 2) & 3)) * 2 + (c & 1)]; };
        typedef typename PackOf<MODE>::T T;
        constexpr int U = PackOf<MODE>::kUnits, Q = 16 / U;
        T *dst = static_cast<T *>(pk) + ((size_t)(ri * kPanel + t) * U * 4 + rb) * 64 + lane;
#pragma unroll
        for (int uu = 0; uu < U / 4; uu++) {
            const int u = U / 4 * w + uu;
            T v;
#pragma unroll
            for (int q = 0; q < Q; q++) v[q] = at(4 * (Q * u + q) + k4);
            dst[256 * u] = v;
        }
    };
#pragma unroll
    for (int t = 0; t < kPanel; t++) {
        const dbl2 *src = reinterpret_cast<const dbl2 *>(row + t * TB);
        const dbl2 lo = src[0], hi = src[1];
        acc[t] = dbl4{lo.x, lo.y, hi.x, hi.y};
    }
    fetch(std::integral_constant<int, 0>{});
    fetch(std::integral_constant<int, 1>{});
    put(Bs, acc[0]);
    __syncthreads();
    get(Bs, y);
    auto step = [&](auto E) {
        constexpr PanelTile q = panel_tile(E);
        if constexpr (E + 2 < kPanelTiles) fetch(std::integral_constant<int, E + 2>{});
        if constexpr (q.t == q.k) {
            const dbl4 v = products(op[E % 3], y, dbl4{0.0, 0.0, 0.0, 0.0});
            store(q.k, v);
        } else {
            // summed apart, as column by column: chained onto the block the 512
            // products leave a residual L L^T - D 1.5 times as large
            acc[q.t] += products(op[E % 3], x, dbl4{0.0, 0.0, 0.0, 0.0});
            asm volatile("" : "+v"(acc[q.t]));  // added here, not where it is next read
        }
        __builtin_amdgcn_sched_barrier(0);
        // the exchanges: column k + 1 once updated by k, read one update
        // later; the solved column after the last update by the one before
        constexpr PanelTile n = panel_tile(E + 1);
        if constexpr (q.t == q.k + 1) put(Bs, acc[q.t]);
        if constexpr (q.t != q.k && (q.t == q.k + 2 || n.t == q.k + 1) && q.t < q.k + 3) {
            __syncthreads();
            get(Bs, y);
        }
        if constexpr (n.t == n.k + 1 || E == kPanelTiles - 1) {
            constexpr int k = E == kPanelTiles - 1 ? kPanel - 1 : n.k;
            __syncthreads();
            get(Xs, x);
            pack(k);
        }
    };
    static_steps(step, std::make_integer_sequence<int, kPanelTiles>{});
}

// Factor and inverse of the diagonal tile (d, d) by one workgroup (the
// first tile of a large or a caller's matrix); clear != 0 also restarts the negative-pivot count.
__global__ void __launch_bounds__(256) k_diag(double *A, int ld, int d, double *Linv, int *neg, int clear) {
    __shared__ double T[kDiagLds];
    if (clear && threadIdx.x == 0) *neg = 0;
    load_tile(A, ld, d * TB, d * TB, T);
    __syncthreads();
    diag_factor_inv(T, T, A, ld, d * TB, Linv + (size_t)d * TB * TB, neg);
}

// rd = s2dt * L * p (rd_cal, func_cuda.cu:634-647): one wavefront per row,
// lane k % 64 over the row; rows outside the hydrodynamic set use their
// self-mobility: s2dt * sqrt(a1 / rad) * p.  With du = D inv(L~)^T p (the
// FP64 refinement of a reduced-precision factor) the HI rows take
// s2dt (L~ p + du) / 2 instead.  L is read where the factor
// leaves it: the diagonal tile of the row in place, the off-diagonal tile
// (ib, t) parked in the upper block (t, ib) (a row of the parked tile is
// contiguous, so every read is one 512-byte segment).
__global__ void __launch_bounds__(256) k_noise(const double *A, int ld, int m, int nD3, const double *p,
                                               const double *du, const double *rad_all, double s2dt, double a1,
                                               double *rd) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= nD3) return;
    if (row >= m) {
        if (lane == 0) rd[row] = s2dt * sqrt(a1 / rad_all[row / 3]) * p[row];
        return;
    }
    const int ib = row / TB, r = row % TB;
    const double *a = A + (size_t)r * ld + ib * TB + lane;  // parked tile (t, ib): a + t*TB*ld
    const double *q = p + lane;
    double v = 0.0;
    int t = 0;
    // eight tiles' loads in flight at a time, summed in tile order
    for (; t + 8 <= ib; t += 8) {
        double x[8], y[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            x[u] = a[(size_t)(t + u) * TB * ld];
            y[u] = q[(t + u) * TB];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) v += x[u] * y[u];
    }
    for (; t < ib; t++) v += a[(size_t)t * TB * ld] * q[t * TB];
    if (lane <= r) v += A[(size_t)row * ld + ib * TB + lane] * p[ib * TB + lane];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) rd[row] = s2dt * (du ? 0.5 * (v + du[row]) : v);
}

// ---------------------------------------------------------------------------
// FP64 refinement of B xi for a factor whose trailing updates ran in FP32 or
// BF16.  With L~ L~^T = D + E and M = inv(L~) D inv(L~)^T = I + X (X small
// and symmetric), B = L~ M^(1/2) satisfies B B^T = D exactly, and to first
// order B xi = L~ (xi + X xi / 2).  Since L~ X xi = D u - L~ xi for
// u = inv(L~)^T xi (L~^T u = xi), that is
//   B xi = (L~ xi + D u) / 2,   B B^T - D = L~ X^2 L~^T / 4 + O(X^3):
// one FP64 triangular solve with the factor (k_bsolve), one matrix-free
// product D u from the bead positions D was assembled from (k_dmul, the RPY
// blocks of k_rpy), and the mean taken in k_noise beside L~ xi.
// ---------------------------------------------------------------------------
__global__ void k_hi_snapshot(Stat s, Geo g, int nhi, double *xs) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nhi) return;
    const double3 r = hi_pos(s, g, b);
    xs[3 * b] = r.x;
    xs[3 * b + 1] = r.y;
    xs[3 * b + 2] = r.z;
}

__global__ void k_refine_init(const double *p, int m, int mpad, double *pw) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < mpad) pw[r] = r < m ? p[r] : 0.0;
}

// Column part of a 64x64 tile T (global, leading dimension ldt) for this
// thread: column e = t % 64, rows 16q .. 16q+15, q = t / 64 (a wavefront
// reads one row per load), loaded into registers ahead of use.
__device__ __forceinline__ void col_load(const double *T, size_t ldt, double (&v)[16]) {
    const int e = threadIdx.x & 63, q = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < 16; j++) v[j] = T[(16 * q + j) * ldt + e];
}
// part[q][e] = sum_j v[j] x[16q + j], then y[e] = sum_q part[q][e] in a
// fixed order for e < 64 (threads 0..63), with barriers around.
__device__ __forceinline__ void col_reduce(const double (&v)[16], const double *x, double *part, double *y,
                                           const double *sub) {
    const int t = threadIdx.x, e = t & 63, q = t >> 6;
    double a = 0.0;
#pragma unroll
    for (int j = 0; j < 16; j++) a += v[j] * x[16 * q + j];
    part[q * TB + e] = a;
    __syncthreads();
    if (t < TB) {
        const double sum = ((part[t] + part[TB + t]) + part[2 * TB + t]) + part[3 * TB + t];
        y[t] = sub ? sub[t] - sum : sum;
    }
    __syncthreads();
}

// Blocks b0 = 2g and b1 = 2g + 1 (if present) of u = inv(L~)^T xi; the
// blocks after them were solved by earlier launches, so pw there is final:
//   u_b1 = inv(L~_b1b1)^T pw_b1,  u_b0 = inv(L~_b0b0)^T (pw_b0 - L~_b1b0^T u_b1)
// in every workgroup (all tiles loaded at the start); workgroup 0 stores
// u_b0 and u_b1, workgroup k >= 1 subtracts L~_b0,i^T u_b0 + L~_b1,i^T u_b1
// from pw_i for tile row i = k - 1 < b0 (L~_b,i parked in block (i, b)).
__global__ void __launch_bounds__(256) k_bsolve(const double *A, int ld, const double *Linv, int nt, int g,
                                                double *pw, double *u) {
    __shared__ double x[2 * TB], u0[TB], u1[TB], part[4 * TB];
    const int t = threadIdx.x, b0 = 2 * g, two = b0 + 1 < nt, i = blockIdx.x - 1;
    double la[16], lc[16], lb[16], r0[16], r1[16];
    if (two) {
        col_load(Linv + (size_t)(b0 + 1) * TB * TB, TB, la);
        col_load(A + (size_t)b0 * TB * ld + (b0 + 1) * TB, ld, lc);
    }
    col_load(Linv + (size_t)b0 * TB * TB, TB, lb);
    if (i >= 0) {
        col_load(A + (size_t)i * TB * ld + b0 * TB, ld, r0);
        if (two) col_load(A + (size_t)i * TB * ld + (b0 + 1) * TB, ld, r1);
    }
    if (t < (two ? 2 : 1) * TB) x[t] = pw[b0 * TB + t];
    __syncthreads();
    if (two) {
        col_reduce(la, x + TB, part, u1, nullptr);
        col_reduce(lc, u1, part, x, x);  // pw_b0 - L~_b1b0^T u_b1, in place
    }
    col_reduce(lb, x, part, u0, nullptr);
    if (i < 0) {
        if (t < TB) u[b0 * TB + t] = u0[t];
        else if (two && t < 2 * TB) u[b0 * TB + t] = u1[t - TB];
        return;
    }
    const int e = t & 63, q = t >> 6;
    double a = 0.0;
#pragma unroll
    for (int j = 0; j < 16; j++) a += r0[j] * u0[16 * q + j];
    if (two)
#pragma unroll
        for (int j = 0; j < 16; j++) a += r1[j] * u1[16 * q + j];
    part[q * TB + e] = a;
    __syncthreads();
    if (t < TB) pw[i * TB + t] -= ((part[t] + part[TB + t]) + part[2 * TB + t]) + part[3 * TB + t];
}

// w = D u for the hydrodynamic set (m = 3 nhi rows): one wavefront per bead
// i, lanes over the beads j, the 3x3 blocks of k_rpy (a1/rad_i on the
// diagonal), lane sums combined in a fixed order.
__global__ void __launch_bounds__(256) k_dmul(const double *xs, const double *rad_all, int nhi, double a1, double a2,
                                              const double *u, double *w) {
    const int lane = threadIdx.x & 63, i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= nhi) return;
    const double3 ri = make_double3(xs[3 * i], xs[3 * i + 1], xs[3 * i + 2]);
    const double radi = rad_all[i];
    double acc[3] = {0.0, 0.0, 0.0};
    for (int j = lane; j < nhi; j += 64) {
        const double uj[3] = {u[3 * j], u[3 * j + 1], u[3 * j + 2]};
        if (j == i) {
            const double d = a1 / radi;
#pragma unroll
            for (int k = 0; k < 3; k++) acc[k] += d * uj[k];
        } else {
            const double3 u3 = rpy_apply(ri, make_double3(xs[3 * j], xs[3 * j + 1], xs[3 * j + 2]), radi, rad_all[j], a1, a2,
                                         make_double3(uj[0], uj[1], uj[2]));
            acc[0] += u3.x;
            acc[1] += u3.y;
            acc[2] += u3.z;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
        for (int o = 32; o > 0; o >>= 1) acc[k] += __shfl_down(acc[k], o, 64);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < 3; k++) w[3 * i + k] = acc[k];
}

// ---------------------------------------------------------------------------
void launch_rpy(const Stat &s, int n_hi, const Geo &g, const double *rad_all, const CholWork &c, hipStream_t q,
                bool factor_first) {
    const int nt = c.mpad / TB;
    // the positions D is built from, kept only where a refinement can read them
    if (refine_active(c)) k_hi_snapshot<<<nblk(c.m / 3, 256), 256, 0, q>>>(s, g, c.m / 3, c.xs);
    // the first tile's factor inside the assembly launch saves a launch on
    // the factor's chain, but gives every workgroup the factor's LDS (43 KB,
    // three per CU): for many tiles the assembly takes its own launch (33 KB,
    // four per CU) and k_diag the first tile.  One launch / two, us: 17 block
    // columns 21 / 26, 33 21 / 29, 52 25 / 39, 66 30 / 42, 99 64 / 70, 164 160
    // / 127, 328 515 / 445; the factor as a whole differs by more than its
    // runs up to 66 only (33: 504 / 515 us, 66: 1357 / 1366)
    if (factor_first && nt < 64) {
        k_rpy<true><<<nt * (nt + 1) / 2, 256, 0, q>>>(s, g, rad_all, c.A, c.m, c.ld, s.a1, s.a2, c.neg, c.Linv);
    } else {
        k_rpy<false><<<nt * (nt + 1) / 2, 256, 0, q>>>(s, g, rad_all, c.A, c.m, c.ld, s.a1, s.a2, c.neg, c.Linv);
        if (factor_first) launch_diag(c, 0, false, q);
    }
    (void)n_hi;
}

namespace {
template <int MODE>
void chol_column(const CholWork &c, int kb, int jcols, hipStream_t q) {
    const int nt = c.mpad / TB, M = nt - kb - 1;
    const int grid = jcols * (jcols + 1) / 2 + (M - jcols) * jcols;
    if (jcols == 0) {
        k_panel<<<M, 256, 0, q>>>(c.A, c.ld, kb, c.Linv);
    } else if (grid >= c.split_tiles) {
        k_panel<<<M, 256, 0, q>>>(c.A, c.ld, kb, c.Linv);
        k_update<MODE><<<grid, 256, 0, q>>>(c.A, c.ld, kb, jcols, c.Linv, c.neg);
    } else if (grid > c.ncu && grid <= kStep2Tiles(c.ncu / 8 * 8)) {
        k_step2<MODE><<<c.ncu / 8 * 8, 512, 0, q>>>(c.A, c.ld, kb, jcols, grid, c.Linv, c.neg);
    } else {
        k_step<MODE><<<grid, 256, 0, q>>>(c.A, c.ld, kb, jcols, c.Linv, c.neg);
    }
}
// tiles lin .. lin + n - 1 of the trailing update from packed panels
template <int MODE>
void trail_tiles(const CholWork &c, int nb, int j0, int lin, int n, hipStream_t q) {
    k_trail_pk<MODE><<<xcd_grid(n), 256, 0, q>>>(c.A, c.ld, c.sp, nb, j0, c.mpad / TB, lin, n, c.Linv, c.neg);
}
template <int MODE>
void trail_direct(const CholWork &c, int k0, int nb, hipStream_t q) {
    const int nt = c.mpad / TB, j0 = k0 + nb, SM = (nt - j0 + 7) / 8;
    k_trail<MODE><<<SM * (SM + 1) / 2 * 64, 256, 0, q>>>(c.A, c.ld, k0, nb, j0, nt, c.Linv, c.neg);
}
template <int MODE>
void chol_trail(const CholWork &c, int k0, int nb, hipStream_t q) {
    const int nt = c.mpad / TB, j0 = k0 + nb, R = nt - j0;
    if (c.sp && nb <= c.sp_nb && R >= c.pack_min_rows) {
        if constexpr (MODE == 2) {
            __bf16 *sp = static_cast<__bf16 *>(c.sp);
            const int S = (R + 1) / 2, n = S * (S + 1) / 2;
            k_split3<<<R * nb, 256, 0, q>>>(c.A, c.ld, k0, nb, j0, sp);
            k_trail_bf<<<xcd_grid(n), 256, 0, q>>>(c.A, c.ld, sp, nb, j0, nt, n, c.Linv, c.neg);
        } else {
            k_pack64<MODE><<<R * nb, 256, 0, q>>>(c.A, c.ld, k0, nb, j0, c.sp);
            trail_tiles<MODE>(c, nb, j0, 0, R * (R + 1) / 2, q);
        }
    } else {
        trail_direct<MODE>(c, k0, nb, q);
    }
}
// Factor in super-panels of kPanel block columns, FP64 and FP32 updates: per
// panel the columns of its diagonal block with the tiles of the last trailing
// update (one round of the CUs each), what is left of these tiles, the
// panel's rows, and the first tiles of its trailing update, among them the
// next diagonal block's.  The last block's columns are factored in c.mode's
// arithmetic, as they are without panels.  Against whole panels column by column and the
// trailing update in one launch (us, FP64): 200 nucleosomes 1449 -> 1375, 300
// 2920 -> 2670, 500 8730 -> 8100, 1000 55200 -> 52100; FP32 300 2400 -> 2140,
// 1000 37500 -> 32600.  In BF16, whose 128x128 blocks make poor company (300
// nucleosomes 2210 -> 2330), the panels stay whole.
template <int MODE>
void chol_panels(const CholWork &c, hipStream_t q, MarkFn mark, void *mark_arg, hipEvent_t gate, int gate_kb) {
    const int nt = c.mpad / TB, ncu = c.ncu;
    auto M_ = [&](int id, int ph) { if (mark) mark(mark_arg, id, ph); };
    auto done = [&](int kb) { if (gate && kb == gate_kb) (void)hipEventRecord(gate, q); };
    int j0 = 0, lin = 0, end = 0;  // the trailing update in progress: blocks lin .. end - 1 left
    for (int k0 = 0;; k0 += kPanel) {
        const int kend = std::min(k0 + kPanel, nt);
        for (int kb = k0; kb + 1 < kend; kb++) {
            if (kend == nt) {
                M_(K_CHOL_STEP, 0);
                chol_column<MODE>(c, kb, nt - kb - 1, q);
                M_(K_CHOL_STEP, 1);
                done(kb);
                continue;
            }
            const int jcols = kend - 1 - kb, G = jcols * (jcols + 1) / 2, n = std::min(end - lin, std::max(0, ncu - G) / 8 * 8);
            M_(K_CHOL_STEP, 0);
            k_block_step<MODE><<<G + xcd_grid(n), 256, 0, q>>>(c.A, c.ld, kb, jcols, c.sp, kPanel, j0, nt, lin, n, c.Linv, c.neg,
                                                              c.Lp + ((kb - k0) * kPanel + kb - k0 + 1) * TB * TB);
            M_(K_CHOL_STEP, 1);
            lin += n;
            done(kb);
        }
        if (kend == nt) break;
        if (lin < end) {
            M_(K_CHOL_TRAIL, 0);
            trail_tiles<MODE>(c, kPanel, j0, lin, end - lin, q);
            M_(K_CHOL_TRAIL, 1);
        }
        j0 = kend;
        const bool packed = c.sp && c.sp_nb >= kPanel && nt - j0 >= c.pack_min_rows;
        M_(K_CHOL_STEP, 0);
        k_panel_rows<MODE><<<4 * (nt - j0), 256, 0, q>>>(c.A, c.ld, k0, c.Linv, c.Lp, packed ? c.sp : nullptr);
        M_(K_CHOL_STEP, 1);
        done(kend - 1);
        M_(K_CHOL_TRAIL, 0);
        if (packed) {
            end = (nt - j0) * (nt - j0 + 1) / 2;
            lin = std::min(end, std::max(kPanel * (kPanel + 1) / 2, ncu / 8 * 8));
            k_block_step<MODE><<<xcd_grid(lin), 256, 0, q>>>(c.A, c.ld, 0, 0, c.sp, kPanel, j0, nt, 0, lin, c.Linv, c.neg, nullptr);
        } else {
            trail_direct<MODE>(c, k0, kPanel, q);
            lin = end = 0;
        }
        M_(K_CHOL_TRAIL, 1);
    }
}
}  // namespace

size_t split_bytes(int ld, int nb) {
    return std::max((size_t)(ld / TB) * nb * 3 * kSplitTile * sizeof(__bf16),
                    (size_t)(ld / TB) * nb * TB * TB * sizeof(double));
}

// Super-panels from 60 block columns in FP64 (us a factor without / with them:
// 56 block columns 1086 / 1088, 59 1181 / 1176, 63 1321 / 1263, 72 1703 /
// 1515).  In the reduced modes from 64: FP32 would gain from 52 (53 952 / 938,
// 63 1233 / 1110), but a panel's own columns are FP64, so the line also says
// which rounding errors a factor has.
int chol_panel_tiles(const CholWork &c) {
    const int nt = c.mpad / TB;
    if (c.panel_tiles > 0) return c.panel_tiles >= 2 && nt > c.panel_tiles ? c.panel_tiles : 0;
    if (c.panel_tiles < 0) return 0;
    return nt >= (c.mode == 0 ? 60 : 64) ? kPanel : 0;
}

void launch_cholesky(const CholWork &c, hipStream_t q, MarkFn mark, void *mark_arg, hipEvent_t gate, int gate_kb) {
    const int nt = c.mpad / TB;
    auto M_ = [&](int id, int ph) { if (mark) mark(mark_arg, id, ph); };
    auto column = [&](int kb, int jcols, int mode) {
        M_(K_CHOL_STEP, 0);
        if (mode == 0) chol_column<0>(c, kb, jcols, q);
        else if (mode == 1) chol_column<1>(c, kb, jcols, q);
        else chol_column<2>(c, kb, jcols, q);
        M_(K_CHOL_STEP, 1);
        if (gate && kb == gate_kb) (void)hipEventRecord(gate, q);
    };
    const int NB = chol_panel_tiles(c);
    int k0 = 0;
    if (NB == kPanel && c.mode != 2) {
        if (c.mode == 0) chol_panels<0>(c, q, mark, mark_arg, gate, gate_kb);
        else chol_panels<1>(c, q, mark, mark_arg, gate, gate_kb);
        if (gate && gate_kb >= nt - 1) (void)hipEventRecord(gate, q);
        return;
    }
    if (NB > 0) {
        // super-panels while a whole one and a trailing matrix remain; the
        // panel's own columns are factored in FP64 in every mode (the
        // reduced-precision modes apply to the trailing update k_trail)
        for (; k0 + NB < nt; k0 += NB) {
            const int kend = k0 + NB;
            for (int kb = k0; kb < kend; kb++) column(kb, kend - 1 - kb, 0);
            M_(K_CHOL_TRAIL, 0);
            if (c.mode == 0) chol_trail<0>(c, k0, NB, q);
            else if (c.mode == 1) chol_trail<1>(c, k0, NB, q);
            else chol_trail<2>(c, k0, NB, q);
            M_(K_CHOL_TRAIL, 1);
        }
    }
    // one launch (or two) per block column, each updating the whole trailing matrix
    for (int kb = k0; kb + 1 < nt; kb++) column(kb, nt - kb - 1, c.mode);
    if (gate && gate_kb >= nt - 1) (void)hipEventRecord(gate, q);
}

void launch_diag(const CholWork &c, int d, bool clear, hipStream_t q) {
    k_diag<<<1, 256, 0, q>>>(c.A, c.ld, d, c.Linv, c.neg, clear ? 1 : 0);
}

// A caller's matrix into the factor's storage: the lower triangle of D
// (row-major, leading dimension ldd), zeros above the diagonal and the
// identity on the padding rows; and back: the factor, unparked (the
// off-diagonal tile (ib, kb) lives in the upper block (kb, ib)), into L
// with zeros above the diagonal.
__global__ void k_pack(const double *__restrict__ D, int ldd, int m, double *__restrict__ A, int ld, int mpad) {
    const long long total = (long long)mpad * mpad;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int r = (int)(e / mpad), c = (int)(e % mpad);
        double v = 0.0;
        if (c <= r) v = (r < m) ? D[(size_t)r * ldd + c] : (r == c ? 1.0 : 0.0);
        A[(size_t)r * ld + c] = v;
    }
}
__global__ void k_unpark(const double *__restrict__ A, int ld, int m, double *__restrict__ L, int ldl) {
    const long long total = (long long)m * m;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(e / m), j = (int)(e % m), ib = i / TB, kb = j / TB;
        double v = 0.0;
        if (kb < ib) v = A[(size_t)(kb * TB + i % TB) * ld + ib * TB + j % TB];
        else if (j <= i) v = A[(size_t)i * ld + j];
        L[(size_t)i * ldl + j] = v;
    }
}

void launch_pack(const double *D, int ldd, const CholWork &c, hipStream_t q) {
    const long long total = (long long)c.mpad * c.mpad;
    const int grid = (int)std::min<long long>((total + 255) / 256, 4096);
    k_pack<<<grid, 256, 0, q>>>(D, ldd, c.m, c.A, c.ld, c.mpad);
}
void launch_unpark(const CholWork &c, double *L, int ldl, hipStream_t q) {
    const long long total = (long long)c.m * c.m;
    const int grid = (int)std::max<long long>(1, std::min<long long>((total + 255) / 256, 4096));
    k_unpark<<<grid, 256, 0, q>>>(c.A, c.ld, c.m, L, ldl);
}

bool refine_active(const CholWork &c) { return c.mode != 0 && c.refine && c.m > 0 && c.xs; }

void launch_refine(const Stat &s, const CholWork &c, const double *p, const double *rad_all, hipStream_t q) {
    const int nt = c.mpad / TB, nhi = c.m / 3, ng = nblk(nt, 2);
    double *pw = c.rv, *u = c.rv + c.ld;
    k_refine_init<<<nblk(c.mpad, 256), 256, 0, q>>>(p, c.m, c.mpad, pw);
    for (int g = ng - 1; g >= 0; g--) k_bsolve<<<1 + 2 * g, 256, 0, q>>>(c.A, c.ld, c.Linv, nt, g, pw, u);
    k_dmul<<<nblk(nhi, 4), 256, 0, q>>>(c.xs, rad_all, nhi, s.a1, s.a2, u, c.pr);
}

void launch_noise(const Stat &s, int n_hi, int n_D3, const CholWork &c, const double *p, const double *rad_all,
                  double *rd, hipStream_t q, const double *du) {
    k_noise<<<nblk(n_D3, 4), 256, 0, q>>>(c.A, c.ld, c.m, n_D3, p, du, rad_all, s.s2dt, s.a1, rd);
    (void)n_hi;
}

}  // namespace bd
