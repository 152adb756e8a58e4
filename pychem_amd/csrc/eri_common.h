// eri_common.h -- device-side types, Boys function and per-class kernel
// templates shared by the generated class translation units and the host code.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#ifndef ERI_BLOCK
#define ERI_BLOCK 256
#endif

struct PairHdr {
    double ab[3];   // X1 - X2 (primary minus secondary centre)
    int off;        // first primitive pair
    int n;          // primitive pairs kept
    int s1, s2;     // shells: primary, secondary
    int pcls;       // pair class 0..5: ss ps pp ds dp dd
    int mol;        // molecule of both shells
};

// One molecule of a (possibly batched) basis: its matrices are the n x n
// block at offset base of the packed matrix arrays; its atoms are
// [atom_lo, atom_hi).  Shell AO offsets are local to the molecule.
struct MolInfo {
    long long base;
    int n;
    int atom_lo, atom_hi;
    int pad;
};

// Ks = K sqrt(p) (2/sqrt(pi))^(1/2): the Coulomb prefactor of a primitive
// quartet, K_P K_Q (2/sqrt(pi)) sqrt(pq/(p+q)), is Ks_P Ks_Q / sqrt(p+q).
// 96 bytes, so that every record starts on a 16-byte boundary.
template <typename real>
struct PrimPair {
    real Px, Py, Pz, p, Ks, PAx, PAy, PAz, inv2p, K, beta, pad;
};

// Constant address space: a load through such a pointer at a wave-uniform
// address is a scalar load.  The primitive pairs are read-only in every
// kernel that reads them this way.
#define ERI_CONST __attribute__((address_space(4)))

__device__ __forceinline__ PrimPair<double> prim_ld_u(const ERI_CONST PrimPair<double>* q)
{
    PrimPair<double> r;
    r.Px = q->Px; r.Py = q->Py; r.Pz = q->Pz;
    r.PAx = q->PAx; r.PAy = q->PAy; r.PAz = q->PAz;
    r.p = q->p; r.inv2p = q->inv2p; r.K = q->K; r.beta = q->beta; r.Ks = q->Ks; r.pad = q->pad;
    return r;
}

template <typename real>
struct EriArgs {
    const int2* quartets;
    const PairHdr* pairs;
    const PrimPair<double>* prims;   // FP64 for both precisions
    real* out;
    int nq;
    const int* order;   // thread t computes quartet order[t] (NULL: quartet t)
    double scatt_S = 0.0;   // momentum transfer of the scattering operator (OP = 1 kernels)
};

struct OneeArgs {
    const int* pair_list;
    const PairHdr* pairs;
    const PrimPair<double>* prims;
    const double* atoms;     // x, y, z, Z per atom
    const int* cart_off;
    const MolInfo* mols;
    double *S, *T, *V;       // packed per-molecule blocks
    int npair;
};
// the six pair classes in one launch: class p covers blocks [block0[p],
// block0[p + 1]) of 128 threads, G lanes per shell pair (G: power of two <= 64)
struct OneeFusedArgs {
    OneeArgs cls[6];
    int block0[7];
    int G;
};

template <typename real>
struct JkArgs {
    const int2* quartets;
    const PairHdr* pairs;
    const int* cart_off;
    const MolInfo* mols;
    const real* vals;
    const double* Dj;   // density for J (ncart x ncart)
    const double* Dk;   // density for K
    double* J;          // accumulates J' (unsymmetrised)
    double* K;          // accumulates K' (unsymmetrised, positive)
    int nq, n;
};

template <typename real>
struct ScatterArgs {
    const int2* quartets;
    const PairHdr* pairs;
    const int* cart_off;
    const real* vals;
    double* out;        // out[m][n][l - l0][s] for l in [l0, l0 + lc)
    int nq, n, l0, lc;
};

template <typename real>
struct PairScatterArgs {
    const int2* quartets;
    const PairHdr* pairs;
    const int* pair_base;    // first packed index of each shell pair
    const real* vals;
    double* out;             // out[P - p0][Q], P in [p0, p0 + rows), Q in [0, np)
    long long p0, rows, np;
    int nq;
};

// index of functions (i, j) of a shell pair within its packed block: all
// N1 x N2 of two shells, i >= j of one shell with itself
__host__ __device__ __forceinline__ int pair_component(bool same, int n2, int i, int j)
{
    return same ? i * (i + 1) / 2 + j : i * n2 + j;
}

// --------------------------------------------------------------------------
// Boys function F_m(T), m = 0..L
//   T < 36: 9-term Taylor expansion of F_L about the nearest grid point
//           (tabulated F_n(k*0.1) from mpmath), then downward recursion
//           F_m = (2T F_{m+1} + e^-T)/(2m+1)
//   T >= 36: F_0 = sqrt(pi/T)/2, upward recursion F_{m+1} = ((2m+1)F_m - e^-T)/(2T)
// --------------------------------------------------------------------------
#include "boys_table.inc"

template <int L>
__device__ __forceinline__ void boys_eval(double T, double* F)
{
    if (T < BOYS_TMAX) {
        const int k = __double2int_rn(T * BOYS_INV_STEP);
        const double x = k * BOYS_STEP - T;
        const double* row = boys_table + k * BOYS_NCOL + L;
        double f = row[8];
#pragma unroll
        for (int j = 8; j >= 1; --j) f = row[j - 1] + f * (x * (1.0 / j));
        F[L] = f;
        if (L > 0) {
            const double e = exp(-T);
            const double t2 = 2.0 * T;
#pragma unroll
            for (int m = L - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * (1.0 / (2 * m + 1));
        }
    } else {
        const double it = 1.0 / T;
        F[0] = 0.88622692545275801365 * sqrt(it);
        if (L > 0) {
            const double e = exp(-T);
            const double h = 0.5 * it;
#pragma unroll
            for (int m = 0; m < L; ++m) F[m + 1] = ((2 * m + 1) * F[m] - e) * h;
        }
    }
}

template <int L>
__device__ __forceinline__ void boys_eval(float T, float* F)
{
    if (T < (float)BOYS_TMAX) {
        const int k = __float2int_rn(T * (float)BOYS_INV_STEP);
        const float x = k * (float)BOYS_STEP - T;
        const double* row = boys_table + k * BOYS_NCOL + L;
        float f = (float)row[5];
#pragma unroll
        for (int j = 5; j >= 1; --j) f = (float)row[j - 1] + f * (x * (1.0f / j));
        F[L] = f;
        if (L > 0) {
            const float e = __expf(-T);
            const float t2 = 2.0f * T;
#pragma unroll
            for (int m = L - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * (1.0f / (2 * m + 1));
        }
    } else {
        const float it = 1.0f / T;
        F[0] = 0.88622692545275801365f * sqrtf(it);
        if (L > 0) {
            const float e = __expf(-T);
            const float h = 0.5f * it;
#pragma unroll
            for (int m = 0; m < L; ++m) F[m + 1] = ((2 * m + 1) * F[m] - e) * h;
        }
    }
}

// The class kernels read the polynomial coefficients from LDS: a lookup
// gathers 8 or 9 doubles at a lane-dependent row, and from global memory that
// costs scattered 16-byte loads per lane and primitive quartet (the (ss|ss)
// and (ps|ss) kernels were bound by them).  The image (boys_stage_copy) holds
// BOYS_COLS doubles per grid point T_k, coefficients of x^c, x = T_k - T,
// divided by c!, so that the expansion is a Horner chain of fused
// multiply-adds:
//   L = 0                    F_0, degree 7
//   L <= BOYS_PAIR_MAX       F_{L-1}, degree 8; its derivative in x is F_L
//   above                    F_L, degree 8, and e^{-T_k}
// The first two are Taylor polynomials of one degree more less their top
// Chebyshev component: off by 4e-19, below the 5e-18 of the degree 8 Taylor
// polynomial they replace.  Rows are an odd number (5) of 16-byte units: a
// random row then spreads over all banks and is read 16 bytes at a time, 46
// cycles of the CU's LDS for the 8 doubles of a wave, where 9 doubles in rows
// of 9 took 96 with 8-byte reads; (ss|ss), whose four SIMDs can issue a
// primitive quartet in some 170 cycles, was bound by those 4 x 96.  The pair
// of orders from one polynomial and the shorter far branch leave (ps|ss) 79
// vector instructions of 124 where a wave takes both branches.  The pass over
// C20H42's lists went from 3.13 to 2.87 ms, over C14H30's from 1.72 to 1.58.
#define BOYS_TERMS 9
#define BOYS_COLS 10
#define BOYS_LDS_DOUBLES (BOYS_NPTS * BOYS_COLS)
#define BOYS_PAIR_MAX 5

// The class kernels copy a prepared image of those LDS rows (generated per
// order L from boys_table.inc): a coalesced copy, two doubles a load.
__device__ __forceinline__ void boys_stage_copy(double* __restrict__ s, const double* __restrict__ src, const int n)
{
    const double2* __restrict__ src2 = (const double2*)src;
    double2* s2 = (double2*)s;
    for (int e = threadIdx.x; e < n / 2; e += blockDim.x) s2[e] = src2[e];
    if ((n & 1) && threadIdx.x == 0) s[n - 1] = src[n - 1];
    __syncthreads();
}

// 1/sqrt(s) for positive normal s: the hardware estimate y (2^-22 relative
// or better) and the next two terms of its error series,
// y (1 - e)^{-1/2} = y + y e (1/2 + 3/8 e) + O(e^3), e = 1 - s y^2.
__device__ __forceinline__ double rsqrt_nr(const double s)
{
    const double y = __builtin_amdgcn_rsq(s);
    const double e = fma(-s * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// e^{-T} for T >= BOYS_TMAX: n = rint(T / ln 2), r = T - n ln 2 in [-0.35,
// 0.35], e^{-r} by its Taylor polynomial of degree DEG, scaled by 2^-n.  In
// the upward recursion above T = 36 the e^{-T} term is at most 1.6e-15,
// 3.7e-14, 5e-13, 5.6e-12, 4.4e-11 and, for m = 7, 8e-9 of (2m+1) F_m, m = 0,
// 1, ..., 4; a polynomial good to 6e-4 (degree 3), 4e-5, 2.4e-6, 1.2e-7, 5e-9
// and 2e-10 (degree 8) leaves F_{m+1} exact to rounding.  2^-n underflows to
// 0 where e^{-T} does.
template <int DEG>
__device__ __forceinline__ double exp_neg_tail(const double T)
{
    const double n = rint(T * -1.4426950408889634);
    const double r = fma(n, 0.69314718055994531, T);
    constexpr double c[9] = {1.0, -1.0, 1.0 / 2, -1.0 / 6, 1.0 / 24, -1.0 / 120, 1.0 / 720, -1.0 / 5040, 1.0 / 40320};
    double p = c[DEG];
#pragma unroll
    for (int j = DEG - 1; j >= 0; --j) p = fma(p, r, c[j]);
    return ldexp(p, (int)fmax(n, -2000.0));
}

template <int L>
__device__ __forceinline__ void boys_eval_s(double T, double* F, const double* __restrict__ s)
{
    if (T < BOYS_TMAX) {
        // 1.5 x 2^52 rounds to the nearest grid point, k in the low word
        const double t = fma(T, BOYS_INV_STEP, 6755399441055744.0);
        const double x = fma(t - 6755399441055744.0, BOYS_STEP, -T);
        const double2* row = (const double2*)s + __umul24(__double2loint(t), BOYS_COLS / 2);
        double c[BOYS_COLS];
#pragma unroll
        for (int j = 0; j < (L == 0 ? 4 : 5); ++j) {
            const double2 v = row[j];
            c[2 * j] = v.x;
            c[2 * j + 1] = v.y;
        }
        if constexpr (L == 0) {
            double f = c[7];
#pragma unroll
            for (int j = 6; j >= 0; --j) f = fma(f, x, c[j]);
            F[0] = f;
        } else if constexpr (L <= BOYS_PAIR_MAX) {
            double d = c[8], f = fma(c[8], x, c[7]);
#pragma unroll
            for (int j = 6; j >= 0; --j) {
                d = fma(d, x, f);
                f = fma(f, x, c[j]);
            }
            F[L] = d;
            F[L - 1] = f;
            if constexpr (L > 1) {   // e^{-T} = (2m+1) F_m - 2T F_{m+1}
                const double t2 = 2.0 * T;
                const double e = fma(-t2, d, (2 * L - 1) * f);
#pragma unroll
                for (int m = L - 2; m >= 0; --m) F[m] = fma(t2, F[m + 1], e) * (1.0 / (2 * m + 1));
            }
        } else {
            double f = c[8];
#pragma unroll
            for (int j = 7; j >= 0; --j) f = fma(f, x, c[j]);
            F[L] = f;
            constexpr double w[8] = {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040};
            double ex = 1.0 / 40320;
#pragma unroll
            for (int j = 7; j >= 0; --j) ex = fma(ex, x, w[j]);
            const double e = c[BOYS_TERMS] * ex;
            const double t2 = 2.0 * T;
#pragma unroll
            for (int m = L - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * (1.0 / (2 * m + 1));
        }
    } else {
        const double y = rsqrt_nr(T);
        F[0] = 0.88622692545275801365 * y;
        if (L > 0) {
            const double e = exp_neg_tail<(L <= 5 ? L + 2 : 8)>(T);
            const double h = 0.5 * y * y;
#pragma unroll
            for (int m = 0; m < L; ++m) F[m + 1] = ((2 * m + 1) * F[m] - e) * h;
        }
    }
}

template <int L>
__device__ __forceinline__ void boys_eval_s(float T, float* F, const double* __restrict__ s)
{
    if (T < (float)BOYS_TMAX) {
        const int k = __float2int_rn(T * (float)BOYS_INV_STEP);
        const float x = k * (float)BOYS_STEP - T;
        const double2* row = (const double2*)s + __umul24(k, BOYS_COLS / 2);
        float c[8];
#pragma unroll
        for (int j = 0; j < (L == 0 || L > BOYS_PAIR_MAX ? 3 : 4); ++j) {
            const double2 v = row[j];
            c[2 * j] = (float)v.x;
            c[2 * j + 1] = (float)v.y;
        }
        constexpr int M = L == 0 || L > BOYS_PAIR_MAX ? L : L - 1;   // the order whose polynomial the row holds
        float f, d = 0.0f;
        if constexpr (M < L) {
            d = c[6];
            f = fmaf(c[6], x, c[5]);
#pragma unroll
            for (int j = 4; j >= 0; --j) {
                d = fmaf(d, x, f);
                f = fmaf(f, x, c[j]);
            }
            F[L] = d;
        } else {
            f = c[5];
#pragma unroll
            for (int j = 4; j >= 0; --j) f = fmaf(f, x, c[j]);
        }
        F[M] = f;
        if (M > 0) {
            const float e = __expf(-T);
            const float t2 = 2.0f * T;
#pragma unroll
            for (int m = M - 1; m >= 0; --m) F[m] = (t2 * F[m + 1] + e) * (1.0f / (2 * m + 1));
        }
    } else {
        boys_eval<L>(T, F);
    }
}

// z^-m j_m(z) for m = 0..L (spherical Bessel functions of the first kind),
// evaluated piecewise as Methods/c_ints/spherical_bessel_j.c:5-81 does: the
// power series about z = 0 below z = 10 (1, 3, 6 or 20 terms above it for z
// below 1e-3, 0.1, 1, 10), the two-term asymptotic form above z = 100, and
// upward recursion of j_m from j_0, j_1 in between; values below 1e-16 in
// magnitude are set to zero.
template <int L>
__device__ __forceinline__ void bessel_zm_jm(double z, double* j)
{
    if (z < 10.0) {
        const int kmax = z < 1e-3 ? 1 : (z < 1e-1 ? 3 : (z < 1.0 ? 6 : 20));
        const double z2 = z * z;
        double df = 1.0;
#pragma unroll
        for (int m = 0; m <= L; ++m) {
            const double mm1 = (double)(2 * m + 1);
            df *= mm1;
            double jsum = 1.0, mm_df = 1.0, mm = mm1, zz = 1.0, sign = 1.0, denom = 1.0;
            for (int k = 1; k <= kmax; ++k) {
                mm += 2.0;
                mm_df *= mm;
                zz *= z2;
                sign = -sign;
                denom *= 2.0 * k;
                jsum += sign * zz / (denom * mm_df);
            }
            j[m] = jsum / df;
        }
    } else if (z > 100.0) {
        const double zinv = 1.0 / z, zinv2 = zinv * zinv;
        double sz, cz;
        sincos(z, &sz, &cz);
        j[0] = sz * zinv;
        double zi = 1.0, zoff = z;
#pragma unroll
        for (int m = 1; m <= L; ++m) {
            const double mm1 = (double)(m * (m + 1) / 2);
            zi *= zinv;
            zoff -= 1.5707963267948966;
            double so, co;
            sincos(zoff, &so, &co);
            j[m] = zi * (zinv * so + mm1 * zinv2 * co);
        }
    } else {
        const double zinv = 1.0 / z;
        double sz, cz;
        sincos(z, &sz, &cz);
        double jm2 = sz * zinv;                            // j_0
        double jm1 = L >= 1 ? (sz - z * cz) * zinv * zinv : 0.0;   // j_1
        j[0] = jm2;
        if (L >= 1) j[1] = jm1 * zinv;
        double zp = zinv;                                  // z^-m
#pragma unroll
        for (int m = 2; m <= L; ++m) {
            const double jm = (2 * m - 1) * jm1 * zinv - jm2;
            jm2 = jm1;
            jm1 = jm;
            zp *= zinv;
            j[m] = jm * zp;
        }
    }
#pragma unroll
    for (int m = 0; m <= L; ++m)
        if (fabs(j[m]) < 1e-16) j[m] = 0.0;
}

// The electron-scattering auxiliary function in the unscaled form of the
// VRR below.  The reference's fundamentals for ints_type 1
// (Methods/c_ints/two_electron_scattering.c:6-84) are
// U_P U_Q exp(-S^2 (sigma_P + sigma_Q)/4) S^(2m) z^-m j_m(z), z = S |P - Q|,
// in its scaled convention (a factor (2 rho)^m over the unscaled one); with
// S below 1e-14 only m = 0 survives (= U_P U_Q), and at |P - Q|^2 below 1e-14
// z^-m j_m(z) is its limit 1/(2m+1)!!.  KK = U_P U_Q times the contraction
// coefficients.
template <int L, typename real>
__device__ __forceinline__ void scatt_aux(double S, double rho, double R2, double sig_sum, double KK, real* F,
                                          real& pref)
{
    if (S < 1e-14) {
        pref = (real)KK;
        F[0] = (real)1.0;
#pragma unroll
        for (int m = 1; m <= L; ++m) F[m] = (real)0.0;
        return;
    }
    const double S2 = S * S;
    pref = (real)(KK * exp(-0.25 * S2 * sig_sum));
    double g[L + 1];
    if (R2 < 1e-14) {
        double df = 1.0;
#pragma unroll
        for (int m = 0; m <= L; ++m) {
            df *= (double)(2 * m + 1);
            g[m] = 1.0 / df;
        }
    } else {
        bessel_zm_jm<L>(S * sqrt(R2), g);
    }
    const double r = S2 / (2.0 * rho);
    double p = 1.0;
#pragma unroll
    for (int m = 0; m <= L; ++m) {
        F[m] = (real)(p * g[m]);
        p *= r;
    }
}

// Per primitive quartet: prefactor and recurrence coefficients for the
// unscaled Obara-Saika VRR.  W - P = -(q/(p+q)) (P-Q), W - Q = (p/(p+q)) (P-Q).
// The geometry (P-Q, T, prefactor) is always formed in FP64 from the FP64
// primitive-pair data; the FP32 kernels round only after that, so centre
// coordinates never lose digits to single precision.
// OP (a template parameter of the class body) selects the operator: 0 the
// Coulomb operator (Boys function), 1 the electron-scattering operator at
// momentum transfer args.scatt_S.
#define ERI_PRIM_SETUP(LL)                                                          \
    const double pd_ = P.p, qd_ = Q.p;                                              \
    const double rs_d = rsqrt_nr(pd_ + qd_);                                        \
    const double ipq_d = rs_d * rs_d;                                               \
    const double rho_d = pd_ * qd_ * ipq_d;                                         \
    const double PQx_d = P.Px - Q.Px, PQy_d = P.Py - Q.Py, PQz_d = P.Pz - Q.Pz;     \
    const double R2_d = PQx_d * PQx_d + PQy_d * PQy_d + PQz_d * PQz_d;              \
    real F[(LL) + 1];                                                               \
    real pref;                                                                      \
    if constexpr (OP == 0) {                                                        \
        boys_eval_s<(LL)>((real)(rho_d * R2_d), F, btab);                           \
        pref = (real)(P.Ks * Q.Ks * rs_d);                                          \
    } else {                                                                        \
        scatt_aux<(LL), real>(args.scatt_S, rho_d, R2_d, 1.0 / pd_ + 1.0 / qd_,     \
                              P.K * Q.K, F, pref);                                  \
    }                                                                               \
    const real ipq = (real)ipq_d;                                                   \
    const real rho_p = (real)(qd_ * ipq_d), rho_q = (real)(pd_ * ipq_d);            \
    const real PQx = (real)PQx_d, PQy = (real)PQy_d, PQz = (real)PQz_d;             \
    const real WPx = -rho_p * PQx, WPy = -rho_p * PQy, WPz = -rho_p * PQz;          \
    const real WQx = rho_q * PQx, WQy = rho_q * PQy, WQz = rho_q * PQz;             \
    const real PAx = (real)P.PAx, PAy = (real)P.PAy, PAz = (real)P.PAz;             \
    const real QCx = (real)Q.PAx, QCy = (real)Q.PAy, QCz = (real)Q.PAz;             \
    const real oo2p = (real)P.inv2p, oo2q = (real)Q.inv2p, oo2pq = (real)0.5 * ipq; \
    (void)WPx; (void)WPy; (void)WPz; (void)WQx; (void)WQy; (void)WQz;               \
    (void)PAx; (void)PAy; (void)PAz; (void)QCx; (void)QCy; (void)QCz;               \
    (void)oo2p; (void)oo2q; (void)oo2pq; (void)rho_p; (void)rho_q;
