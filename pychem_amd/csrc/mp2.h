// mp2.h -- internal launchers of mp2.hip / mp2_bf16.hip (matrix-core
// products, MP2 energy).
#pragma once
#include <hip/hip_runtime.h>

struct GemmF64Args {
    const double* A;
    const double* B;
    double* C;
    long long lda, ldb, ldc;      // leading dimensions (elements)
    long long sA, sB, sC;         // batch strides (elements)
    int M, N, K;
    int ta, tb;                   // A stored k-major (K x M) / B stored n-major (N x K)
    double alpha, beta;
};

// One product out(m, c) = sum_k P(m, k) Q(c, k) with a short side m (an
// orbital space, in tiles of MB * 16 rows) and a long side c (in tiles of
// PQ_TC columns).
//   P: k-major P[k * ldp + m] (pk) or P[m * ldp + k].
//   Q: by qmode, k-major Q[k * ldq + c] (PQ_QK), Q[c * ldq + k] (PQ_QROW), or
//      a row of symmetric packed matrices (PQ_QSYM): c = g * cn + nu, element
//      Q[g * ldq + tab[k * cn + nu]]; tab has PQ_TABPAD rows of zeros past K.
//   out: m * ldc + c; with cn > 0 (c / cn) * s1 + c % cn + m * ldc; with sw
//      (the operands of the matrix instruction swapped, so that a lane's
//      neighbours hold neighbouring m) c * ldc + m.
struct LongGemm {
    const double* P;
    const double* Q;
    double* C;
    const int* tab;
    long long ldp, ldq, ldc, s1;
    long long sP, sQ, sC;
    int M, N, K, cn;
    int pk, qmode, sw;
    double alpha, beta;
    int mt, nt, mb;               // set by the launcher: tiles along m and c, 16-row blocks per m tile
};

#define PQ_QK 0
#define PQ_QROW 1
#define PQ_QSYM 2
#define PQ_TC 128
#define PQ_MBMAX 5
#define PQ_TABPAD 64

// m tiles of equal height, at most 80 rows: 41 orbitals are one tile of 48
// rows, 81 two of 48, 153 two of 80.  (64-row tiles for every product ran the
// 41-row quarter transform at 64 % use.)
static inline void long_gemm_tiles(LongGemm& g)
{
    const int blocks = (g.M + 15) / 16;
    g.mt = (blocks + PQ_MBMAX - 1) / PQ_MBMAX;
    g.mb = (blocks + g.mt - 1) / g.mt;
    g.nt = (int)(((long long)g.N + PQ_TC - 1) / PQ_TC);
}

// block index -> (m tile, c tile): blocks go round the eight XCDs, so the m
// tiles of one c tile get indices 8 apart and share that XCD's L2 copy of Q
__device__ __forceinline__ bool long_gemm_tile(const LongGemm& g, int& m0, int& c0)
{
    const int xcd = blockIdx.x & 7, s = blockIdx.x >> 3;
    const int t = (s / g.mt) * 8 + xcd;
    if (t >= g.nt) return false;
    m0 = (s % g.mt) * g.mb * 16;
    c0 = t * PQ_TC;
    return true;
}

static inline dim3 long_gemm_grid(const LongGemm& g, int batch)
{
    return dim3((unsigned)(8LL * g.mt * ((g.nt + 7) / 8)), 1, (unsigned)batch);
}

int long_gemm_f64(LongGemm g, int batch, hipStream_t st);
// Same product with split-BF16 (hi*hi + hi*lo + lo*hi) MFMA, FP32 accumulation, FP64 in/out.
int long_gemm_bf16x3(LongGemm g, int batch, hipStream_t st);

// op(A) op(B) as a LongGemm: the longer of M and N is the long side
static inline LongGemm long_gemm_of(const GemmF64Args& a)
{
    LongGemm g = {};
    g.C = a.C;
    g.ldc = a.ldc;
    g.sC = a.sC;
    g.K = a.K;
    g.alpha = a.alpha;
    g.beta = a.beta;
    if (a.N >= a.M) {
        g.P = a.A; g.ldp = a.lda; g.sP = a.sA; g.M = a.M; g.pk = a.ta;
        g.Q = a.B; g.ldq = a.ldb; g.sQ = a.sB; g.N = a.N; g.qmode = a.tb ? PQ_QROW : PQ_QK;
    } else {
        g.sw = 1;
        g.P = a.B; g.ldp = a.ldb; g.sP = a.sB; g.M = a.N; g.pk = !a.tb;
        g.Q = a.A; g.ldq = a.lda; g.sQ = a.sA; g.N = a.M; g.qmode = a.ta ? PQ_QK : PQ_QROW;
    }
    return g;
}

// the kernel of one (mb, pk, qmode, sw); QSYM exists for k-major P without sw
#define LONG_GEMM_CASE(KERN, MB)                                                                                       \
    case MB:                                                                                                           \
        if (g.qmode == PQ_QSYM) hipLaunchKernelGGL((KERN<MB, 1, PQ_QSYM, 0>), grid, block, 0, st, g);                  \
        else if (g.qmode == PQ_QK) {                                                                                   \
            if (g.sw) {                                                                                                \
                if (g.pk) hipLaunchKernelGGL((KERN<MB, 1, PQ_QK, 1>), grid, block, 0, st, g);                          \
                else hipLaunchKernelGGL((KERN<MB, 0, PQ_QK, 1>), grid, block, 0, st, g);                               \
            } else {                                                                                                   \
                if (g.pk) hipLaunchKernelGGL((KERN<MB, 1, PQ_QK, 0>), grid, block, 0, st, g);                          \
                else hipLaunchKernelGGL((KERN<MB, 0, PQ_QK, 0>), grid, block, 0, st, g);                               \
            }                                                                                                          \
        } else {                                                                                                       \
            if (g.sw) {                                                                                                \
                if (g.pk) hipLaunchKernelGGL((KERN<MB, 1, PQ_QROW, 1>), grid, block, 0, st, g);                        \
                else hipLaunchKernelGGL((KERN<MB, 0, PQ_QROW, 1>), grid, block, 0, st, g);                             \
            } else {                                                                                                   \
                if (g.pk) hipLaunchKernelGGL((KERN<MB, 1, PQ_QROW, 0>), grid, block, 0, st, g);                        \
                else hipLaunchKernelGGL((KERN<MB, 0, PQ_QROW, 0>), grid, block, 0, st, g);                             \
            }                                                                                                          \
        }                                                                                                              \
        break;

#define LONG_GEMM_LAUNCH(KERN)                                                                                         \
    if (g.M <= 0 || g.N <= 0 || batch <= 0) return 0;                                                                  \
    if (g.K <= 0) return -1;                                                                                           \
    if (g.qmode == PQ_QSYM && (!g.pk || g.sw || !g.tab || g.cn <= 0)) return -1;                                       \
    long_gemm_tiles(g);                                                                                                \
    const dim3 grid = long_gemm_grid(g, batch), block(256);                                                            \
    switch (g.mb) {                                                                                                    \
        LONG_GEMM_CASE(KERN, 1)                                                                                        \
        LONG_GEMM_CASE(KERN, 2)                                                                                        \
        LONG_GEMM_CASE(KERN, 3)                                                                                        \
        LONG_GEMM_CASE(KERN, 4)                                                                                        \
        LONG_GEMM_CASE(KERN, 5)                                                                                        \
    default: return -1;                                                                                                \
    }                                                                                                                  \
    return hipGetLastError() == hipSuccess ? 0 : -1;

int mp2_energy_launch(const double* ovov, const double* eo1, const double* ev1, const double* eo2, const double* ev2,
                      int o1, int v1, int o2, int v2, int mode, double* out, hipStream_t st);
