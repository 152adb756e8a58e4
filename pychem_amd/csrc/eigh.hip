// eigh.hip -- eigenvalues and eigenvectors of many small symmetric matrices
// at once (the batched SCF's overlap matrices, one per molecule).
//
// One workgroup per matrix, the matrix and the accumulated rotations in LDS.
// Cyclic Jacobi in the round-robin (tournament) order: index 0 stays, the
// others rotate one place per round, so each of the m - 1 rounds of a sweep
// rotates m / 2 disjoint pairs together (m: the last row that couples to
// another, plus one, rounded up to even; the rows behind it, a small
// molecule's padding, are eigenvectors as they stand).  Each rotation zeroes
// its pair's off-diagonal element, with Rutishauser's formula: theta = (a_qq -
// a_pp) / (2 a_pq), t = sign(theta) / (|theta| + sqrt(theta^2 + 1)), c = 1 /
// sqrt(t^2 + 1), s = t c, and rows, then columns of A and the columns of V are
// updated as A <- J^T A J, V <- V J: the 2 x 2 block of two pairs by one lane,
// rows and columns in one pass, a half wave or a wave along one pair's row of
// blocks.  Sweeps stop when the off-diagonal sum of squares is below 1e-30
// times the diagonal's (of the coupled rows: a padding of 1e3 must not loosen
// it).  Eigenvalues are returned in ascending order with
// their eigenvectors as columns.
//
// Bound by the rounds' latency (two barriers and the chain of two divisions
// and two square roots): 512 matrices of 61 rows, molecules of 7 to 61
// functions, 1.44 ms (2.97 with the padding rotated too, separate passes over
// rows and columns and a division per element).
#include <hip/hip_runtime.h>
#include <math.h>

#include <string>

#include "scf.h"

#define EIGH_MAXN 90    // 2 n^2 doubles of LDS: 129.6 KB at n = 90
#define EIGH_MAX_SWEEPS 30

__device__ __forceinline__ double eigh_block_sum(double v, double* red)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    return s;
}

#define EIGH_W 8        // waves per matrix
__global__ void __launch_bounds__(64 * EIGH_W) eigh_jacobi_kernel(const double* __restrict__ A, int n,
                                                                  double* __restrict__ w, double* __restrict__ V)
{
    extern __shared__ double sh[];
    double* a = sh;           // n x n, row-major
    double* v = sh + n * n;   // n x n, the rotations' product
    __shared__ double cs[EIGH_MAXN / 2 + 1], sn[EIGH_MAXN / 2 + 1];
    __shared__ int pp[EIGH_MAXN / 2 + 1], qq[EIGH_MAXN / 2 + 1];
    __shared__ int perm[EIGH_MAXN], s_me;
    __shared__ double red[16], lam[EIGH_MAXN];
    const int tid = threadIdx.x, nt = 64 * EIGH_W, wave = tid >> 6, lane = tid & 63;
    const size_t off = (size_t)blockIdx.x * n * n;
    if (tid == 0) s_me = 0;
    __syncthreads();
    int me = 0;
    for (int i = tid; i < n * n; i += nt) {
        const int r = i / n, c = i - r * n;
        const double x = A[off + i];
        a[i] = x;
        v[i] = r == c ? 1.0 : 0.0;
        if (r != c && x != 0.0) me = max(me, max(r, c) + 1);
    }
    if (me) atomicMax(&s_me, me);
    __syncthreads();
    me = s_me;
    const int m = me + (me & 1);   // index me is a dummy when me is odd
    const int np = m / 2;
    // a row of 2 x 2 blocks along a half wave, two rows a wave, up to 64 players
    const int half = np <= 32 ? 32 : 64, pj = lane & (half - 1), pi0 = wave * (64 / half) + lane / half,
              pis = EIGH_W * (64 / half);
    for (int sweep = 0; sweep < EIGH_MAX_SWEEPS; ++sweep) {
        double o = 0.0, d = 0.0;
        for (int r = wave; r < me; r += EIGH_W)
            for (int c = r + 1 + lane; c < me; c += 64) o += a[r * n + c] * a[r * n + c];
        for (int i = tid; i < me; i += nt) d += a[i * n + i] * a[i * n + i];
        o = eigh_block_sum(o, red);
        d = eigh_block_sum(d, red);
        if (o <= 1e-30 * d || o == 0.0) break;
        for (int round = 0; round < m - 1; ++round) {
            if (tid < np) {
                // players at positions tid and m - 1 - tid of this round
                auto player = [&](int k) {
                    const int x = k - 1 + round;   // < 2 (m - 1)
                    return k == 0 ? 0 : (x >= m - 1 ? x - (m - 1) : x) + 1;
                };
                int p = player(tid), q = player(m - 1 - tid);
                if (p > q) {
                    const int x = p;
                    p = q;
                    q = x;
                }
                double c = 1.0, s = 0.0;
                if (q < me) {
                    const double apq = a[p * n + q];
                    if (apq != 0.0) {
                        const double theta = (a[q * n + q] - a[p * n + p]) / (2.0 * apq);
                        const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
                        c = 1.0 / sqrt(t * t + 1.0);
                        s = t * c;
                    }
                }
                pp[tid] = p;
                qq[tid] = q < me ? q : -1;   // a dummy pair rotates nothing
                cs[tid] = c;
                sn[tid] = s;
            }
            __syncthreads();
            if (pj < np) {   // rows of pair i, then columns of pair j
                const int pc = pp[pj], qc = qq[pj];
                const double cj = cs[pj], sj = sn[pj];
                for (int i = pi0; i < np; i += pis) {
                    const int pr = pp[i], qr = qq[i];
                    const double ci = cs[i], si = sn[i];
                    double* const x0 = a + pr * n;
                    double* const x1 = a + max(qr, 0) * n;
                    double a00 = x0[pc], a01 = qc >= 0 ? x0[qc] : 0.0;
                    double a10 = 0.0, a11 = 0.0;
                    if (qr >= 0) {
                        a10 = x1[pc];
                        a11 = qc >= 0 ? x1[qc] : 0.0;
                        const double t0 = ci * a00 - si * a10, t1 = ci * a01 - si * a11;
                        a10 = si * a00 + ci * a10;
                        a11 = si * a01 + ci * a11;
                        a00 = t0;
                        a01 = t1;
                    }
                    if (qc >= 0) {
                        const double t0 = cj * a00 - sj * a01, t1 = cj * a10 - sj * a11;
                        a01 = sj * a00 + cj * a01;
                        a11 = sj * a10 + cj * a11;
                        a00 = t0;
                        a10 = t1;
                        x0[qc] = a01;
                        if (qr >= 0) x1[qc] = a11;
                    }
                    x0[pc] = a00;
                    if (qr >= 0) x1[pc] = a10;
                }
            }
            for (int j = wave; j < np; j += EIGH_W) {   // columns p, q of V
                const int p = pp[j], q = qq[j];
                if (q < 0) continue;
                const double c = cs[j], s = sn[j];
                for (int k = lane; k < me; k += 64) {
                    const double xv = v[k * n + p], yv = v[k * n + q];
                    v[k * n + p] = c * xv - s * yv;
                    v[k * n + q] = s * xv + c * yv;
                }
            }
            __syncthreads();
        }
    }
    for (int i = tid; i < n; i += nt) {
        lam[i] = a[i * n + i];
        perm[i] = i;
    }
    __syncthreads();
    for (int i = tid; i < n; i += nt) {   // ascending order, equal ones as they come
        int rank = 0;
        for (int j = 0; j < n; ++j) rank += lam[j] < lam[i] || (lam[j] == lam[i] && j < i);
        perm[rank] = i;
    }
    __syncthreads();
    for (int i = tid; i < n; i += nt) w[(size_t)blockIdx.x * n + i] = lam[perm[i]];
    for (int i = tid; i < n * n; i += nt) {
        const int r = i / n, c = i - r * n;
        V[off + i] = v[r * n + perm[c]];
    }
}

extern "C" int pq_eigh_batched(const double* A, int batch, int n, double* w, double* V, void* stream)
{
    if (!A || !w || !V) return pq_set_error("pq_eigh_batched: null argument");
    if (batch < 0 || n < 1) return pq_set_error("pq_eigh_batched: need batch >= 0 and n >= 1");
    if (n > EIGH_MAXN)
        return pq_set_error(("pq_eigh_batched: n = " + std::to_string(n) + " exceeds the LDS-resident limit of " +
                             std::to_string(EIGH_MAXN)).c_str());
    if (batch == 0) return 0;
    const size_t lds = sizeof(double) * 2 * (size_t)n * n;
    static bool attr = false;
    if (!attr) {
        if (hipFuncSetAttribute((const void*)eigh_jacobi_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(sizeof(double) * 2 * EIGH_MAXN * EIGH_MAXN)) != hipSuccess)
            return pq_set_error("pq_eigh_batched: cannot raise the kernel's LDS limit");
        attr = true;
    }
    hipLaunchKernelGGL(eigh_jacobi_kernel, dim3(batch), dim3(64 * EIGH_W), lds, (hipStream_t)stream, A, n, w, V);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pq_set_error((std::string("pq_eigh_batched: ") + hipGetErrorString(e)).c_str());
    return 0;
}

// ---------------------------------------------------------------------------
// Density projectors of many small Fock matrices at once (the batched SCF):
// trace-correcting purification (TC2: Niklasson, Phys. Rev. B 66, 155115
// (2002)) with one workgroup per matrix, X in LDS.  X0 = (e_max - M) / (e_max
// - e_min) with Gershgorin bounds; each step forms X^2 on the FP64 matrix
// cores (X symmetric: (X^2)_ij = sum_k X_ki X_kj, both operands read along row
// k of X; wave w owns the 16 x 16 tiles w, w + 8, ...; v_mfma_f64_16x16x4f64
// step t gives lane l the k = 4 t + l / 16, its A element X[k][i0 + l % 16]
// and B element X[k][j0 + l % 16], and result register r of lane l is
// (X^2)[i0 + 4 r + l / 16][j0 + l % 16]), then keeps X^2 or 2X - X^2,
// whichever trace is nearer nocc; once tr(X - X^2) < tol one more step is
// taken.  P = (X + X^T) / 2; steps[b] = the steps taken (max_steps + 1 when
// the tolerance was never met).
//
// A batch is padded to its largest molecule: on average a third of the rows
// belong to a molecule, the rest couple to nothing.  Only the leading block up
// to the last coupled row, me rounded up to 16, is multiplied; the diagonal
// beyond it is squared element by element, which is the same arithmetic.  X^2
// stays in registers until the traces have chosen, so that X is the only
// matrix in LDS and several workgroups share a CU.  512 molecules of 7 to 61
// functions: 228 us, 338 with every row multiplied and X^2 in LDS.
#define PURIFY_W 8
#define PURIFY_MAXT ((EIGH_MAXN + 15) / 16 * ((EIGH_MAXN + 15) / 16))
__global__ void __launch_bounds__(64 * PURIFY_W) purify_small_kernel(const double* __restrict__ M,
                                                                     const int* __restrict__ nocc, int m, double tol,
                                                                     int max_steps, double* __restrict__ P,
                                                                     int* __restrict__ steps)
{
    typedef double pd4 __attribute__((ext_vector_type(4)));
    constexpr int NT = (PURIFY_MAXT + PURIFY_W - 1) / PURIFY_W;   // tiles of a wave
    extern __shared__ double sh[];
    __shared__ double red[2][2][PURIFY_W], d[EIGH_MAXN];
    __shared__ int s_me;
    const int tid = threadIdx.x, nt = 64 * PURIFY_W;
    const int wave = tid >> 6, lane = tid & 63, li = lane & 15, lq = lane >> 4;
    const size_t off = (size_t)blockIdx.x * m * m;
    if (tid == 0) s_me = 0;
    __syncthreads();
    // Gershgorin bounds (row i: M_ii -/+ sum_{j != i} |M_ij|) and the last
    // row with a coupling
    double lo = 1e300, hi = -1e300;
    int me = 0;
    for (int r = wave; r < m; r += PURIFY_W) {
        double rad = 0.0;
        for (int c = lane; c < m; c += 64) {
            const double v = M[off + (size_t)r * m + c];
            if (c == r) continue;
            rad += fabs(v);
            if (v != 0.0) me = max(me, max(r, c) + 1);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) rad += __shfl_xor(rad, o, 64);
        const double v = M[off + (size_t)r * m + r];
        lo = fmin(lo, v - rad);
        hi = fmax(hi, v + rad);
    }
    if (me) atomicMax(&s_me, me);
    if (lane == 0) {
        red[0][0][wave] = lo;
        red[0][1][wave] = hi;
    }
    __syncthreads();
    double emin = red[0][0][0], emax = red[0][1][0];
    for (int w = 1; w < PURIFY_W; ++w) {
        emin = fmin(emin, red[0][0][w]);
        emax = fmax(emax, red[0][1][w]);
    }
    me = s_me;
    const int nb = (me + 15) / 16, mp = 16 * nb, ntile = nb * nb, mx = min(m, mp);
    double* const X = sh;   // mp x mp
    const double inv = 1.0 / (emax - emin);
    for (int i = tid; i < mp * mp; i += nt) {
        const int r = i / mp, c = i - r * mp;
        X[i] = (r < m && c < m) ? ((r == c ? emax : 0.0) - M[off + (size_t)r * m + c]) * inv : 0.0;
    }
    for (int i = mx + tid; i < m; i += nt) d[i] = (emax - M[off + (size_t)i * m + i]) * inv;
    __syncthreads();
    const double nf = (double)nocc[blockIdx.x];
    int k = 0;
    bool last = false;
    for (; k < max_steps; ++k) {
        pd4 acc[NT];
        double t1 = 0.0, t2 = 0.0;
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int t = wave + PURIFY_W * u;
            if (t >= ntile) break;
            const int i0 = 16 * (t / nb), j0 = 16 * (t % nb);
            pd4 a = (pd4){0.0, 0.0, 0.0, 0.0};
            const double* pa = X + lq * mp + i0 + li;
            const double* pb = X + lq * mp + j0 + li;
#pragma unroll 4
            for (int q = 0; q < mp / 4; ++q)
                a = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[4 * q * mp], pb[4 * q * mp], a, 0, 0, 0);
            acc[u] = a;
            if (i0 == j0) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (4 * r + lq == li) {
                        t1 += X[(i0 + li) * mp + i0 + li];
                        t2 += a[r];
                    }
            }
        }
        for (int i = mx + tid; i < m; i += nt) {
            t1 += d[i];
            t2 += d[i] * d[i];
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            t1 += __shfl_xor(t1, o, 64);
            t2 += __shfl_xor(t2, o, 64);
        }
        if (lane == 0) {
            red[k & 1][0][wave] = t1;
            red[k & 1][1][wave] = t2;
        }
        __syncthreads();   // every wave has read X
        t1 = t2 = 0.0;
#pragma unroll
        for (int w = 0; w < PURIFY_W; ++w) {
            t1 += red[k & 1][0][w];
            t2 += red[k & 1][1][w];
        }
        const bool up = fabs(t2 - nf) < fabs(2.0 * t1 - t2 - nf);
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int t = wave + PURIFY_W * u;
            if (t >= ntile) break;
            const int i0 = 16 * (t / nb), j0 = 16 * (t % nb);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                double* x = X + (i0 + 4 * r + lq) * mp + j0 + li;
                *x = up ? acc[u][r] : 2.0 * *x - acc[u][r];
            }
        }
        for (int i = mx + tid; i < m; i += nt) d[i] = up ? d[i] * d[i] : 2.0 * d[i] - d[i] * d[i];
        __syncthreads();
        if (last) break;
        if (t1 - t2 < tol) last = true;
    }
    for (int i = tid; i < m * m; i += nt) {
        const int r = i / m, c = i - r * m;
        P[off + i] = r < mx && c < mx ? 0.5 * (X[r * mp + c] + X[c * mp + r]) : (r == c ? d[r] : 0.0);
    }
    if (tid == 0) steps[blockIdx.x] = last ? k + 1 : max_steps + 1;
}

extern "C" int pq_purify_batched(const double* M, const int* nocc, int batch, int m, double tol, int max_steps,
                                 double* P, int* steps, void* stream)
{
    if (!M || !nocc || !P || !steps) return pq_set_error("pq_purify_batched: null argument");
    if (batch < 0 || m < 1 || max_steps < 1) return pq_set_error("pq_purify_batched: bad sizes");
    if (m > EIGH_MAXN)
        return pq_set_error(("pq_purify_batched: m = " + std::to_string(m) + " exceeds the LDS-resident limit of " +
                             std::to_string(EIGH_MAXN)).c_str());
    if (batch == 0) return 0;
    const int mp = (m + 15) & ~15;
    const size_t lds = sizeof(double) * (size_t)mp * mp;
    static bool attr = false;
    if (!attr) {
        const int mpmax = (EIGH_MAXN + 15) & ~15;   // 96: 74 KB
        if (hipFuncSetAttribute((const void*)purify_small_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(sizeof(double) * mpmax * mpmax)) != hipSuccess)
            return pq_set_error("pq_purify_batched: cannot raise the kernel's LDS limit");
        attr = true;
    }
    hipLaunchKernelGGL(purify_small_kernel, dim3(batch), dim3(64 * PURIFY_W), lds, (hipStream_t)stream, M, nocc, m, tol,
                       max_steps, P, steps);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return pq_set_error((std::string("pq_purify_batched: ") + hipGetErrorString(e)).c_str());
    return 0;
}
