// scf_batch.hip -- the batched SCF's work between its matrix products, one
// workgroup per molecule.  A cycle over 512 small molecules (26 functions on
// average, 11 MB a matrix) spent 0.8 ms in its J/K build and 1.9 ms in some 75
// elementwise, reduction and solver launches of 2 to 10 us each behind gaps of
// 10 to 30 us: packing and unpacking, the convergence test, the DIIS Gram
// products, bordered systems and combinations, the spectrum's shift.  Each of
// these five is one launch here, bound by a pass over the matrices it reads.
//
// Matrices are [batch][m][m], molecule b's in the leading n[b] x n[b] corner,
// zero outside; packed arrays hold the n[b] x n[b] blocks from base[b] on.
#include <hip/hip_runtime.h>
#include <string>

#include "scf.h"

#define SB_THREADS 256
#define SB_DOTS 8      // Gram products per pass over the matrices
#define SB_LDS_K 64    // largest DIIS space whose bordered system is kept in LDS

// maximum that keeps a NaN
__device__ __forceinline__ double max_nan(double a, double b) { return (a > b || a != a) ? a : b; }

template <bool MAX>
__device__ __forceinline__ double block_reduce(double v, double* part)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const double u = __shfl_xor(v, o, 64);
        v = MAX ? max_nan(v, u) : v + u;
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = part[0];
#pragma unroll
    for (int w = 1; w < SB_THREADS / 64; ++w) v = MAX ? max_nan(v, part[w]) : v + part[w];
    return v;
}

// D <- Dn where not done (Dn may be NULL); Dj = 2 D, Dk = D packed.
__global__ void __launch_bounds__(SB_THREADS) batch_pack_kernel(int m, const long long* __restrict__ base,
                                                                const long long* __restrict__ n, double* D,
                                                                const double* Dn, const unsigned char* done,
                                                                double* __restrict__ Dj, double* __restrict__ Dk)
{
    const int b = blockIdx.x, nb = (int)n[b];
    const bool take = Dn && !done[b];
    const size_t off = (size_t)b * m * m;
    for (int e = threadIdx.x; e < m * m; e += SB_THREADS) {
        const int i = e / m, j = e - i * m;
        double d;
        if (take) {
            d = Dn[off + e];
            D[off + e] = d;
        } else {
            d = D[off + e];
        }
        if (i < nb && j < nb) {
            const long long p = base[b] + (long long)i * nb + j;
            Dj[p] = 2.0 * d;
            Dk[p] = d;
        }
    }
}

// F = H + J + K, J and K packed.
__global__ void __launch_bounds__(SB_THREADS) batch_fock_kernel(int m, const long long* __restrict__ base,
                                                                const long long* __restrict__ n,
                                                                const double* __restrict__ H,
                                                                const double* __restrict__ J,
                                                                const double* __restrict__ K, double* __restrict__ F)
{
    const int b = blockIdx.x, nb = (int)n[b];
    const size_t off = (size_t)b * m * m;
    for (int e = threadIdx.x; e < m * m; e += SB_THREADS) {
        const int i = e / m, j = e - i * m;
        double f = H[off + e];
        if (i < nb && j < nb) {
            const long long p = base[b] + (long long)i * nb + j;
            f = f + J[p] + K[p];
        }
        F[off + e] = f;
    }
}

// Energy sum D (H + F) + enuc and largest residual of each molecule; one that
// is not done takes them, and is done from here when its energy moved by less
// than conv and the residual is at most rtol.  flags: [0] any newly done, [1]
// molecules not done.
__global__ void __launch_bounds__(SB_THREADS) batch_test_kernel(int m, const long long* __restrict__ n,
                                                                const double* __restrict__ D,
                                                                const double* __restrict__ H,
                                                                const double* __restrict__ F,
                                                                const double* __restrict__ R, const double* enuc,
                                                                double conv, double rtol, int it, double* E,
                                                                long long* iters, unsigned char* done,
                                                                unsigned char* newly, int* flags)
{
    __shared__ double part[SB_THREADS / 64];
    const int b = blockIdx.x, nb = (int)n[b];
    const size_t off = (size_t)b * m * m;
    double ev = 0.0, rm = 0.0;
    for (int e = threadIdx.x; e < m * m; e += SB_THREADS) {
        const int i = e / m, j = e - i * m;
        if (i < nb && j < nb) ev += D[off + e] * (H[off + e] + F[off + e]);
        rm = max_nan(rm, fabs(R[off + e]));
    }
    ev = block_reduce<false>(ev, part);
    rm = block_reduce<true>(rm, part);
    if (threadIdx.x) return;
    ev += enuc[b];
    const bool was = done[b];
    const bool nw = !was && fabs(ev - E[b]) < conv && rm <= rtol && it > 1;
    if (!was) {
        E[b] = ev;
        iters[b] = it;
    }
    newly[b] = nw;
    done[b] = was || nw;
    if (nw) atomicOr(&flags[0], 1);
    if (!was && !nw) atomicAdd(&flags[1], 1);
}

// Slot `newest` of the ring of S takes F and R; row and column of the Gram
// matrix; the bordered system of the last k slots, oldest first,
//   (G + ridge) c - 1 lambda = 0, -sum c = -1, ridge = 1e-14 mean(diag) + 1e-300,
// by Gaussian elimination with partial pivoting; Fx = sum c F.  One pass
// over the residuals for up to SB_DOTS products, one over the Fock matrices.
// flags[2] counts singular systems (a zero pivot).
__global__ void __launch_bounds__(SB_THREADS) batch_diis_kernel(int mm, const double* __restrict__ F,
                                                                const double* __restrict__ R, double* Fbuf,
                                                                double* Rbuf, double* G, int S, int newest, int k,
                                                                double* __restrict__ Fx, double* work, int* flags)
{
    extern __shared__ double lds[];
    __shared__ double part[SB_THREADS / 64];
    const int b = blockIdx.x, tid = threadIdx.x;
    const double* const f = F + (size_t)b * mm;
    const double* const r = R + (size_t)b * mm;
    double* const fb = Fbuf + (size_t)b * S * mm;
    double* const rb = Rbuf + (size_t)b * S * mm;
    double* const g = G + (size_t)b * S * S;
    auto slot = [&](int j) { return (newest - (k - 1) + j + 2 * S) % S; };   // j = 0 oldest ... k - 1 newest
    for (int j0 = 0; j0 < k; j0 += SB_DOTS) {
        const double* p[SB_DOTS];
        double acc[SB_DOTS];
#pragma unroll
        for (int u = 0; u < SB_DOTS; ++u) {
            const int j = min(j0 + u, k - 1);
            p[u] = j == k - 1 ? r : rb + (size_t)slot(j) * mm;
            acc[u] = 0.0;
        }
        for (int e = tid; e < mm; e += SB_THREADS) {
            const double x = r[e];
#pragma unroll
            for (int u = 0; u < SB_DOTS; ++u) acc[u] += x * p[u][e];
            if (j0 == 0) {
                rb[(size_t)newest * mm + e] = x;
                fb[(size_t)newest * mm + e] = f[e];
            }
        }
#pragma unroll
        for (int u = 0; u < SB_DOTS; ++u) {
            if (j0 + u >= k) break;
            const double d = block_reduce<false>(acc[u], part);
            if (tid == 0) {
                const int s = slot(j0 + u);
                g[newest * S + s] = d;
                g[s * S + newest] = d;
            }
        }
    }
    if (k < 2) {
        for (int e = tid; e < mm; e += SB_THREADS) Fx[(size_t)b * mm + e] = f[e];
        return;
    }
    const int q = k + 1, w = q + 1;   // unknowns; row length with the right-hand side
    double* const A = q <= SB_LDS_K + 1 ? lds : work + (size_t)b * q * w;
    __threadfence_block();
    __syncthreads();
    double mean = 0.0;
    for (int j = 0; j < k; ++j) mean += g[slot(j) * S + slot(j)];
    const double ridge = 1e-14 * (mean / k) + 1e-300;
    for (int e = tid; e < q * w; e += SB_THREADS) {
        const int i = e / w, j = e - i * w;
        double v;
        if (i < k && j < k) v = g[slot(i) * S + slot(j)] + (i == j ? ridge : 0.0);
        else if (i == k) v = j < k || j == q ? -1.0 : 0.0;   // -sum c = -1
        else v = j == k ? -1.0 : 0.0;
        A[e] = v;
    }
    __syncthreads();
    for (int p = 0; p < q; ++p) {
        int piv = p;
        double best = fabs(A[p * w + p]);
        for (int i = p + 1; i < q; ++i) {
            const double v = fabs(A[i * w + p]);
            if (v > best) { best = v; piv = i; }
        }
        __syncthreads();
        if (best == 0.0 && tid == 0) atomicAdd(&flags[2], 1);
        if (piv != p)
            for (int j = tid; j < w; j += SB_THREADS) {
                const double v = A[p * w + j];
                A[p * w + j] = A[piv * w + j];
                A[piv * w + j] = v;
            }
        __syncthreads();
        const double inv = 1.0 / A[p * w + p];
        const int cols = w - (p + 1);
        for (int e = tid; e < (q - p - 1) * cols; e += SB_THREADS) {
            const int i = p + 1 + e / cols, j = p + 1 + e % cols;
            A[i * w + j] -= (A[i * w + p] * inv) * A[p * w + j];
        }
        __syncthreads();
    }
    if (tid == 0)
        for (int i = q - 1; i >= 0; --i) {
            double v = A[i * w + q];
            for (int j = i + 1; j < q; ++j) v -= A[i * w + j] * A[j * w + q];
            A[i * w + q] = v / A[i * w + i];
        }
    __threadfence_block();
    __syncthreads();
    for (int e = tid; e < mm; e += SB_THREADS) {
        double x = 0.0;
        for (int j = 0; j < k; ++j) x += A[j * w + q] * (j == k - 1 ? f[e] : fb[(size_t)slot(j) * mm + e]);
        Fx[(size_t)b * mm + e] = x;
    }
}

// M += diag(dropped (max(0, max_i (M_ii + sum_{j != i} |M_ij|)) + 1)): the
// dropped columns' states above the rest of the spectrum (Gershgorin).
__global__ void __launch_bounds__(SB_THREADS) batch_lift_kernel(int m, double* M, const double* __restrict__ dropped)
{
    __shared__ double part[SB_THREADS / 64];
    const int b = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double* const a = M + (size_t)b * m * m;
    double top = 0.0;
    for (int i = wave; i < m; i += SB_THREADS / 64) {
        double s = 0.0;
        for (int j = lane; j < m; j += 64) s += fabs(a[(size_t)i * m + j]);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
        const double d = a[(size_t)i * m + i];
        top = max_nan(top, d + s - fabs(d));
    }
    top = block_reduce<true>(top, part) + 1.0;
    for (int i = threadIdx.x; i < m; i += SB_THREADS) a[(size_t)i * m + i] += dropped[(size_t)b * m + i] * top;
}

namespace {
int done_launch(const char* who)
{
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : pq_set_error((std::string(who) + ": " + hipGetErrorString(e)).c_str());
}
}  // namespace

extern "C" int pq_batch_pack(int batch, int m, const long long* base, const long long* n, double* D, const double* Dn,
                             const unsigned char* done, double* Dj, double* Dk, void* stream)
{
    if (batch < 0 || m < 1 || m > 30000) return pq_set_error("pq_batch_pack: need batch >= 0 and 1 <= m <= 30000");
    if (!base || !n || !D || !Dj || !Dk || (Dn && !done)) return pq_set_error("pq_batch_pack: null argument");
    if (batch == 0) return 0;
    hipLaunchKernelGGL(batch_pack_kernel, dim3(batch), dim3(SB_THREADS), 0, (hipStream_t)stream, m, base, n, D, Dn, done,
                       Dj, Dk);
    return done_launch("pq_batch_pack");
}

extern "C" int pq_batch_fock(int batch, int m, const long long* base, const long long* n, const double* H,
                             const double* J, const double* K, double* F, void* stream)
{
    if (batch < 0 || m < 1 || m > 30000) return pq_set_error("pq_batch_fock: need batch >= 0 and 1 <= m <= 30000");
    if (!base || !n || !H || !J || !K || !F) return pq_set_error("pq_batch_fock: null argument");
    if (batch == 0) return 0;
    hipLaunchKernelGGL(batch_fock_kernel, dim3(batch), dim3(SB_THREADS), 0, (hipStream_t)stream, m, base, n, H, J, K, F);
    return done_launch("pq_batch_fock");
}

extern "C" int pq_batch_test(int batch, int m, const long long* n, const double* D, const double* H, const double* F,
                             const double* R, const double* enuc, double conv, double rtol, int it, double* E,
                             long long* iters, unsigned char* done, unsigned char* newly, int* flags, void* stream)
{
    if (batch < 0 || m < 1 || m > 30000) return pq_set_error("pq_batch_test: need batch >= 0 and 1 <= m <= 30000");
    if (!n || !D || !H || !F || !R || !enuc || !E || !iters || !done || !newly || !flags)
        return pq_set_error("pq_batch_test: null argument");
    if (batch == 0) return 0;
    hipLaunchKernelGGL(batch_test_kernel, dim3(batch), dim3(SB_THREADS), 0, (hipStream_t)stream, m, n, D, H, F, R, enuc,
                       conv, rtol, it, E, iters, done, newly, flags);
    return done_launch("pq_batch_test");
}

extern "C" long long pq_batch_diis_work(int batch, int k)
{
    return k <= SB_LDS_K ? 0 : (long long)batch * (k + 1) * (k + 2);
}

extern "C" int pq_batch_diis(int batch, int m, const double* F, const double* R, double* Fbuf, double* Rbuf, double* G,
                             int slots, int newest, int k, double* Fx, double* work, int* flags, void* stream)
{
    if (batch < 0 || m < 1 || m > 30000) return pq_set_error("pq_batch_diis: need batch >= 0 and 1 <= m <= 30000");
    if (slots < 1 || slots > 10000 || newest < 0 || newest >= slots || k < 1 || k > slots)
        return pq_set_error("pq_batch_diis: need 0 <= newest < slots and 1 <= k <= slots <= 10000");
    if (!F || !R || !Fbuf || !Rbuf || !G || !Fx || !flags || (k > SB_LDS_K && !work))
        return pq_set_error("pq_batch_diis: null argument");
    if (batch == 0) return 0;
    const size_t lds = k >= 2 && k <= SB_LDS_K ? sizeof(double) * (size_t)(k + 1) * (k + 2) : 0;
    hipLaunchKernelGGL(batch_diis_kernel, dim3(batch), dim3(SB_THREADS), lds, (hipStream_t)stream, m * m, F, R, Fbuf,
                       Rbuf, G, slots, newest, k, Fx, work, flags);
    return done_launch("pq_batch_diis");
}

extern "C" int pq_batch_lift(int batch, int m, double* M, const double* dropped, void* stream)
{
    if (batch < 0 || m < 1 || m > 30000) return pq_set_error("pq_batch_lift: need batch >= 0 and 1 <= m <= 30000");
    if (!M || !dropped) return pq_set_error("pq_batch_lift: null argument");
    if (batch == 0) return 0;
    hipLaunchKernelGGL(batch_lift_kernel, dim3(batch), dim3(SB_THREADS), 0, (hipStream_t)stream, m, M, dropped);
    return done_launch("pq_batch_lift");
}
