// mp2.hip -- dense contractions of the MP2 AO->MO transform on the FP64
// matrix cores, and the MP2 energy reduction.
//
// long_gemm_f64_kernel: out(m, c) = sum_k P(m, k) Q(c, k) (mp2.h) on
// v_mfma_f64_16x16x4f64.  Bound by the matrix cores once the rows fit the
// tile: an instruction of 2048 flops holds a SIMD's matrix core for 64 cycles,
// against which the operand reads from LDS ((MB + 2) 8-byte reads for 2 MB
// products) and from memory are small.  Block tile MB * 16 (m) x 128 (c), four
// waves of MB * 16 x 32, K 16 at a time through two LDS buffers with one
// barrier per step; the next step's global loads are in flight during the
// products.  MB (1..5) is the host's choice so that an orbital space fills its
// tiles (mp2.h).  Two waves a SIMD as launch bound keep the accumulators in
// vector registers (at one the compiler moved them between the two register
// files around every step).  C10H22's transform (n = 194, o = 41, v = 153): the
// second quarter 41 TFLOP/s, the third and fourth 40; 27 in 64-row tiles with
// guarded loads (large square products of this card reach 72).  What is left is
// each block's start and end around only 13 steps of K.
//
// MFMA 16x16x4 f64 operand layout (measured on gfx950): lane l supplies
// A[l%16][k0 + l/16] and B[k0 + l/16][l%16]; result register r of lane l is
// D[4*r + l/16][l%16], r = 0..3.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mp2.h"

typedef double double4_t __attribute__((ext_vector_type(4)));

#define XD_K 16
#define XD_CROW (XD_K + 2)        // LDS row of a Q tile stored [c][k]
#define XD_KROW (PQ_TC + 16)      // LDS row of a Q tile stored [k][c]

template <int MB, int PK, int QM, int SW>
__global__ void __launch_bounds__(256, 2) long_gemm_f64_kernel(const LongGemm g)
{
    constexpr int TM = MB * 16, PROW = (MB & 1) ? TM : TM + 16;   // rows k, k + 1 32 banks apart
    constexpr int QN = QM == PQ_QROW ? PQ_TC * XD_CROW : XD_K * XD_KROW;
    __shared__ double Ps[2][XD_K * PROW];
    __shared__ double Qs[2][QN];
    int m0, c0;
    if (!long_gemm_tile(g, m0, c0)) return;
    const double* __restrict__ P = g.P + blockIdx.z * g.sP;
    const double* __restrict__ Q = g.Q + blockIdx.z * g.sQ;
    double* __restrict__ C = g.C + blockIdx.z * g.sC;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int M = g.M, N = g.N, K = g.K;
    // Element t of this thread in a step of the P tile and of the Q tile.  Rows
    // past M and columns past N are read at a clamped address and give
    // results that are not stored; k past K is clamped and zeroed.
    auto p_m = [&](int t) { return PK ? (tid + 256 * t) % TM : (tid + 256 * t) >> 4; };
    auto p_k = [&](int t) { return PK ? (tid + 256 * t) / TM : tid & 15; };
    auto q_c = [&](int t) { return QM == PQ_QROW ? (tid >> 4) + 16 * t : tid & 127; };
    auto q_k = [&](int t) { return QM == PQ_QROW ? tid & 15 : (tid >> 7) + 2 * t; };
    const int cc = min(c0 + (tid & 127), N - 1);
    // Whole steps advance one pointer per element (or one for all, plus a
    // uniform distance): FP64 matrix instructions and vector instructions do
    // not overlap on a SIMD, so index arithmetic is taken from the products.
    const double* pp[MB];
    const double* qp[QM == PQ_QROW ? 8 : 1];
    const int* tp = nullptr;
#pragma unroll
    for (int t = 0; t < MB; ++t) {
        const long long gm = min(m0 + p_m(t), M - 1);
        pp[t] = PK ? P + (long long)p_k(t) * g.ldp + gm : P + gm * g.ldp + p_k(t);
    }
    if (QM == PQ_QROW) {
#pragma unroll
        for (int t = 0; t < (QM == PQ_QROW ? 8 : 1); ++t) qp[t] = Q + (long long)min(c0 + q_c(t), N - 1) * g.ldq + (tid & 15);
    } else if (QM == PQ_QK) {
        qp[0] = Q + (long long)(tid >> 7) * g.ldq + cc;
    } else {
        const int gi = cc / g.cn;
        qp[0] = Q + (long long)gi * g.ldq;
        tp = g.tab + (cc - gi * g.cn) + (tid >> 7) * g.cn;
    }
    double rp[MB], rq[8];
    unsigned id[8];
    // packed indices of the step at k0 (the table has two steps of rows past K)
    auto load_tab = [&](int k0) {
#pragma unroll
        for (int t = 0; t < 8; ++t) id[t] = tp[(long long)(k0 + 2 * t) * g.cn];
    };
    // a whole step, and the last, partial one
    auto load = [&](int k0) {
#pragma unroll
        for (int t = 0; t < MB; ++t) {
            rp[t] = *pp[t];
            pp[t] += PK ? XD_K * g.ldp : (long long)XD_K;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            if (QM == PQ_QROW) {
                rq[t] = *qp[t];
                qp[t] += XD_K;
            } else if (QM == PQ_QK) {
                rq[t] = qp[0][(long long)(k0 + 2 * t) * g.ldq];
            } else {
                rq[t] = qp[0][id[t]];
            }
        }
        if (QM == PQ_QSYM) load_tab(k0 + XD_K);
    };
    auto load_tail = [&](int k0) {
#pragma unroll
        for (int t = 0; t < MB; ++t) {
            const long long back = max(k0 + p_k(t) - (K - 1), 0);
            rp[t] = *(pp[t] - back * (PK ? g.ldp : 1LL));
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const long long back = max(k0 + q_k(t) - (K - 1), 0);
            if (QM == PQ_QROW) rq[t] = *(qp[t] - back);
            else if (QM == PQ_QK) rq[t] = qp[0][(k0 + 2 * t - back) * g.ldq];
            else rq[t] = qp[0][id[t]];
        }
        const int left = K - k0;
#pragma unroll
        for (int t = 0; t < MB; ++t) rp[t] = p_k(t) < left ? rp[t] : 0.0;
#pragma unroll
        for (int t = 0; t < 8; ++t) rq[t] = q_k(t) < left ? rq[t] : 0.0;
    };
    auto stage = [&](int b) {
#pragma unroll
        for (int t = 0; t < MB; ++t) Ps[b][p_k(t) * PROW + p_m(t)] = rp[t];
#pragma unroll
        for (int t = 0; t < 8; ++t) Qs[b][QM == PQ_QROW ? q_c(t) * XD_CROW + q_k(t) : q_k(t) * XD_KROW + q_c(t)] = rq[t];
    };
    double4_t acc[MB][2];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (double4_t){0.0, 0.0, 0.0, 0.0};
    double p[2][MB], q[2][2];
    auto read = [&](int kk, int b, int s) {
        const int kr = kk + (lane >> 4);
#pragma unroll
        for (int i = 0; i < MB; ++i) p[s][i] = Ps[b][kr * PROW + i * 16 + (lane & 15)];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int c = wave * 32 + j * 16 + (lane & 15);
            q[s][j] = QM == PQ_QROW ? Qs[b][c * XD_CROW + kr] : Qs[b][kr * XD_KROW + c];
        }
    };
    auto multiply = [&](int s) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[i][j] = SW ? __builtin_amdgcn_mfma_f64_16x16x4f64(q[s][j], p[s][i], acc[i][j], 0, 0, 0)
                               : __builtin_amdgcn_mfma_f64_16x16x4f64(p[s][i], q[s][j], acc[i][j], 0, 0, 0);
    };
    // the operands of the next four k are read from LDS ahead of the current
    // ones' products
    auto products = [&](int b) {
        read(0, b, 0);
#pragma unroll
        for (int u = 0; u < XD_K / 4; ++u) {
            if (u + 1 < XD_K / 4) read(4 * (u + 1), b, (u + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(u & 1);
        }
    };
    if (QM == PQ_QSYM) load_tab(0);
    if (XD_K <= K) load(0);
    else load_tail(0);
    stage(0);
    __syncthreads();
    // the main loop has no branches (around its accumulators they cost a copy
    // each way)
    int k0 = 0, b = 0;
    for (; k0 + 2 * XD_K <= K; k0 += XD_K, b ^= 1) {
        load(k0 + XD_K);
        products(b);
        stage(b ^ 1);
        __syncthreads();
    }
    if (k0 + XD_K < K) {
        load_tail(k0 + XD_K);
        products(b);
        stage(b ^ 1);
        __syncthreads();
        k0 += XD_K;
        b ^= 1;
    }
    for (int kk = 0; kk < K - k0; kk += 4) {
        read(kk, b, 0);
        multiply(0);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int cb = c0 + wave * 32 + j * 16;
        if (SW) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int c = cb + 4 * r + (lane >> 4), m = m0 + i * 16 + (lane & 15);
                    if (m < M && c < N) {
                        double* dst = &C[(long long)c * g.ldc + m];
                        const double v = g.alpha * acc[i][j][r];
                        *dst = g.beta == 0.0 ? v : v + g.beta * *dst;
                    }
                }
        } else {
            const int c = cb + (lane & 15);
            const long long off = QM == PQ_QSYM ? (long long)(c / g.cn) * g.s1 + c % g.cn : c;
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = m0 + i * 16 + 4 * r + (lane >> 4);
                    if (m < M && c < N) {
                        double* dst = &C[m * g.ldc + off];
                        const double v = g.alpha * acc[i][j][r];
                        *dst = g.beta == 0.0 ? v : v + g.beta * *dst;
                    }
                }
        }
    }
}

int long_gemm_f64(LongGemm g, int batch, hipStream_t st) { LONG_GEMM_LAUNCH(long_gemm_f64_kernel) }

// MP2 energy over (ia|jb) stored [o1][v1][o2][v2]:
//   mode 0 (closed shell): sum v (2 v - (ib|ja)) / D          (o1 = o2, v1 = v2)
//   mode 1 (same spin):    1/4 sum [(ia|jb) - (ib|ja)]^2 / D  (Methods/mp2.py:77-88, i>=j, p>=q)
//   mode 2 (opposite spin): sum (ia|jb)^2 / D                 (Methods/mp2.py:90-94)
// D = e_i + e_j - e_a - e_b.  Bound by memory: a block strides over 32 x 32
// (a, b) tiles of the (i, j) pairs, (ib|ja) read as the transposed tile
// through LDS (C10H22: 146 us for 0.63 GB; read element by element across
// rows 532 us).  One atomic per block.
#define ME_T 32
#define ME_BLOCKS 2048
__global__ void __launch_bounds__(256) mp2_energy_kernel(const double* __restrict__ ovov, const double* __restrict__ eo1,
                                                          const double* __restrict__ ev1, const double* __restrict__ eo2,
                                                          const double* __restrict__ ev2, int o1, int v1, int o2, int v2,
                                                          int mode, double* out)
{
    __shared__ double xt[ME_T][ME_T + 1];
    __shared__ double red[4];
    const int ta = (v1 + ME_T - 1) / ME_T, tb = (v2 + ME_T - 1) / ME_T;
    const long long tiles = (long long)o1 * o2 * ta * tb;
    const int lx = threadIdx.x & 31, ly = threadIdx.x >> 5;
    double s = 0.0;
    for (long long t = blockIdx.x; t < tiles; t += gridDim.x) {
        const int b0 = (int)(t % tb) * ME_T;
        long long r = t / tb;
        const int a0 = (int)(r % ta) * ME_T;
        r /= ta;
        const int j = (int)(r % o2), i = (int)(r / o2);
        double v[ME_T / 8];
#pragma unroll
        for (int u = 0; u < ME_T / 8; ++u) {
            const int a = a0 + ly + 8 * u, b = b0 + lx;
            v[u] = (a < v1 && b < v2) ? ovov[(((long long)i * v1 + a) * o2 + j) * v2 + b] : 0.0;
        }
        if (mode != 2) {
#pragma unroll
            for (int u = 0; u < ME_T / 8; ++u) {   // (ib|ja), b along the tile's rows
                const int b = b0 + ly + 8 * u, a = a0 + lx;
                xt[ly + 8 * u][lx] = (a < v1 && b < v2) ? ovov[(((long long)i * v1 + b) * o2 + j) * v2 + a] : 0.0;
            }
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < ME_T / 8; ++u) {
            const int a = a0 + ly + 8 * u, b = b0 + lx;
            if (a < v1 && b < v2) {
                const double den = eo1[i] + eo2[j] - ev1[a] - ev2[b];
                if (mode == 2) {
                    s += v[u] * v[u] / den;
                } else {
                    const double x = xt[lx][ly + 8 * u];
                    s += mode == 0 ? v[u] * (2.0 * v[u] - x) / den : 0.25 * (v[u] - x) * (v[u] - x) / den;
                }
            }
        }
        if (mode != 2) __syncthreads();
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) unsafeAtomicAdd(out, (red[0] + red[1]) + (red[2] + red[3]));
}

int mp2_energy_launch(const double* ovov, const double* eo1, const double* ev1, const double* eo2, const double* ev2,
                      int o1, int v1, int o2, int v2, int mode, double* out, hipStream_t st)
{
    const long long tiles = (long long)o1 * o2 * ((v1 + ME_T - 1) / ME_T) * ((v2 + ME_T - 1) / ME_T);
    const long long blocks = tiles > ME_BLOCKS ? ME_BLOCKS : (tiles < 1 ? 1 : tiles);
    hipLaunchKernelGGL(mp2_energy_kernel, dim3((unsigned)blocks), dim3(256), 0, st, ovov, eo1, ev1, eo2, ev2, o1, v1, o2,
                       v2, mode, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
