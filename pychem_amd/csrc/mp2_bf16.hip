// mp2_bf16.hip -- the products of mp2.h with FP32-accumulated split-BF16
// matrix-core products.  Each FP64 operand element x is split into
// hi = bf16(x) and lo = bf16(fp32(x) - hi); a*b is taken as hi_a hi_b +
// hi_a lo_b + lo_a hi_b (the lo_a lo_b term, ~2^-16 relative, is dropped) on
// v_mfma_f32_16x16x32_bf16, accumulated in FP32 and written as FP64.  The
// matrix cores finish a step of K = 32 in a tenth of the FP64 time, so the
// kernel is bound by the FP64 operands' loads and their conversion: block tile
// MB * 16 (m) x 128 (c), four waves of MB * 16 x 32, one LDS buffer (33 KB at
// most, four blocks a CU) with the next step's loads in flight during the
// products.
//
// The MFMA layout (measured on gfx950): lane l supplies A[l%16][8*(l/16) + i]
// and B[8*(l/16) + i][l%16], i = 0..7; result register r of lane l is
// D[4*(l/16) + r][l%16] (rows in the other order from the FP64 16x16x4
// instruction's D[4*r + l/16][l%16]).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mp2.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

#define XB_K 32
#define XB_LD 40   // LDS row stride in bf16 (80 bytes: 16-byte aligned fragments)

// hi is x rounded once, from 64 bits to BF16.  Through FP32 that is the same
// except where the FP32 value lies halfway between two BF16 values and x does
// not: there (one value in 2^16) x decides, by a step of the FP32 value off
// the tie.  The direct conversion costs eight more instructions per element.
__device__ __forceinline__ void split_bf16(double x, __bf16& hi, __bf16& lo)
{
    const float f = (float)x;
    float t = f;
    if (__builtin_expect((__float_as_uint(f) & 0xffffu) == 0x8000u, 0)) {
        const double d = (double)f;
        if (fabs(x) > fabs(d)) t = __uint_as_float(__float_as_uint(f) + 1u);
        if (fabs(x) < fabs(d)) t = __uint_as_float(__float_as_uint(f) - 1u);
    }
    hi = (__bf16)t;
    lo = (__bf16)(f - (float)hi);
}

template <int MB, int PK, int QM, int SW>
__global__ void __launch_bounds__(256, 2) long_gemm_bf16x3_kernel(const LongGemm g)
{
    constexpr int TM = MB * 16;
    __shared__ __attribute__((aligned(16))) __bf16 Ph[TM * XB_LD], Pl[TM * XB_LD];
    __shared__ __attribute__((aligned(16))) __bf16 Qh[PQ_TC * XB_LD], Ql[PQ_TC * XB_LD];
    int m0, c0;
    if (!long_gemm_tile(g, m0, c0)) return;
    const double* __restrict__ P = g.P + blockIdx.z * g.sP;
    const double* __restrict__ Q = g.Q + blockIdx.z * g.sQ;
    double* __restrict__ C = g.C + blockIdx.z * g.sC;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int M = g.M, N = g.N, K = g.K;
    double rp[2 * MB], rq[16];
    int id[16];
    const int cc = min(c0 + (tid & 127), N - 1);
    const int* __restrict__ tab = g.tab;
    if (QM == PQ_QSYM) {
        const int gi = cc / g.cn;
        Q += (long long)gi * g.ldq;
        tab += cc - gi * g.cn;
    }
    // lanes along c take pairs of k: element t is k = 2 (tid / 128 + 2 (t / 2)) + t % 2
    auto k_of = [&](int t) { return 2 * ((tid >> 7) + 2 * (t >> 1)) + (t & 1); };
    auto load_tab = [&](int k0) {
#pragma unroll
        for (int t = 0; t < 16; ++t) id[t] = tab[(long long)min(k0 + k_of(t), K - 1) * g.cn];
    };
    auto load = [&](int k0) {
#pragma unroll
        for (int t = 0; t < 2 * MB; ++t) {
            const int e = tid + 256 * t;
            const int mm = PK ? e % TM : e >> 5, kk = PK ? e / TM : e & 31;
            const long long gm = min(m0 + mm, M - 1), gk = min(k0 + kk, K - 1);
            rp[t] = PK ? P[gk * g.ldp + gm] : P[gm * g.ldp + gk];
        }
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            if (QM == PQ_QROW) {
                const long long gc = min(c0 + (tid >> 5) + 8 * t, N - 1), gk = min(k0 + (tid & 31), K - 1);
                rq[t] = Q[gc * g.ldq + gk];
            } else if (QM == PQ_QK) {
                rq[t] = Q[(long long)min(k0 + k_of(t), K - 1) * g.ldq + cc];
            } else {
                rq[t] = Q[id[t]];
            }
        }
        if (QM == PQ_QSYM) load_tab(k0 + XB_K);
    };
    auto stage = [&](int k0) {
        const int left = K - k0;
#pragma unroll
        for (int t = 0; t < 2 * MB; ++t) {
            const int e = tid + 256 * t;
            const int mm = PK ? e % TM : e >> 5, kk = PK ? e / TM : e & 31;
            split_bf16(kk < left ? rp[t] : 0.0, Ph[mm * XB_LD + kk], Pl[mm * XB_LD + kk]);
        }
        if (QM == PQ_QROW) {
            const int kk = tid & 31;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int at = ((tid >> 5) + 8 * t) * XB_LD + kk;
                split_bf16(kk < left ? rq[t] : 0.0, Qh[at], Ql[at]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < 16; t += 2) {
                const int kk = k_of(t), at = (tid & 127) * XB_LD + kk;
                __bf16 h0, l0, h1, l1;
                split_bf16(kk < left ? rq[t] : 0.0, h0, l0);
                split_bf16(kk + 1 < left ? rq[t + 1] : 0.0, h1, l1);
                *(bf16x2_t*)&Qh[at] = (bf16x2_t){h0, h1};
                *(bf16x2_t*)&Ql[at] = (bf16x2_t){l0, l1};
            }
        }
    };
    floatx4_t acc[MB][2];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
    if (QM == PQ_QSYM) load_tab(0);
    load(0);
    for (int k0 = 0; k0 < K; k0 += XB_K) {
        stage(k0);
        __syncthreads();
        if (k0 + XB_K < K) load(k0 + XB_K);
        const int fr = lane & 15, fk = 8 * (lane >> 4);
        bf16x8_t qh[2], ql[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            qh[j] = *(const bf16x8_t*)&Qh[(wave * 32 + j * 16 + fr) * XB_LD + fk];
            ql[j] = *(const bf16x8_t*)&Ql[(wave * 32 + j * 16 + fr) * XB_LD + fk];
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const bf16x8_t ph = *(const bf16x8_t*)&Ph[(i * 16 + fr) * XB_LD + fk];
            const bf16x8_t pl = *(const bf16x8_t*)&Pl[(i * 16 + fr) * XB_LD + fk];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                // first operand's lo * hi, hi * lo, hi * hi
                const bf16x8_t ah = SW ? qh[j] : ph, al = SW ? ql[j] : pl, bh = SW ? ph : qh[j], bl = SW ? pl : ql[j];
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int cb = c0 + wave * 32 + j * 16;
        if (SW) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int c = cb + 4 * (lane >> 4) + r, m = m0 + i * 16 + (lane & 15);
                    if (m < M && c < N) {
                        double* dst = &C[(long long)c * g.ldc + m];
                        const double v = g.alpha * (double)acc[i][j][r];
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
                    const int m = m0 + i * 16 + 4 * (lane >> 4) + r;
                    if (m < M && c < N) {
                        double* dst = &C[m * g.ldc + off];
                        const double v = g.alpha * (double)acc[i][j][r];
                        *dst = g.beta == 0.0 ? v : v + g.beta * *dst;
                    }
                }
        }
    }
}

int long_gemm_bf16x3(LongGemm g, int batch, hipStream_t st) { LONG_GEMM_LAUNCH(long_gemm_bf16x3_kernel) }
