// mlp.hip -- training and inference kernels of the learned SCF guess (a
// small multilayer perceptron, FP32).
//
//   forward   Z = X W + b, A = act(Z)             (act: 0 identity, 1 tanh)
//   backward  dZ = dA * act'(Z); dX = dZ W^T; dW = X^T dZ; db = sum_rows dZ
//   loss      masked mean-squared error and its gradient
//   optimiser Adam
//
// Shapes: X [B x I], W [I x O] (row-major), b [O], Z/A/dA/dZ [B x O].  The
// products run on the FP32 matrix cores.  A whole network (hidden layers
// tanh, last layer linear) goes through three kernels: net_fwd_kernel (every
// layer of a 16-row strip), net_bwd_kernel (its dZ chain) and dw_kernel (all
// layers' weight and bias gradients); mm_kernel is the single-layer product
// and the path of layers too wide for a strip in LDS.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "mlp.h"

// C[M x N] = op(A) op(B) with op(A)(m,k) = ta ? A[k*M+m] : A[m*K+k],
// op(B)(k,n) = tb ? B[n*K+k] : B[k*N+n]; optional epilogue bias + activation.
// A 256-thread block computes a 32 x 32 tile, each of its four waves one
// 16 x 16 quarter on the matrix cores (v_mfma_f32_16x16x4f32: lane l
// supplies A[l%16][l/16] and B[l/16][l%16] of a 16 x 4 by 4 x 16 step and
// holds D[4(l/16)+r][l%16] in result register r).  K advances 16 at a time
// through LDS, the operand tiles staged with bounds checks (zero fill), so
// any M, N, K work.
#define MT 32
#define KC 16
typedef float mlp_f4 __attribute__((ext_vector_type(4)));

template <bool TA, bool TB>
__global__ void __launch_bounds__(256) mm_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                 const float* __restrict__ bias, float* __restrict__ Z,
                                                 float* __restrict__ Act, int M, int N, int K, int act)
{
    __shared__ float As[MT][KC + 1];   // [m][k]
    __shared__ float Bs[KC][MT + 1];   // [k][n]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bm = blockIdx.y * MT, bn = blockIdx.x * MT;
    const int wm = (wave >> 1) * 16, wn = (wave & 1) * 16;
    mlp_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int k0 = 0; k0 < K; k0 += KC) {
        // 512 elements of each operand tile, two per thread
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = tid + 256 * h;
            {   // A: e -> (m, k), k fastest for the row-major operand, m fastest when transposed
                const int mi = TA ? e % MT : e / KC, ki = TA ? e / MT : e % KC;
                const int m = bm + mi, k = k0 + ki;
                float v = 0.0f;
                if (m < M && k < K) v = TA ? A[(long long)k * M + m] : A[(long long)m * K + k];
                As[mi][ki] = v;
            }
            {   // B: e -> (k, n), n fastest unless transposed
                const int ki = TB ? e % KC : e / MT, ni = TB ? e / KC : e % MT;
                const int k = k0 + ki, n = bn + ni;
                float v = 0.0f;
                if (k < K && n < N) v = TB ? B[(long long)n * K + k] : B[(long long)k * N + n];
                Bs[ki][ni] = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < KC; kk += 4) {
            const float a = As[wm + (lane & 15)][kk + (lane >> 4)];
            const float b = Bs[kk + (lane >> 4)][wn + (lane & 15)];
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = bm + wm + 4 * (lane >> 4) + r, n = bn + wn + (lane & 15);
        if (m < M && n < N) {
            float v = acc[r];
            if (bias) v += bias[n];
            if (Z) Z[(long long)m * N + n] = v;
            if (Act) Act[(long long)m * N + n] = act == 1 ? tanhf(v) : v;
        }
    }
}

static void mm(bool ta, bool tb, const float* A, const float* B, const float* bias, float* Z, float* Act, int M,
               int N, int K, int act, hipStream_t st)
{
    dim3 grid((N + MT - 1) / MT, (M + MT - 1) / MT), block(256);
    if (ta && tb) hipLaunchKernelGGL((mm_kernel<true, true>), grid, block, 0, st, A, B, bias, Z, Act, M, N, K, act);
    else if (ta) hipLaunchKernelGGL((mm_kernel<true, false>), grid, block, 0, st, A, B, bias, Z, Act, M, N, K, act);
    else if (tb) hipLaunchKernelGGL((mm_kernel<false, true>), grid, block, 0, st, A, B, bias, Z, Act, M, N, K, act);
    else hipLaunchKernelGGL((mm_kernel<false, false>), grid, block, 0, st, A, B, bias, Z, Act, M, N, K, act);
}

// dZ = dA * act'(Z) with tanh' = 1 - tanh(Z)^2 (A holds tanh(Z))
__global__ void act_bwd_kernel(const float* dA, const float* A, float* dZ, long long n, int act)
{
    const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    dZ[i] = act == 1 ? dA[i] * (1.0f - A[i] * A[i]) : dA[i];
}

// ---------------------------------------------------------------------------
// Whole-network kernels.
//
// Bound by latency: a network of 37-128-128-128-30 on the 156 atom pairs of a
// molecule is 13 MFLOP.  A block of eight waves takes 16 rows of the batch
// through all layers, the rows' activations in LDS (two buffers of 16 x ldw
// floats), so that a network is one launch instead of one per layer: 44 ->
// 12 us per call at 156 rows (four launches of 8.6 us before), 44 -> 20 us of
// kernel at 2048 rows and 225 outputs.  Wave w owns the 16-column tiles w, w +
// 8, ... of a layer; its weights come from L2 in chunks of 128 k values (32
// registers), the next chunk (of this tile, the next tile or the next layer:
// weights depend on nothing) loaded before the current one's products, at
// clamped addresses (with a branch per load the kernel took 25 us at 156 rows
// instead of 13).  k ascends as in mm_kernel, so the outputs are the same.
// ---------------------------------------------------------------------------
#define NET_ROWS 16
#define NET_WAVES 8
#define NET_CHUNK 32   // MFMA steps (of 4 k) per register chunk of weights

struct NetFwd {
    const float* X;
    const float* W[MLP_MAX_LAYERS];
    const float* b[MLP_MAX_LAYERS];
    float* A[MLP_MAX_LAYERS];      // activations out (NULL: not wanted)
    int dims[MLP_MAX_LAYERS + 1];
    int nlayer, B, ldw;
};

// columns of a strip in LDS, zero from the width up: operands are read 32 k
// (eight products) at a time
__device__ __forceinline__ int net_pad(int d) { return (d + 31) & ~31; }

// the walk over (layer, tile, chunk) that one wave does
struct NetStep {
    int l, t, c;
};

__device__ __forceinline__ void net_fwd_next(const NetFwd& a, int wave, NetStep& s)
{
    const int I = a.dims[s.l];
    ++s.c;
    if (s.c * (4 * NET_CHUNK) >= I) {
        s.c = 0;
        s.t += NET_WAVES;
    }
    while (s.l < a.nlayer && s.t * 16 >= net_pad(a.dims[s.l + 1])) {
        ++s.l;
        s.t = wave;
        s.c = 0;
    }
}

__device__ __forceinline__ void net_fwd_load(const NetFwd& a, const NetStep& s, int lane, float (&w)[NET_CHUNK])
{
    if (s.l >= a.nlayer) return;
    const int I = a.dims[s.l], O = a.dims[s.l + 1];
    const float* __restrict__ W = a.W[s.l];
    const int n = s.t * 16 + (lane & 15), kb = s.c * (4 * NET_CHUNK) + (lane >> 4);
    const int nc = min(n, O - 1);
    // clamped addresses: every load issues, with no branch between them; what
    // lies past K is zeroed where it is used, columns past O are not stored
#pragma unroll
    for (int i = 0; i < NET_CHUNK; ++i) w[i] = W[min(kb + 4 * i, I - 1) * O + nc];
}

__global__ void __launch_bounds__(64 * NET_WAVES) net_fwd_kernel(const NetFwd a)
{
    extern __shared__ float net_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = blockIdx.x * NET_ROWS;
    NetStep s{0, wave, -1}, nx;
    float w[NET_CHUNK], wn[NET_CHUNK];
    net_fwd_next(a, wave, s);
    net_fwd_load(a, s, lane, w);
    {   // the input rows, zero past the batch and the width
        const int I = a.dims[0], Ip = net_pad(I);
        for (int e = tid; e < NET_ROWS * Ip; e += blockDim.x) {
            const int r = e / Ip, c = e - r * Ip;
            net_lds[r * a.ldw + c] = (row0 + r < a.B && c < I) ? a.X[(long long)(row0 + r) * I + c] : 0.0f;
        }
    }
    __syncthreads();
    for (int l = 0; l < a.nlayer; ++l) {
        const int I = a.dims[l], O = a.dims[l + 1];
        const float* xs = net_lds + (l & 1) * NET_ROWS * a.ldw;
        float* ys = net_lds + ((l + 1) & 1) * NET_ROWS * a.ldw;
        float* Ag = a.A[l];
        mlp_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        while (s.l == l) {
            nx = s;
            net_fwd_next(a, wave, nx);
            net_fwd_load(a, nx, lane, wn);
            const float* xr = xs + (lane & 15) * a.ldw + s.c * (4 * NET_CHUNK) + (lane >> 4);
            const int left = I - s.c * (4 * NET_CHUNK), groups = (left + 31) >> 5;
            float x[2][8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[0][i] = xr[4 * i];
#pragma unroll
            for (int g = 0; g < NET_CHUNK / 8; ++g)
                if (g < groups) {
                    // the next group's operands are in flight during this group's products
                    if (g + 1 < groups) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) x[(g + 1) & 1][i] = xr[32 * (g + 1) + 4 * i];
                    }
                    if (left < 32 * (g + 1)) {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            if (32 * g + 4 * i + (lane >> 4) >= left) w[8 * g + i] = 0.0f;
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[g & 1][i], w[8 * g + i], acc, 0, 0, 0);
                }
            if (nx.l != s.l || nx.t != s.t) {   // the tile's last chunk
                const int n = s.t * 16 + (lane & 15);
                const float bias = n < O ? a.b[l][n] : 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = 4 * (lane >> 4) + r;
                    float v = acc[r] + bias;
                    if (l + 1 < a.nlayer) v = tanhf(v);
                    if (l + 1 < a.nlayer) ys[m * a.ldw + n] = n < O ? v : 0.0f;
                    if (Ag && n < O && row0 + m < a.B) Ag[(long long)(row0 + m) * O + n] = v;
                }
                acc = (mlp_f4){0.0f, 0.0f, 0.0f, 0.0f};
            }
            s = nx;
#pragma unroll
            for (int i = 0; i < NET_CHUNK; ++i) w[i] = wn[i];
        }
        __syncthreads();
    }
}

// The dZ chain of a 16-row strip: dA = dZ W^T, dZ of the layer below = dA (1 -
// A^2), from the last layer down, every hidden layer's dZ also stored for
// dw_kernel.  The k index of a group of 16 runs 16 j + 4 (lane/16) + step, so
// that a lane's four weights are consecutive in its row of W (the row-major W
// is read along k) and its four activations are one 16-byte LDS read.
struct NetBwd {
    const float* dY;
    const float* W[MLP_MAX_LAYERS];
    const float* A[MLP_MAX_LAYERS];    // A[l]: tanh output of hidden layer l
    float* dZ[MLP_MAX_LAYERS];         // dZ[l] out of hidden layer l
    int dims[MLP_MAX_LAYERS + 1];
    int nlayer, B, ldw;
    int vec;                           // bit l: the rows of W[l] are 16-byte aligned
};

#define NETB_GROUPS 8                  // groups of 16 k per register chunk

__device__ __forceinline__ void net_bwd_next(const NetBwd& a, int wave, NetStep& s)
{
    ++s.c;
    if (s.c * (16 * NETB_GROUPS) >= a.dims[s.l + 1]) {
        s.c = 0;
        s.t += NET_WAVES;
    }
    while (s.l > 0 && s.t * 16 >= net_pad(a.dims[s.l])) {
        --s.l;
        s.t = wave;
        s.c = 0;
    }
}

__device__ __forceinline__ void net_bwd_load(const NetBwd& a, const NetStep& s, int lane,
                                             float (&w)[4 * NETB_GROUPS])
{
    if (s.l <= 0) return;
    const int I = a.dims[s.l], O = a.dims[s.l + 1];
    const float* __restrict__ W = a.W[s.l];
    const int n = s.t * 16 + (lane & 15), kb = s.c * (16 * NETB_GROUPS) + 4 * (lane >> 4);
    const int row = min(n, I - 1) * O;
    if (a.vec & (1 << s.l)) {   // rows of W on 16 bytes: O is a multiple of 4, so a group of four is in or out
#pragma unroll
        for (int j = 0; j < NETB_GROUPS; ++j) {
            const mlp_f4 v = *(const mlp_f4*)(W + row + min(kb + 16 * j, O - 4));
#pragma unroll
            for (int i = 0; i < 4; ++i) w[4 * j + i] = v[i];
        }
    } else {
#pragma unroll
        for (int j = 0; j < NETB_GROUPS; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) w[4 * j + i] = W[row + min(kb + 16 * j + i, O - 1)];
    }
}

__global__ void __launch_bounds__(64 * NET_WAVES) net_bwd_kernel(const NetBwd a)
{
    extern __shared__ float net_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = blockIdx.x * NET_ROWS, last = a.nlayer - 1;
    NetStep s{last, wave, -1}, nx;
    float w[4 * NETB_GROUPS], wn[4 * NETB_GROUPS];
    net_bwd_next(a, wave, s);
    net_bwd_load(a, s, lane, w);
    {
        const int O = a.dims[a.nlayer], Op = net_pad(O);
        for (int e = tid; e < NET_ROWS * Op; e += blockDim.x) {
            const int r = e / Op, c = e - r * Op;
            net_lds[r * a.ldw + c] = (row0 + r < a.B && c < O) ? a.dY[(long long)(row0 + r) * O + c] : 0.0f;
        }
    }
    __syncthreads();
    for (int l = last; l > 0; --l) {
        const int I = a.dims[l], O = a.dims[l + 1];
        const float* xs = net_lds + ((last - l) & 1) * NET_ROWS * a.ldw;
        float* ys = net_lds + ((last - l + 1) & 1) * NET_ROWS * a.ldw;
        mlp_f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        while (s.l == l) {
            nx = s;
            net_bwd_next(a, wave, nx);
            const bool tile_end = nx.l != s.l || nx.t != s.t;
            const int n = s.t * 16 + (lane & 15);
            float t[4];   // the layer below's outputs, in flight during the products
            if (tile_end) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    t[r] = a.A[l - 1][(long long)min(row0 + 4 * (lane >> 4) + r, a.B - 1) * I + min(n, I - 1)];
            }
            net_bwd_load(a, nx, lane, wn);
            const float* xr = xs + (lane & 15) * a.ldw + s.c * (16 * NETB_GROUPS) + 4 * (lane >> 4);
            const int left = O - s.c * (16 * NETB_GROUPS), groups = (left + 31) >> 5;
            mlp_f4 x[2][2];
            x[0][0] = *(const mlp_f4*)xr;
            x[0][1] = *(const mlp_f4*)(xr + 16);
#pragma unroll
            for (int g = 0; g < NETB_GROUPS / 2; ++g)
                if (g < groups) {
                    if (g + 1 < groups) {
                        x[(g + 1) & 1][0] = *(const mlp_f4*)(xr + 32 * (g + 1));
                        x[(g + 1) & 1][1] = *(const mlp_f4*)(xr + 32 * (g + 1) + 16);
                    }
                    if (left < 32 * (g + 1)) {
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            if (32 * g + 16 * (i >> 2) + 4 * (lane >> 4) + (i & 3) >= left) w[8 * g + i] = 0.0f;
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[g & 1][i >> 2][i & 3], w[8 * g + i], acc, 0, 0, 0);
                }
            if (tile_end) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = 4 * (lane >> 4) + r;
                    const long long g = (long long)(row0 + m) * I + n;
                    const bool in = n < I && row0 + m < a.B;
                    const float v = in ? acc[r] * (1.0f - t[r] * t[r]) : 0.0f;
                    ys[m * a.ldw + n] = v;
                    if (in) a.dZ[l - 1][g] = v;
                }
                acc = (mlp_f4){0.0f, 0.0f, 0.0f, 0.0f};
            }
            s = nx;
#pragma unroll
            for (int i = 0; i < 4 * NETB_GROUPS; ++i) w[i] = wn[i];
        }
        __syncthreads();
    }
}

// dW = X^T dZ and db = column sums of dZ of every layer in one launch.  A
// block owns a 16 x 32 tile of one layer's dW; its 16 waves split the batch
// rows and add their partial tiles through LDS, so the long reduction over
// the batch runs 16 ways in a block and needs neither atomics nor a second
// pass.  The tile of the first 16 rows of W also sums dZ's columns.  (One
// thread per column and a 16-block product over the whole batch took 1.4 ms
// and 0.52 ms of a 2.0 ms training step at 2048 rows, 37-128-128-128-225;
// this takes 12 us, the whole step 75 us, of which the host's calls are most.)
#define DW_WAVES 16
#define DW_UNROLL 8

struct DwJob {
    const float* X;       // [B x I]
    const float* dZ;      // [B x O]
    float* dW;
    float* db;
    int I, O, tn;         // tn: tiles along O
    int block0;           // first block of this layer
};

struct DwArgs {
    DwJob job[MLP_MAX_LAYERS];
    int njob, B;
};

__global__ void __launch_bounds__(64 * DW_WAVES) dw_kernel(const DwArgs a)
{
    __shared__ float part[DW_WAVES][8][64];
    __shared__ float bpart[DW_WAVES][32];
    int j = 0;
    while (j + 1 < a.njob && (int)blockIdx.x >= a.job[j + 1].block0) ++j;
    const DwJob& q = a.job[j];
    const int I = q.I, O = q.O, B = a.B;
    const int tile = blockIdx.x - q.block0;
    const int m0 = (tile / q.tn) * 16, n0 = (tile % q.tn) * 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = m0 + (lane & 15), n = n0 + (lane & 15), kq = lane >> 4;
    const bool vm = m < I, v0 = n < O, v1 = n + 16 < O;
    const int mc = min(m, I - 1), nc0 = min(n, O - 1), nc1 = min(n + 16, O - 1);
    const float* __restrict__ X = q.X;
    const float* __restrict__ dZ = q.dZ;
    // this wave's rows, whole groups of 4
    const int per = ((B + 4 * DW_WAVES - 1) / (4 * DW_WAVES)) * 4;
    const int k0 = wave * per, k1 = min(B, k0 + per);
    mlp_f4 c0 = {0.0f, 0.0f, 0.0f, 0.0f}, c1 = c0;
    float s0 = 0.0f, s1 = 0.0f;
    for (int k = k0; k < k1; k += 4 * DW_UNROLL) {
        float x[DW_UNROLL], z0[DW_UNROLL], z1[DW_UNROLL];
        // clamped addresses keep branches out from between the loads
#pragma unroll
        for (int u = 0; u < DW_UNROLL; ++u) {
            const long long kk = min(k + 4 * u + kq, B - 1);
            x[u] = X[kk * I + mc];
            z0[u] = dZ[kk * O + nc0];
            z1[u] = dZ[kk * O + nc1];
        }
#pragma unroll
        for (int u = 0; u < DW_UNROLL; ++u) {
            const bool in = k + 4 * u + kq < k1;
            x[u] = in && vm ? x[u] : 0.0f;
            z0[u] = in && v0 ? z0[u] : 0.0f;
            z1[u] = in && v1 ? z1[u] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < DW_UNROLL; ++u) {
            c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], z0[u], c0, 0, 0, 0);
            c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], z1[u], c1, 0, 0, 0);
            s0 += z0[u];
            s1 += z1[u];
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        part[wave][r][lane] = c0[r];
        part[wave][4 + r][lane] = c1[r];
    }
    if (m0 == 0) {
        s0 += __shfl_xor(s0, 16, 64);
        s0 += __shfl_xor(s0, 32, 64);
        s1 += __shfl_xor(s1, 16, 64);
        s1 += __shfl_xor(s1, 32, 64);
        if (lane < 16) {
            bpart[wave][lane] = s0;
            bpart[wave][16 + lane] = s1;
        }
    }
    __syncthreads();
    if (tid < 512) {   // element: register r of half h, lane ln of the tile
        const int ln = tid & 63, r = (tid >> 6) & 3, h = tid >> 8;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < DW_WAVES; ++w) v += part[w][4 * h + r][ln];
        const int mm = m0 + 4 * (ln >> 4) + r, nn = n0 + 16 * h + (ln & 15);
        if (mm < I && nn < O) q.dW[(long long)mm * O + nn] = v;
    } else if (m0 == 0 && tid < 544) {
        const int c = tid - 512;
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < DW_WAVES; ++w) v += bpart[w][c];
        if (n0 + c < O) q.db[n0 + c] = v;
    }
}

// loss = sum mask (Y - T)^2 / norm ; dY = 2 mask (Y - T) / norm.  At most 256
// blocks stride over the elements: one atomic per block onto the scalar loss
// (1800 blocks at 2048 x 225 queued 25 us of atomics on one address).
#define MSE_BLOCKS 256
__global__ void __launch_bounds__(256) mse_kernel(const float* __restrict__ Y, const float* __restrict__ T,
                                                  const float* __restrict__ mask, float* __restrict__ dY, float* loss,
                                                  long long n, float inv_norm)
{
    __shared__ float red[4];
    float l = 0.0f;
#pragma unroll 4
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
        const float w = mask ? mask[i] : 1.0f;
        const float d = (Y[i] - T[i]) * w;
        dY[i] = 2.0f * d * inv_norm;
        l += d * d * inv_norm;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) l += __shfl_xor(l, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, (red[0] + red[1]) + (red[2] + red[3]));
}

__device__ __forceinline__ void adam_element(float* p, const float* g, float* m, float* v, long long i, float lr,
                                             float b1, float b2, float eps, float c1, float c2)
{
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// one Adam step of several tensors in one launch: block -> tensor by the
// first-block table
struct AdamArgs {
    float* p[MLP_MAX_TENSORS];
    const float* g[MLP_MAX_TENSORS];
    float* m[MLP_MAX_TENSORS];
    float* v[MLP_MAX_TENSORS];
    long long n[MLP_MAX_TENSORS];
    int block0[MLP_MAX_TENSORS];
    int nt;
    float lr, b1, b2, eps, c1, c2;
};

__global__ void __launch_bounds__(256) adam_multi_kernel(const AdamArgs a)
{
    int t = 0;
    while (t + 1 < a.nt && (int)blockIdx.x >= a.block0[t + 1]) ++t;
    const long long i = (long long)((int)blockIdx.x - a.block0[t]) * 256 + threadIdx.x;
    if (i >= a.n[t]) return;
    adam_element(a.p[t], a.g[t], a.m[t], a.v[t], i, a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
}

int mlp_linear_fwd(const float* X, const float* W, const float* b, float* Z, float* A, int B, int I, int O, int act,
                   hipStream_t st)
{
    if (B <= 0 || I <= 0 || O <= 0) return -1;
    mm(false, false, X, W, b, Z, A, B, O, I, act, st);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// gradients of `njob` layers over the same batch
static int dw_launch(DwArgs& a, hipStream_t st)
{
    int blocks = 0;
    for (int j = 0; j < a.njob; ++j) {
        DwJob& q = a.job[j];
        q.tn = (q.O + 31) / 32;
        q.block0 = blocks;
        blocks += q.tn * ((q.I + 15) / 16);
    }
    hipLaunchKernelGGL(dw_kernel, dim3(blocks), dim3(64 * DW_WAVES), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int mlp_linear_bwd(const float* X, const float* W, const float* A, const float* dA, float* dZ, float* dX, float* dW,
                   float* db, int B, int I, int O, int act, hipStream_t st)
{
    if (B <= 0 || I <= 0 || O <= 0) return -1;
    const long long n = (long long)B * O;
    hipLaunchKernelGGL(act_bwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dA, A, dZ, n, act);
    if (dX) mm(false, true, dZ, W, nullptr, dX, nullptr, B, I, O, 0, st);          // dX = dZ W^T
    DwArgs a;
    a.njob = 1;
    a.B = B;
    a.job[0] = DwJob{X, dZ, dW, db, I, O, 0, 0};
    return dw_launch(a, st);
}

// LDS row length of a strip: a multiple of 64 plus 4 floats, so that the 16
// rows x 4 k of one operand read fall on 64 different banks and rows stay
// 16-byte aligned
static int net_ldw(int nlayer, const int* dims)
{
    int d = 0;
    for (int l = 0; l <= nlayer; ++l) d = dims[l] > d ? dims[l] : d;
    return (d + 63) / 64 * 64 + 4;
}

// both strips of 16 rows within 64 KiB of LDS
static bool net_fits(int ldw) { return 2 * NET_ROWS * ldw * (int)sizeof(float) <= 65536; }

static bool net_bad(int nlayer, const int* dims, int B)
{
    if (nlayer <= 0 || nlayer > MLP_MAX_LAYERS || B <= 0) return true;
    for (int l = 0; l <= nlayer; ++l)
        if (dims[l] <= 0) return true;
    return false;
}

int mlp_forward(int nlayer, const int* dims, const float* X, const float* const* W, const float* const* b,
                float* const* A, int B, hipStream_t st)
{
    if (net_bad(nlayer, dims, B)) return -1;
    const int ldw = net_ldw(nlayer, dims);
    if (!net_fits(ldw)) {
        // a layer wider than 448: one product per layer, which needs every
        // layer's output buffer
        for (int l = 0; l < nlayer; ++l) {
            if (!A[l]) return -2;
            mm(false, false, l ? A[l - 1] : X, W[l], b[l], nullptr, A[l], B, dims[l + 1], dims[l], l + 1 < nlayer, st);
        }
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    NetFwd a;
    a.X = X;
    for (int l = 0; l < nlayer; ++l) {
        a.W[l] = W[l];
        a.b[l] = b[l];
        a.A[l] = A[l];
    }
    for (int l = 0; l <= nlayer; ++l) a.dims[l] = dims[l];
    a.nlayer = nlayer;
    a.B = B;
    a.ldw = ldw;
    hipLaunchKernelGGL(net_fwd_kernel, dim3((B + NET_ROWS - 1) / NET_ROWS), dim3(64 * NET_WAVES),
                       2 * NET_ROWS * ldw * sizeof(float), st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int mlp_backward(int nlayer, const int* dims, const float* X, const float* const* A, const float* const* W,
                 const float* dY, float* const* dZ, float* const* dW, float* const* db, int B, hipStream_t st)
{
    if (net_bad(nlayer, dims, B)) return -1;
    const int ldw = net_ldw(nlayer, dims);
    if (nlayer > 1 && net_fits(ldw)) {
        NetBwd a;
        a.dY = dY;
        for (int l = 0; l < nlayer; ++l) {
            a.W[l] = W[l];
            a.A[l] = l + 1 < nlayer ? A[l] : nullptr;
            a.dZ[l] = l + 1 < nlayer ? dZ[l] : nullptr;
        }
        for (int l = 0; l <= nlayer; ++l) a.dims[l] = dims[l];
        a.nlayer = nlayer;
        a.B = B;
        a.ldw = ldw;
        a.vec = 0;
        for (int l = 1; l < nlayer; ++l)
            if (dims[l + 1] % 4 == 0 && (uintptr_t)W[l] % 16 == 0) a.vec |= 1 << l;
        hipLaunchKernelGGL(net_bwd_kernel, dim3((B + NET_ROWS - 1) / NET_ROWS), dim3(64 * NET_WAVES),
                           2 * NET_ROWS * ldw * sizeof(float), st, a);
    } else {
        for (int l = nlayer - 1; l > 0; --l) {
            const float* dz = l + 1 < nlayer ? dZ[l] : dY;
            const long long n = (long long)B * dims[l];
            mm(false, true, dz, W[l], nullptr, dZ[l - 1], nullptr, B, dims[l], dims[l + 1], 0, st);
            hipLaunchKernelGGL(act_bwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dZ[l - 1], A[l - 1],
                               dZ[l - 1], n, 1);
        }
    }
    DwArgs d;
    d.njob = nlayer;
    d.B = B;
    for (int l = 0; l < nlayer; ++l)
        d.job[l] = DwJob{l ? A[l - 1] : X, l + 1 < nlayer ? dZ[l] : dY, dW[l], db[l], dims[l], dims[l + 1], 0, 0};
    return dw_launch(d, st);
}

int mlp_mse(const float* Y, const float* T, const float* mask, float* dY, float* loss, long long n, float inv_norm,
            hipStream_t st)
{
    if (n <= 0) return -1;
    const long long blocks = (n + 255) / 256;
    hipLaunchKernelGGL(mse_kernel, dim3((unsigned)(blocks < MSE_BLOCKS ? blocks : MSE_BLOCKS)), dim3(256), 0, st, Y, T,
                       mask, dY, loss, n, inv_norm);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int mlp_adam(int nt, float* const* p, const float* const* g, float* const* m, float* const* v, const long long* n,
             float lr, float b1, float b2, float eps, int step, hipStream_t st)
{
    if (nt <= 0 || nt > MLP_MAX_TENSORS || step <= 0) return -1;
    AdamArgs a;
    a.nt = nt;
    a.lr = lr;
    a.b1 = b1;
    a.b2 = b2;
    a.eps = eps;
    a.c1 = 1.0f / (1.0f - powf(b1, (float)step));
    a.c2 = 1.0f / (1.0f - powf(b2, (float)step));
    long long blocks = 0;
    for (int t = 0; t < nt; ++t) {
        if (n[t] <= 0) return -1;
        a.p[t] = p[t];
        a.g[t] = g[t];
        a.m[t] = m[t];
        a.v[t] = v[t];
        a.n[t] = n[t];
        a.block0[t] = (int)blocks;
        blocks += (n[t] + 255) / 256;
        if (blocks > 0x7fffffff) return -1;
    }
    hipLaunchKernelGGL(adam_multi_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
