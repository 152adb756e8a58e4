// jk_common.h -- J/K digestion and dense-scatter kernel templates over the
// stored ERI classes.
#pragma once
#include "eri_common.h"

// --------------------------------------------------------------------------
// J/K digestion of one stored quartet block (8-fold symmetry, shell-level
// degeneracy factor).  For each element v = (mn|ls) with symmetric D:
//   J'_mn += 4s Dj_ls v   J'_ls += 4s Dj_mn v
//   K'_ml += 2s Dk_ns v   K'_nl += 2s Dk_ms v   K'_ms += 2s Dk_nl v   K'_ns += 2s Dk_ml v
// and J = (J' + J'^T)/2, K = (K' + K'^T)/2 afterwards.
// --------------------------------------------------------------------------
__device__ __forceinline__ void atomic_addd(double* p, double v)
{
    unsafeAtomicAdd(p, v);
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sums of T per-lane values over the wave: value 4 u + {0, 2, 1, 3}[lane / 16]
// ends in out[u] of that row's lanes.  The first two halvings swap halves and
// rows between two values, so that each swap and addition serves both; within a
// row of 16 lanes the values rotate (DPP).  No LDS: a shuffle per step and
// value was a third of the digestion's LDS instructions (18 values: 216 of
// them, against 102 vector instructions here).
__device__ __forceinline__ double swap_add32(double a, double b)
{
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

__device__ __forceinline__ double swap_add16(double a, double b)
{
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

template <int CTRL>
__device__ __forceinline__ double rotate_add(double a)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(a), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(a), CTRL, 0xf, 0xf, false);
    return a + __hiloint2double(hi, lo);
}

template <int T>
__device__ __forceinline__ void wave_sums(const double (&v)[T], double (&out)[(T + 3) / 4])
{
    constexpr int H = (T + 1) / 2, U = (T + 3) / 4;
    double h[H];
#pragma unroll
    for (int i = 0; i < H; ++i) h[i] = swap_add32(v[2 * i], 2 * i + 1 < T ? v[2 * i + 1] : 0.0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        double s = swap_add16(h[2 * u], 2 * u + 1 < H ? h[2 * u + 1] : 0.0);
        s = rotate_add<0x128>(s);   // row_ror 8, 4, 2, 1
        s = rotate_add<0x124>(s);
        s = rotate_add<0x122>(s);
        out[u] = rotate_add<0x121>(s);
    }
}

// One thread per stored quartet.  Lists are sorted by bra pair, so a wave
// usually shares one bra pair: then the bra-side J block is summed across the
// wave and written with one atomic per element instead of 64 colliding ones.
// Lanes past the end of the list stay active with zero weight so that the
// cross-lane sums see every lane of the wave.
template <int LA, int LB, int LC, int LD, typename real>
__global__ void __launch_bounds__(128) jk_kernel(const JkArgs<real> a)
{
    constexpr int N1 = (LA + 1) * (LA + 2) / 2, N2 = (LB + 1) * (LB + 2) / 2;
    constexpr int N3 = (LC + 1) * (LC + 2) / 2, N4 = (LD + 1) * (LD + 2) / 2;
    const int q0 = blockIdx.x * blockDim.x + threadIdx.x;
    if ((int)(blockIdx.x * blockDim.x + (threadIdx.x & ~63)) >= a.nq) return;   // whole wave past the end
    const bool valid = q0 < a.nq;
    const int q = valid ? q0 : a.nq - 1;
    const int2 pr = a.quartets[q];
    const PairHdr bh = a.pairs[pr.x], kh = a.pairs[pr.y];
    const int o1 = a.cart_off[bh.s1], o2 = a.cart_off[bh.s2];
    const int o3 = a.cart_off[kh.s1], o4 = a.cart_off[kh.s2];
    const MolInfo mi = a.mols[bh.mol];
    double sc = valid ? 1.0 : 0.0;
    if (bh.s1 == bh.s2) sc *= 0.5;
    if (kh.s1 == kh.s2) sc *= 0.5;
    if (pr.x == pr.y) sc *= 0.5;
    const int bra0 = __shfl(pr.x, 0, 64);
    const bool uniform = __all(pr.x == bra0);
    const int lane = threadIdx.x & 63;
    const int n = mi.n;
    const double* Dj = a.Dj + mi.base;
    const double* Dk = a.Dk + mi.base;
    double* const Jm = a.J + mi.base;
    double* const Km = a.K + mi.base;
    const size_t nq = a.nq;
    double j34[N3 * N4], k23[N2 * N3], k24[N2 * N4];
#pragma unroll
    for (int i = 0; i < N3 * N4; ++i) j34[i] = 0.0;
#pragma unroll
    for (int i = 0; i < N2 * N3; ++i) k23[i] = 0.0;
#pragma unroll
    for (int i = 0; i < N2 * N4; ++i) k24[i] = 0.0;
#pragma unroll
    for (int ia = 0; ia < N1; ++ia) {
        double k13[N3], k14[N4];
#pragma unroll
        for (int i = 0; i < N3; ++i) k13[i] = 0.0;
#pragma unroll
        for (int i = 0; i < N4; ++i) k14[i] = 0.0;
#pragma unroll
        for (int ib = 0; ib < N2; ++ib) {
            const double d12 = Dj[(size_t)(o1 + ia) * n + o2 + ib];
            double j12 = 0.0;
#pragma unroll
            for (int ic = 0; ic < N3; ++ic) {
                const double d13 = Dk[(size_t)(o1 + ia) * n + o3 + ic];
                const double d23 = Dk[(size_t)(o2 + ib) * n + o3 + ic];
#pragma unroll
                for (int id = 0; id < N4; ++id) {
                    const double v = (double)a.vals[(size_t)(((ia * N2 + ib) * N3 + ic) * N4 + id) * nq + q];
                    j12 += Dj[(size_t)(o3 + ic) * n + o4 + id] * v;
                    j34[ic * N4 + id] += d12 * v;
                    k13[ic] += Dk[(size_t)(o2 + ib) * n + o4 + id] * v;
                    k23[ib * N3 + ic] += Dk[(size_t)(o1 + ia) * n + o4 + id] * v;
                    k14[id] += d23 * v;
                    k24[ib * N4 + id] += d13 * v;
                }
            }
            double* dst = &Jm[(size_t)(o1 + ia) * n + o2 + ib];
            if (uniform) {
                const double s = wave_sum(4.0 * sc * j12);
                if (lane == 0) atomic_addd(dst, s);
            } else if (valid) {
                atomic_addd(dst, 4.0 * sc * j12);
            }
        }
        if (valid) {
#pragma unroll
            for (int ic = 0; ic < N3; ++ic) atomic_addd(&Km[(size_t)(o1 + ia) * n + o3 + ic], 2.0 * sc * k13[ic]);
#pragma unroll
            for (int id = 0; id < N4; ++id) atomic_addd(&Km[(size_t)(o1 + ia) * n + o4 + id], 2.0 * sc * k14[id]);
        }
    }
    if (!valid) return;
#pragma unroll
    for (int ic = 0; ic < N3; ++ic)
#pragma unroll
        for (int id = 0; id < N4; ++id) atomic_addd(&Jm[(size_t)(o3 + ic) * n + o4 + id], 4.0 * sc * j34[ic * N4 + id]);
#pragma unroll
    for (int ib = 0; ib < N2; ++ib) {
#pragma unroll
        for (int ic = 0; ic < N3; ++ic) atomic_addd(&Km[(size_t)(o2 + ib) * n + o3 + ic], 2.0 * sc * k23[ib * N3 + ic]);
#pragma unroll
        for (int id = 0; id < N4; ++id) atomic_addd(&Km[(size_t)(o2 + ib) * n + o4 + id], 2.0 * sc * k24[ib * N4 + id]);
    }
}

// Tiled J/K digestion.  A work item is a contiguous range of quartets that
// share one bra pair (a,b) (the class lists are sorted by bra pair).  Every K
// contribution of such a range lands in rows of shells a and b, so those rows
// are accumulated in LDS and flushed to global memory once per item, and the
// bra rows of Dk that every K term reads are staged in LDS beside them.  The
// bra-side J block is summed over each wave.  The ket J block of every
// quartet is stored, not added: jkbuf[(tile * N3 * N4 + cd) * nq + q] holds
// 4 s sum_ab Dj_ab (ab|cd) for it, and a reduction over the bras that reach
// each ket (jket_reduce) adds those into J' with one atomic per ket element.
//
// The bra components are cut into tiles of TA x TB (first x second shell
// components); blockIdx.y selects the tile.  Each lane holds, per quartet,
// TA*TB*N3*N4 values and 2(TA+TB)(N4+1) + 2 TA TB accumulators and density
// elements, which is what bounds the register file: the generator picks the
// tile per class.  The ket loop runs c outer, d inner, so the ket J sum of
// element (c,d) is complete in a register when it is written.
struct JkItem {
    int start, end;   // quartet range [start, end)
    int bra;          // o1 | o2 << 15 | (s1 == s2) << 30, offsets local to the molecule
    int mol;
};

template <typename real>
struct JkTileList {
    const unsigned* kets;    // per quartet: o3 | o4 << 15 | (s3 == s4) << 30 | (P == Q) << 31
    const real* vals;
    double* jkbuf;           // [ntiles * N3 * N4][nq] ket J values per quartet
    int nq;
};

// Both stored lists of one class (FP64 values, and FP32 values below the
// Schwarz split).  A work item is a chunk of one bra pair's kets: its FP64
// quartets [start, end) then its FP32 quartets items32[item] (the bra's FP32
// kets follow its FP64 kets in bound order), digested with the same staged
// rows.
struct JkClassArgs {
    const JkItem* items;
    const int2* items32;     // FP32 quartet range per item (NULL: FP64 list only)
    JkTileList<double> l64;
    JkTileList<float> l32;
    int nitems, grid;        // grid: blocks per bra tile (<= nitems; each strides over items when smaller)
    int block0;              // first block of the class in its launch
    int cls;
};

// Several classes in one launch (jk_group_kernel_*): a Fock build is a handful
// of launches instead of one per class.  clock (NULL: off): per class the
// earliest start and latest end of its blocks in ticks of the realtime clock.
#define JK_MAXCLASS 21
struct JkGroupArgs {
    JkClassArgs c[JK_MAXCLASS];
    int n;
    const MolInfo* mols;
    const double* Dj;
    const double* Dk;
    double* J;
    double* K;
    unsigned long long* clock;
};

// The TA + TB rows lie in LDS column by column, element (row r, column c) at
// c * JkRows::stride + r: what a quartet reads or adds at one column is one
// address with constant offsets (and pairs of reads are one instruction), where
// rows n apart cost an address each: with the division-free staging half the
// vector instructions of a C20H42 build (2.45e8 -> 1.40e8), 86 registers
// instead of 100 in the lightest group and 128 instead of 156 in the (ds| one.
// The stride is odd, so that the columns that a wave's lanes hold spread over
// all banks.
template <int TA, int TB>
struct JkRows {
    static constexpr int count = TA + TB, stride = count | 1;
};

// The quartets [q0, q1) of one list for the current item and tile.  Quartet
// q0 + i goes to thread (i + shift) mod blockDim: with shift = the number of
// quartets of the FP64 range, the FP32 range continues where the FP64 range
// ended, so that in a short item no thread takes a quartet of each list.
//
// Classes with at least three ket components (every ket but ss) digest one
// (quartet, ket row c) unit per thread instead of a quartet: N3 times the
// independent units of an item, and only one row's values in registers.  Unit
// u of the range is row u / len, quartet q0 + u % len (consecutive lanes read
// consecutive quartets of one row).  The K contributions of row c go to the
// LDS rows at once, the ket J values to their own jkbuf slots.  A ket of two s
// shells is one row.
template <int LA, int LB, int LC, int LD, int TA, int TB, typename real>
struct JkUnit {
    static constexpr int N2 = (LB + 1) * (LB + 2) / 2;
    static constexpr int N3 = (LC + 1) * (LC + 2) / 2, N4 = (LD + 1) * (LD + 2) / 2;
    static constexpr int RS = JkRows<TA, TB>::stride;
    // what a unit reads from memory, all loads in flight together; values in
    // the list's own type until use (an FP32 row takes half the registers)
    unsigned w;
    int q, c;
    real vv[N4][TA][TB];
    double dj[N4];

    __device__ __forceinline__ void load(const JkTileList<real>& L, int u, int q0, int len, int n,
                                         const double* __restrict__ Dj, int a0, int b0)
    {
        c = N3 > 1 ? u / len : 0;
        q = q0 + (u - c * len);
        const size_t nq = L.nq;
        const real* __restrict__ vals = L.vals;
        w = L.kets[q];
#pragma unroll
        for (int d = 0; d < N4; ++d)
#pragma unroll
            for (int x = 0; x < TA; ++x)
#pragma unroll
                for (int y = 0; y < TB; ++y)
                    vv[d][x][y] = vals[(size_t)((((a0 + x) * N2 + b0 + y) * N3 + c) * N4 + d) * nq + q];
        const int o3 = w & 0x7fff, o4 = (w >> 15) & 0x7fff;
#pragma unroll
        for (int d = 0; d < N4; ++d) dj[d] = Dj[(size_t)(o3 + c) * n + o4 + d];
    }

    __device__ __forceinline__ void digest(const JkTileList<real>& L, const double* drows, double* krows, double sbra,
                                           const double (&d12)[TA][TB], double (&j12)[TA][TB], int tile) const
    {
        const int o3 = w & 0x7fff, o4 = (w >> 15) & 0x7fff;
        double sc = sbra;
        if ((w >> 30) & 1u) sc *= 0.5;
        if (w >> 31) sc *= 0.5;
        const double* dc = drows + (o3 + c) * RS;
        double* kc = krows + (o3 + c) * RS;
        double d13[TA], d23[TB], k13[TA], k23[TB];
#pragma unroll
        for (int x = 0; x < TA; ++x) {
            d13[x] = dc[x];
            k13[x] = 0.0;
        }
#pragma unroll
        for (int y = 0; y < TB; ++y) {
            d23[y] = dc[TA + y];
            k23[y] = 0.0;
        }
        double* __restrict__ jkbuf = L.jkbuf + (size_t)(tile * N3 * N4 + c * N4) * L.nq + q;
#pragma unroll
        for (int d = 0; d < N4; ++d) {
            const double* dd = drows + (o4 + d) * RS;
            double* kd = krows + (o4 + d) * RS;
            double d14[TA], d24[TB], k14[TA], k24[TB];
#pragma unroll
            for (int x = 0; x < TA; ++x) {
                d14[x] = dd[x];
                k14[x] = 0.0;
            }
#pragma unroll
            for (int y = 0; y < TB; ++y) {
                d24[y] = dd[TA + y];
                k24[y] = 0.0;
            }
            double jcd = 0.0;
#pragma unroll
            for (int x = 0; x < TA; ++x)
#pragma unroll
                for (int y = 0; y < TB; ++y) {
                    const double v = sc * (double)vv[d][x][y];
                    j12[x][y] += dj[d] * v;
                    jcd += d12[x][y] * v;
                    k13[x] += d24[y] * v;
                    k14[x] += d23[y] * v;
                    k23[y] += d14[x] * v;
                    k24[y] += d13[x] * v;
                }
            jkbuf[(size_t)d * L.nq] = 4.0 * jcd;
#pragma unroll
            for (int x = 0; x < TA; ++x) atomicAdd(&kd[x], 2.0 * k14[x]);
#pragma unroll
            for (int y = 0; y < TB; ++y) atomicAdd(&kd[TA + y], 2.0 * k24[y]);
        }
#pragma unroll
        for (int x = 0; x < TA; ++x) atomicAdd(&kc[x], 2.0 * k13[x]);
#pragma unroll
        for (int y = 0; y < TB; ++y) atomicAdd(&kc[TA + y], 2.0 * k23[y]);
    }
};

template <int LA, int LB, int LC, int LD, int TA, int TB>
__device__ __forceinline__ void jk_tile_item(const JkGroupArgs& g, const JkClassArgs& a, int item, double* lds, int tile)
{
    constexpr int N1 = (LA + 1) * (LA + 2) / 2, N2 = (LB + 1) * (LB + 2) / 2, N3 = (LC + 1) * (LC + 2) / 2;
    static_assert(N1 % TA == 0 && N2 % TB == 0, "tile must divide the bra components");
    constexpr int NTB = N2 / TB, NR = TA + TB, RS = JkRows<TA, TB>::stride;
    const int a0 = (tile / NTB) * TA, b0 = (tile % NTB) * TB;
    const int tid = threadIdx.x, nt = blockDim.x;
    const JkItem it = a.items[item];
    const MolInfo mi = g.mols[it.mol];
    const int n = mi.n;
    double* drows = lds;            // rows of Dk: o1+a0.., then o2+b0..
    double* krows = lds + RS * n;   // K' rows, same order
    const int o1 = it.bra & 0x7fff, o2 = (it.bra >> 15) & 0x7fff;
    const double sbra = ((it.bra >> 30) & 1) ? 0.5 : 1.0;
    const double* __restrict__ Dj = g.Dj + mi.base;
    const double* __restrict__ Dk = g.Dk + mi.base;
    double* const Jm = g.J + mi.base;
    double* const Km = g.K + mi.base;
    // the first unit's loads are in flight while the rows are staged
    const int len = it.end - it.start, total = N3 * len;
    JkUnit<LA, LB, LC, LD, TA, TB, double> un;
    if (tid < total) un.load(a.l64, tid, it.start, len, n, Dj, a0, b0);
    const double* __restrict__ ra = Dk + (size_t)(o1 + a0) * n;
    const double* __restrict__ rb = Dk + (size_t)(o2 + b0) * n;
    for (int c = tid; c < n; c += nt) {
        double v[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] = r < TA ? ra[(size_t)r * n + c] : rb[(size_t)(r - TA) * n + c];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            drows[c * RS + r] = v[r];
            krows[c * RS + r] = 0.0;
        }
    }
    double d12[TA][TB], j12[TA][TB];
#pragma unroll
    for (int x = 0; x < TA; ++x)
#pragma unroll
        for (int y = 0; y < TB; ++y) {
            d12[x][y] = Dj[(size_t)(o1 + a0 + x) * n + o2 + b0 + y];
            j12[x][y] = 0.0;
        }
    __syncthreads();
    for (int u = tid; u < total;) {
        un.digest(a.l64, drows, krows, sbra, d12, j12, tile);
        u += nt;
        if (u < total) un.load(a.l64, u, it.start, len, n, Dj, a0, b0);
    }
    if (a.items32) {
        const int2 r32 = a.items32[item];
        const int len32 = r32.y - r32.x, total32 = N3 * len32;
        JkUnit<LA, LB, LC, LD, TA, TB, float> uf;
        for (int u = (tid - total % nt + nt) % nt; u < total32; u += nt) {
            uf.load(a.l32, u, r32.x, len32, n, Dj, a0, b0);
            uf.digest(a.l32, drows, krows, sbra, d12, j12, tile);
        }
    }
    {
        double flat[TA * TB], sum[(TA * TB + 3) / 4];
#pragma unroll
        for (int t = 0; t < TA * TB; ++t) flat[t] = 4.0 * j12[t / TB][t % TB];
        wave_sums(flat, sum);
        if ((tid & 15) == 0) {
            const int row = (tid >> 4) & 3, first = row == 1 ? 2 : (row == 2 ? 1 : row);
#pragma unroll
            for (int u = 0; u < (TA * TB + 3) / 4; ++u) {
                const int t = 4 * u + first;
                if (t < TA * TB && sum[u] != 0.0)
                    atomic_addd(&Jm[(size_t)(o1 + a0 + t / TB) * n + o2 + b0 + t % TB], sum[u]);
            }
        }
    }
    __syncthreads();
    double* const ka = Km + (size_t)(o1 + a0) * n;
    double* const kb = Km + (size_t)(o2 + b0) * n;
    for (int c = tid; c < n; c += nt) {
        double v[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) v[r] = krows[c * RS + r];
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (v[r] != 0.0) atomic_addd(r < TA ? &ka[(size_t)r * n + c] : &kb[(size_t)(r - TA) * n + c], v[r]);
    }
    __syncthreads();
}

// block `local` of a class: bra tile local / grid, items local % grid, + grid, ...
template <int LA, int LB, int LC, int LD, int TA, int TB>
__device__ __forceinline__ void jk_tile_class(const JkGroupArgs& g, const JkClassArgs& a, int local, double* lds)
{
    const int tile = local / a.grid;
    for (int item = local - tile * a.grid; item < a.nitems; item += a.grid)
        jk_tile_item<LA, LB, LC, LD, TA, TB>(g, a, item, lds, tile);
}

__device__ __forceinline__ int jk_group_slot(const JkGroupArgs& g)
{
    int s = 0;
    while (s + 1 < g.n && (int)blockIdx.x >= g.c[s + 1].block0) ++s;
    return s;
}

// (start, end) of a class in the timed builds, in JK_CLOCK_SLOTS copies that
// the blocks share out among themselves: one copy for 60 000 blocks took
// C20H42's build from 1.12 to 1.43 ms.
#define JK_CLOCK_SLOTS 64
#define JK_CLOCK_CLASSES 32
__host__ __device__ __forceinline__ int jk_clock_at(int slot, int cls) { return 2 * (slot * JK_CLOCK_CLASSES + cls); }

__device__ __forceinline__ void jk_clock(const JkGroupArgs& g, int cls, int end)
{
    if (!g.clock || threadIdx.x) return;
    const unsigned long long t = wall_clock64();
    unsigned long long* c = g.clock + jk_clock_at(blockIdx.x & (JK_CLOCK_SLOTS - 1), cls);
    if (end) atomicMax(c + 1, t);
    else atomicMin(c, t);
}

// Dense scatter with 8-fold permutational symmetry (Methods/hartree_fock.py:314-325)
// into a slab of third indices l in [l0, l0 + lc): out[m][n][l - l0][s].  One
// thread per (component, quartet), component-major, so that consecutive
// threads read consecutive values: a single high-l quartet (an atom's
// (dd|dd)) spreads over its components instead of one thread writing them
// all.
template <int LA, int LB, int LC, int LD, typename real>
__global__ void __launch_bounds__(256) scatter_kernel(const ScatterArgs<real> a)
{
    constexpr int N2 = (LB + 1) * (LB + 2) / 2;
    constexpr int N3 = (LC + 1) * (LC + 2) / 2, N4 = (LD + 1) * (LD + 2) / 2;
    constexpr int N1 = (LA + 1) * (LA + 2) / 2, NC = N1 * N2 * N3 * N4;
    const long long nq = a.nq;
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= nq * NC) return;
    const int comp = (int)(t / nq);
    const long long q = t - comp * nq;
    const int id = comp % N4, ic = (comp / N4) % N3, ib = (comp / (N3 * N4)) % N2, ia = comp / (N2 * N3 * N4);
    const int2 pr = a.quartets[q];
    const PairHdr bh = a.pairs[pr.x], kh = a.pairs[pr.y];
    // Positions reached from two components (a pair of one shell with
    // itself, a quartet of one pair with itself) hold values equal up to
    // rounding; one canonical component writes them, so that the result
    // does not depend on the order of the threads.  The symmetric images
    // of the kept components still cover every position.
    if (bh.s1 == bh.s2 && ia < ib) return;
    if (kh.s1 == kh.s2 && ic < id) return;
    if (pr.x == pr.y && ia * N2 + ib < ic * N4 + id) return;
    const long long n = a.n, l0 = a.l0, lc = a.lc;
    const long long m = a.cart_off[bh.s1] + ia, nn = a.cart_off[bh.s2] + ib;
    const long long l = a.cart_off[kh.s1] + ic, s = a.cart_off[kh.s2] + id;
    const double v = (double)a.vals[(size_t)comp * nq + q];
    auto put = [&](long long i, long long j, long long k, long long r) {
        const long long u = k - l0;
        if (u >= 0 && u < lc) a.out[((i * n + j) * lc + u) * n + r] = v;
    };
    put(m, nn, l, s);
    put(nn, m, l, s);
    put(m, nn, s, l);
    put(nn, m, s, l);
    put(l, s, m, nn);
    put(l, s, nn, m);
    put(s, l, m, nn);
    put(s, l, nn, m);
}

// The stored quartets as a symmetric matrix over packed function pairs (a shell
// pair's functions are neighbours, PairScatterArgs): out[P - p0][Q] and its
// image [Q][P] for rows in [p0, p0 + rows).  Bound by the scattered writes:
// two of 8 bytes per stored value against the eight that the dense tensor
// takes (C10H22: 11.0 ms for its 560 M writes, 1.7 ms for these 140 M).  A thread writes AB rows of
// its quartet's bra functions times all ket functions, so that the 8 to 288
// contiguous bytes of a block's row leave together; consecutive lanes take
// consecutive quartets, whose values are neighbours.
template <int N12, int N34>
struct PairScatterSplit {
    static constexpr int pick(int d) { return (N12 % d == 0 && d * N34 <= 54) || d == 1 ? d : pick(d - 1); }
    static constexpr int AB = pick(N12);
};

template <int LA, int LB, int LC, int LD, typename real>
__global__ void __launch_bounds__(256) pair_scatter_kernel(const PairScatterArgs<real> a)
{
    constexpr int N1 = (LA + 1) * (LA + 2) / 2, N2 = (LB + 1) * (LB + 2) / 2;
    constexpr int N3 = (LC + 1) * (LC + 2) / 2, N4 = (LD + 1) * (LD + 2) / 2;
    constexpr int N34 = N3 * N4, AB = PairScatterSplit<N1 * N2, N34>::AB;
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= a.nq) return;
    const int ab0 = blockIdx.y * AB;
    const size_t nq = a.nq;
    const int2 pr = a.quartets[q];
    const PairHdr bh = a.pairs[pr.x], kh = a.pairs[pr.y];
    const bool sb = LA == LB && bh.s1 == bh.s2, sk = LC == LD && kh.s1 == kh.s2;
    const bool same = LA == LC && LB == LD && pr.x == pr.y;
    const long long P0 = a.pair_base[pr.x], Q0 = a.pair_base[pr.y];
    real v[AB][N34];
#pragma unroll
    for (int x = 0; x < AB; ++x)
#pragma unroll
        for (int c = 0; c < N34; ++c) v[x][c] = a.vals[(size_t)((ab0 + x) * N34 + c) * nq + q];
#pragma unroll
    for (int x = 0; x < AB; ++x) {
        const int ab = ab0 + x, i = ab / N2, j = ab % N2;
        if (sb && i < j) continue;
        const long long P = P0 + pair_component(sb, N2, i, j);
#pragma unroll
        for (int c = 0; c < N34; ++c) {
            const int k = c / N4, l = c % N4;
            // of two components at one position (equal up to rounding) the
            // canonical one is written, whatever the order of the threads
            if (sk && k < l) continue;
            if (same && ab < c) continue;
            const long long Q = Q0 + pair_component(sk, N4, k, l);
            const double w = (double)v[x][c];
            const long long rp = P - a.p0, rq = Q - a.p0;
            if (rp >= 0 && rp < a.rows) a.out[rp * a.np + Q] = w;
            if (rq >= 0 && rq < a.rows) a.out[rq * a.np + P] = w;
        }
    }
}
