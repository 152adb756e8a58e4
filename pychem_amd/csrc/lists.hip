// lists.hip -- device construction of the screened quartet lists and the ket
// J reduction (the list layout and its monotonicity are described in lists.h).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lists.h"

// First index in [lo, hi) where pred holds, for a predicate that is false
// then true along the range; hi when it never holds.
template <typename Pred>
__device__ __forceinline__ int first_true(int lo, int hi, Pred pred)
{
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if (pred(mid)) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// Largest i in [0, n) with v[i] <= x (v non-decreasing, v[0] <= x).
__device__ __forceinline__ int last_le(const long long* v, int n, long long x)
{
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = lo + (hi - lo) / 2;
        if (v[mid] <= x) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Per bra: its FP64 ket run [j0, f64) and FP32 run [f64, fa) with
//   fa  = first ket with !(bound_i bound_j > thr), at least one past the
//         diagonal when bra and ket lists agree;
//   f64 = first ket with bound_i bound_j < thr32 (thr32 > 0), clipped to
//         [j0 + diagonal, fa].
__device__ __forceinline__ void list_count_one(const ListArgs& a, const ListBras& b64, const ListBras& b32, int i)
{
    const int P = a.bra[i];
    const PairHdr ph = a.pairs[P];
    const double qb = a.bound[P];
    const int e = a.ket_seg[ph.mol + 1];
    const int j0 = a.same ? i : a.ket_seg[ph.mol];
    int fa = first_true(j0, e, [&](int j) { return !(qb * a.bound[a.ket[j]] > a.thr); });
    if (a.same && fa < j0 + 1) fa = j0 + 1;
    int f64 = a.thr32 > 0.0 ? first_true(j0, e, [&](int j) { return qb * a.bound[a.ket[j]] < a.thr32; }) : e;
    if (f64 > fa) f64 = fa;
    if (a.same && f64 < j0 + 1) f64 = j0 + 1;
    const long long npb = ph.n;
    b64.j0[i] = j0;
    b64.cnt[i] = f64 - j0;
    b64.np[i] = npb * (a.ket_npcum[f64] - a.ket_npcum[j0]);
    b32.j0[i] = f64;
    b32.cnt[i] = fa - f64;
    b32.np[i] = npb * (a.ket_npcum[fa] - a.ket_npcum[f64]);
}

__global__ void list_count_kernel(const ListArgs a, const ListBras b64, const ListBras b32)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.nb) list_count_one(a, b64, b32, i);
}

// Single-workgroup exclusive scan: each thread scans a contiguous chunk,
// chunk sums are scanned in LDS.
__device__ __forceinline__ void list_scan_one(const long long* in, long long* out, int n, long long* total)
{
    __shared__ long long part[1024];
    const int t = threadIdx.x;
    const int per = (n + 1023) / 1024;
    const int lo = min(n, t * per), hi = min(n, lo + per);
    long long s = 0;
    for (int i = lo; i < hi; ++i) s += in[i];
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const long long v = t >= off ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    long long run = part[t] - s;
    for (int i = lo; i < hi; ++i) {
        const long long x = in[i];
        out[i] = run;
        run += x;
    }
    if (t == 1023) *total = part[1023];
}

__global__ void __launch_bounds__(1024) list_scan_kernel(const long long* in, long long* out, int n, long long* total)
{
    list_scan_one(in, out, n, total);
}

__global__ void __launch_bounds__(1024) list_scan_batch_kernel(const ScanJob* jobs)
{
    const ScanJob j = jobs[blockIdx.x];
    list_scan_one(j.in, j.out, j.n, j.total);
}

// Items of a class: per bra, its FP64 kets then its FP32 kets cut into
// chunks of `run` quartets.
__global__ void list_items_count_kernel(const long long* cnt64, const long long* cnt32, long long* nit, int nb,
                                        long long run)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nb) nit[i] = (cnt64[i] + (cnt32 ? cnt32[i] : 0) + run - 1) / run;
}

// One thread per quartet: its bra is the last with qs <= q (bras without
// kets share the next bra's qs and are never last).
__device__ __forceinline__ void list_fill_one(const ListArgs& a, const ListBras& b, long long q, int2* quartets,
                                              unsigned* kets)
{
    const int i = last_le(b.qs, a.nb, q);
    const int j = b.j0[i] + (int)(q - b.qs[i]);
    const int P = a.bra[i], Q = a.ket[j];
    quartets[q] = make_int2(P, Q);
    kets[q] = a.ket_rec[j] | (P == Q ? 1u << 31 : 0u);
}

__global__ void list_fill_kernel(const ListArgs a, const ListBras b, long long nq, int2* quartets, unsigned* kets)
{
    const long long q = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (q < nq) list_fill_one(a, b, q, quartets, kets);
}

// Item t covers positions [lo, hi) of its bra's concatenated run (FP64
// kets, then FP32 kets): FP64 quartets qs64 + [min(lo, c64), min(hi, c64)),
// FP32 quartets qs32 + [max(lo - c64, 0), max(hi - c64, 0)).
__device__ __forceinline__ void list_items_fill_one(const ListArgs& a, const ListBras& b, const ListBras& b32,
                                                    long long t, long long run, JkItem* items, int2* items32)
{
    const int i = last_le(b.its, a.nb, t);
    const long long r = t - b.its[i];
    const long long c64 = b.cnt[i], c32 = items32 ? b32.cnt[i] : 0;
    const long long lo = r * run, hi = lo + run < c64 + c32 ? lo + run : c64 + c32;
    const PairHdr bh = a.pairs[a.bra[i]];
    JkItem it;
    it.start = (int)(b.qs[i] + (lo < c64 ? lo : c64));
    it.end = (int)(b.qs[i] + (hi < c64 ? hi : c64));
    it.bra = a.cart_off[bh.s1] | (a.cart_off[bh.s2] << 15) | ((bh.s1 == bh.s2) ? (1 << 30) : 0);
    it.mol = bh.mol;
    items[t] = it;
    if (items32) {
        const long long s0 = lo > c64 ? lo - c64 : 0, s1 = hi > c64 ? hi - c64 : 0;
        items32[t] = make_int2((int)(b32.qs[i] + s0), (int)(b32.qs[i] + s1));
    }
}

__global__ void list_items_fill_kernel(const ListArgs a, const ListBras b, const ListBras b32, long long nitems,
                                       long long run, JkItem* items, int2* items32)
{
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t < nitems) list_items_fill_one(a, b, b32, t, run, items, items32);
}

// ---- batched phases: job of a block from the first-block table (uniform)
__device__ __forceinline__ int list_job_of(const ListBlocks& blk, int& local)
{
    const int b = blockIdx.x;
    int j = 0;
    while (j + 1 < blk.n && blk.block0[j + 1] <= b) ++j;
    local = (b - blk.block0[j]) * 256 + threadIdx.x;
    return j;
}

__global__ void __launch_bounds__(256) list_count_batch_kernel(const ListJob* jobs, const ListBlocks blk)
{
    int i;
    const int j = list_job_of(blk, i);
    const ListJob& J = jobs[j];
    if (i < J.a.nb) list_count_one(J.a, J.b64, J.b32, i);
}

// Bucket of a quartet of `work` primitive quartets: 0 holds the most, half an
// octave per bucket.
__device__ __forceinline__ int order_bucket(int work)
{
    work = max(1, work);
    const int lg = 31 - __clz(work);                                  // floor(log2 work)
    const int k = 2 * lg + (lg > 0 ? (work >> (lg - 1)) & 1 : 0);   // half-octaves
    return ORD_NB - 1 - min(k, ORD_NB - 1);
}

// list of block blockIdx.x (blocks of ORD_PT * 256 quartets) and the
// block's index within it
__device__ __forceinline__ int order_job_of(const ListBlocks& blk, int& lb)
{
    const int b = blockIdx.x;
    int j = 0;
    while (j + 1 < blk.n && blk.block0[j + 1] <= b) ++j;
    lb = b - blk.block0[j];
    return j;
}

// lanes of the wave that hold a quartet (ok) of the same bucket as this one
__device__ __forceinline__ unsigned long long bucket_peers(int bucket, bool ok)
{
    unsigned long long m = __ballot(ok);
#pragma unroll
    for (int k = 0; (1 << k) < ORD_NB; ++k) {
        const bool bit = (bucket >> k) & 1;
        const unsigned long long v = __ballot(bit);
        m &= bit ? v : ~v;
    }
    return m;
}

// Quartets q0 ... of one list, ORD_PT * 256 to a block: the bras of the
// block's first and last quartet are searched once, each quartet's bra
// between them, and what a quartet needs of its ket lies in ket order (one
// search over all bras and three gathers, each behind the last, per quartet:
// C14H30 122 us, 87 now).  Bucket and bucket counts are taken here, where both
// pairs' primitive counts are at hand.
__global__ void __launch_bounds__(256) list_fill_batch_kernel(const ListJob* jobs, const ListBlocks blk, int* cnt)
{
    __shared__ int h[ORD_NB], ends[2];
    int lb;
    const int jw = order_job_of(blk, lb), w = jw & 1;
    const ListJob& J = jobs[jw >> 1];
    // copies: the stores below could alias the job
    const ListArgs a = J.a;
    const ListBras b = w ? J.b32 : J.b64;
    const long long q0 = (long long)lb * 256 * ORD_PT, left = J.nq[w] - q0;
    const int nq = left < 256 * ORD_PT ? (int)left : 256 * ORD_PT;
    int2* const quartets = J.q[w];
    unsigned* const kets = J.k[w];
    unsigned char* const bk = J.bk[w];
    if (threadIdx.x < ORD_NB) h[threadIdx.x] = 0;
    if (threadIdx.x < 2) ends[threadIdx.x] = last_le(b.qs, a.nb, threadIdx.x ? q0 + nq - 1 : q0);
    __syncthreads();
    const int i0 = ends[0], ni = ends[1] - i0 + 1;
#pragma unroll 4
    for (int u = 0; u < ORD_PT; ++u) {
        const int t = 256 * u + threadIdx.x;
        const bool ok = t < nq;
        int bucket = 0;
        if (ok) {
            const long long q = q0 + t;
            const int i = i0 + last_le(b.qs + i0, ni, q);
            const int j = b.j0[i] + (int)(q - b.qs[i]), P = a.bra[i], Q = a.ket[j];
            quartets[q] = make_int2(P, Q);
            kets[q] = a.ket_rec[j] | (P == Q ? 1u << 31 : 0u);
            if (bk) {
                bucket = order_bucket(a.pairs[P].n * (int)(a.ket_npcum[j + 1] - a.ket_npcum[j]));
                bk[q] = (unsigned char)bucket;
            }
        }
        if (bk) {
            const unsigned long long m = bucket_peers(bucket, ok);
            if (ok && __ffsll((long long)m) - 1 == (int)(threadIdx.x & 63)) atomicAdd(&h[bucket], __popcll(m));
        }
    }
    __syncthreads();
    if (bk && threadIdx.x < ORD_NB && h[threadIdx.x]) atomicAdd(&cnt[jw * ORD_NB + threadIdx.x], h[threadIdx.x]);
}

// cur[list][bucket] = exclusive scan of the list's bucket counts
__global__ void __launch_bounds__(64) list_order_scan_kernel(const int* cnt, int* cur, int nlist)
{
    for (int j = threadIdx.x; j < nlist; j += blockDim.x) {
        int s = 0;
        for (int k = 0; k < ORD_NB; ++k) {
            cur[j * ORD_NB + k] = s;
            s += cnt[j * ORD_NB + k];
        }
    }
}

// Every quartet takes a slot in its bucket: one global atomic per block and
// bucket reserves the block's range, and within it the quartets keep their
// list order (ranks within a wave by ballots, then a scan over the block's 64
// groups of 64), so that neighbouring slots share a bra as often as they can.
// With the buckets counted and kept by list_fill_batch_kernel the order costs
// C14H30 36 us; counting and filling from the pairs' records took 130.
__global__ void __launch_bounds__(256) list_order_fill_kernel(const ListJob* jobs, const ListBlocks blk, int* cur)
{
    constexpr int NG = ORD_PT * 4, NSEG = 256 / ORD_NB, PER = NG / NSEG;
    __shared__ int c[NG][ORD_NB], part[NSEG][ORD_NB], base[ORD_NB];
    int lb;
    const int jw = order_job_of(blk, lb), w = jw & 1;
    const ListJob& J = jobs[jw >> 1];
    const unsigned char* const bk = J.bk[w];
    int* const ord = J.ord[w];
    const long long nq = J.nq[w];
    if (!bk) return;
    const long long q0 = (long long)lb * 256 * ORD_PT + threadIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int e = threadIdx.x; e < NG * ORD_NB; e += 256) ((int*)c)[e] = 0;
    __syncthreads();
    int bu[ORD_PT], rk[ORD_PT];
#pragma unroll
    for (int u = 0; u < ORD_PT; ++u) {
        const bool ok = q0 + 256 * u < nq;
        bu[u] = ok ? bk[q0 + 256 * u] : -1;
    }
#pragma unroll
    for (int u = 0; u < ORD_PT; ++u) {
        const unsigned long long m = bucket_peers(bu[u] & (ORD_NB - 1), bu[u] >= 0);
        rk[u] = __popcll(m & ((1ULL << lane) - 1));
        if (bu[u] >= 0 && rk[u] == 0) c[4 * u + wave][bu[u]] = __popcll(m);
    }
    __syncthreads();
    const int k = threadIdx.x & (ORD_NB - 1), seg = threadIdx.x / ORD_NB;
    int s = 0;
    for (int g = 0; g < PER; ++g) s += c[seg * PER + g][k];
    part[seg][k] = s;
    __syncthreads();
    int before = 0;
    for (int g = 0; g < seg; ++g) before += part[g][k];
    if (seg == NSEG - 1) base[k] = before + s ? atomicAdd(&cur[jw * ORD_NB + k], before + s) : 0;
    __syncthreads();
    int at = base[k] + before;
    for (int g = 0; g < PER; ++g) {
        const int n = c[seg * PER + g][k];
        c[seg * PER + g][k] = at;
        at += n;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ORD_PT; ++u)
        if (bu[u] >= 0) ord[c[4 * u + wave][bu[u]] + rk[u]] = (int)(q0 + 256 * u);
}

__global__ void __launch_bounds__(256) list_items_count_batch_kernel(const ListJob* jobs, const ListBlocks blk)
{
    int i;
    const int j = list_job_of(blk, i);
    const ListJob& J = jobs[j];
    if (i < J.nb_items)
        J.b64.nit[i] = (J.b64.cnt[i] + (J.has32 ? J.b32.cnt[i] : 0) + J.run - 1) / J.run;
}

__global__ void __launch_bounds__(256) list_items_fill_batch_kernel(const ListJob* jobs, const ListBlocks blk)
{
    int t;
    const int j = list_job_of(blk, t);
    const ListJob& J = jobs[j];
    if (t < J.nitems) list_items_fill_one(J.a, J.b64, J.has32 ? J.b32 : J.b64, t, J.run, J.items, J.items32);
}

// Ket J reduction over tiles of up to 64 consecutive kets (one per lane) x up
// to 256 bras of one molecule (a quarter per wave) x one ket component.  The
// tile's bra data (first quartet minus first ket, ket range, bound) is staged
// in LDS, so that each bra costs one global load per lane: the value of the
// lane's ket under that bra, and neighbouring lanes read neighbouring values.
// The four waves combine in LDS and the tile adds its sums into J' with one
// atomic per ket element.  The bras reaching ket j are re-derived with the
// predicates of list_count_kernel, for kets in descending bound order:
//   FP64: bound_i bound_j > thr and (no split or >= thr32), a prefix of the
//         molecule's bras (bras below j when the lists agree), plus (j|j);
//   FP32: thr < bound_i bound_j < thr32, a contiguous range (no diagonal).
#define JRED_BRAS 256
__device__ __forceinline__ void jket_reduce_tile(const ListArgs& a, const ListBras& b, int w, const double* jkbuf,
                                                 long long nq, int ntiles, int ncd, int n4, const MolInfo* mols,
                                                 double* J, int4 tl, int cd)
{
    __shared__ long long s_base[JRED_BRAS];
    __shared__ double s_bound[JRED_BRAS];
    __shared__ int s_j0[JRED_BRAS], s_cnt[JRED_BRAS];
    __shared__ double part[3][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int cb = tl.z;              // first bra of the tile
    const int nbt = tl.w;             // bras in the tile (<= JRED_BRAS)
    for (int t = threadIdx.x; t < nbt; t += blockDim.x) {
        const int i = cb + t;
        s_j0[t] = b.j0[i];
        s_cnt[t] = (int)b.cnt[i];
        s_base[t] = b.qs[i] - b.j0[i];
        s_bound[t] = a.bra_bound[i];
    }
    __syncthreads();
    const int j = tl.x + lane;
    const bool valid = lane < tl.y;
    double sum = 0.0;
    const int Q = valid ? a.ket[j] : 0;
    const PairHdr kh = a.pairs[Q];
    if (valid) {
        const double qk = a.bound[Q];
        // this wave's bras, as tile-local indices
        const int w0 = wv * (JRED_BRAS / 4);
        const int lo = max(a.bra_seg[kh.mol] - cb, w0);
        const int hi = min(min(a.bra_seg[kh.mol + 1] - cb, w0 + JRED_BRAS / 4), nbt);
        const int hnd = a.same ? min(hi, j - cb) : hi;   // non-diagonal bras
        const bool split = a.thr32 > 0.0;
        int r0 = lo, r1 = lo;
        if (w == 0) {
            r1 = first_true(lo, hnd, [&](int t) {
                const double est = s_bound[t] * qk;
                return !(est > a.thr) || (split && est < a.thr32);
            });
        } else if (split) {
            r0 = first_true(lo, hnd, [&](int t) { return s_bound[t] * qk < a.thr32; });
            r1 = first_true(r0, hnd, [&](int t) { return !(s_bound[t] * qk > a.thr); });
        }
        const double* col = jkbuf + (size_t)cd * nq + j;
        const size_t tstride = (size_t)ncd * nq;
        auto add = [&](int t) {
            const int k = j - s_j0[t];
            if (k < 0 || k >= s_cnt[t]) return;   // never taken: the predicates match the counts
            const double* p = col + s_base[t];
            for (int tt = 0; tt < ntiles; ++tt) sum += p[(size_t)tt * tstride];
        };
        // eight bras at a time with no branch between their loads, so that the
        // eight loads are in flight together: a bra past the range (or one
        // whose run missed the ket, which the predicates rule out) reads
        // jkbuf[0], always in bounds, and contributes zero
        for (int t0 = r0; t0 < r1; t0 += 8) {
            const double* p[8];
            bool ok[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = min(t0 + u, r1 - 1);
                const int k = j - s_j0[t];
                ok[u] = t0 + u < r1 && k >= 0 && k < s_cnt[t];
                p[u] = ok[u] ? col + s_base[t] : jkbuf;
            }
            for (int tt = 0; tt < ntiles; ++tt) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = p[u][(size_t)tt * tstride];
#pragma unroll
                for (int u = 0; u < 8; ++u) sum += ok[u] ? v[u] : 0.0;
            }
        }
        if (w == 0 && a.same && j - cb >= lo && j - cb < hi) add(j - cb);
    }
    if (wv > 0) part[wv - 1][lane] = sum;
    __syncthreads();
    if (wv == 0 && valid) {
        sum += part[0][lane] + part[1][lane] + part[2][lane];
        if (sum != 0.0) {
            const MolInfo mi = mols[kh.mol];
            const int c = cd / n4, d = cd - (cd / n4) * n4;
            const int o3 = a.cart_off[kh.s1], o4 = a.cart_off[kh.s2];
            atomic_addd(&J[mi.base + (size_t)(o3 + c) * mi.n + o4 + d], sum);
        }
    }
}

__global__ void __launch_bounds__(256) jket_reduce_kernel(const JredList L, const MolInfo* mols, double* J)
{
    const int t = blockIdx.x % L.ntile, cd = blockIdx.x / L.ntile;
    jket_reduce_tile(L.a, L.b, L.w, L.jkbuf, L.nq, L.ntiles, L.ncd, L.n4, mols, J, L.tiles[t], cd);
}

// A run of the table's lists in one launch: block -> list by their first-block
// offsets (a handful of entries, scanned by every thread alike).
__global__ void __launch_bounds__(256) jket_reduce_all_kernel(const JredList* lists, int nlist, const MolInfo* mols,
                                                              double* J)
{
    int c = 0;
    const long long b = blockIdx.x + lists[0].block0;
    while (c + 1 < nlist && lists[c + 1].block0 <= b) ++c;
    const JredList& L = lists[c];
    const long long r = b - L.block0;
    const int t = (int)(r % L.ntile), cd = (int)(r / L.ntile);
    jket_reduce_tile(L.a, L.b, L.w, L.jkbuf, L.nq, L.ntiles, L.ncd, L.n4, mols, J, L.tiles[t], cd);
}

static inline unsigned blocks_of(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

void list_count(const ListArgs& a, const ListBras& b64, const ListBras& b32, hipStream_t st)
{
    if (a.nb > 0) hipLaunchKernelGGL(list_count_kernel, dim3(blocks_of(a.nb, 256)), dim3(256), 0, st, a, b64, b32);
}

void list_scan(const long long* in, long long* out, int n, long long* total, hipStream_t st)
{
    hipLaunchKernelGGL(list_scan_kernel, dim3(1), dim3(1024), 0, st, in, out, n, total);
}

void list_items_count(const ListBras& b64, const ListBras* b32, int nb, long long run, hipStream_t st)
{
    if (nb > 0)
        hipLaunchKernelGGL(list_items_count_kernel, dim3(blocks_of(nb, 256)), dim3(256), 0, st,
                           (const long long*)b64.cnt, b32 ? (const long long*)b32->cnt : (const long long*)nullptr,
                           b64.nit, nb, run);
}

void list_fill(const ListArgs& a, const ListBras& b, long long nq, int2* quartets, unsigned* kets, hipStream_t st)
{
    if (nq > 0) hipLaunchKernelGGL(list_fill_kernel, dim3(blocks_of(nq, 256)), dim3(256), 0, st, a, b, nq, quartets, kets);
}

void list_items_fill(const ListArgs& a, const ListBras& b64, const ListBras* b32, long long nitems, long long run,
                     JkItem* items, int2* items32, hipStream_t st)
{
    if (nitems > 0)
        hipLaunchKernelGGL(list_items_fill_kernel, dim3(blocks_of(nitems, 256)), dim3(256), 0, st, a, b64,
                           b32 ? *b32 : b64, nitems, run, items, b32 ? items32 : (int2*)nullptr);
}

void list_count_batch(const ListJob* jobs, const ListBlocks& blk, hipStream_t st)
{
    if (blk.n > 0 && blk.block0[blk.n] > 0)
        hipLaunchKernelGGL(list_count_batch_kernel, dim3(blk.block0[blk.n]), dim3(256), 0, st, jobs, blk);
}

void list_scan_batch(const ScanJob* jobs, int n, hipStream_t st)
{
    if (n > 0) hipLaunchKernelGGL(list_scan_batch_kernel, dim3(n), dim3(1024), 0, st, jobs);
}

void list_fill_batch(const ListJob* jobs, const ListBlocks& blk, int* cnt, hipStream_t st)
{
    if (blk.n <= 0 || blk.block0[blk.n] <= 0) return;
    hipMemsetAsync(cnt, 0, sizeof(int) * ORD_NB * blk.n, st);
    hipLaunchKernelGGL(list_fill_batch_kernel, dim3(blk.block0[blk.n]), dim3(256), 0, st, jobs, blk, cnt);
}

void list_order_batch(const ListJob* jobs, const ListBlocks& blk, const int* cnt, int* cur, hipStream_t st)
{
    if (blk.n <= 0 || blk.block0[blk.n] <= 0) return;
    hipLaunchKernelGGL(list_order_scan_kernel, dim3(1), dim3(64), 0, st, cnt, cur, blk.n);
    hipLaunchKernelGGL(list_order_fill_kernel, dim3(blk.block0[blk.n]), dim3(256), 0, st, jobs, blk, cur);
}

void list_items_count_batch(const ListJob* jobs, const ListBlocks& blk, hipStream_t st)
{
    if (blk.n > 0 && blk.block0[blk.n] > 0)
        hipLaunchKernelGGL(list_items_count_batch_kernel, dim3(blk.block0[blk.n]), dim3(256), 0, st, jobs, blk);
}

void list_items_fill_batch(const ListJob* jobs, const ListBlocks& blk, hipStream_t st)
{
    if (blk.n > 0 && blk.block0[blk.n] > 0)
        hipLaunchKernelGGL(list_items_fill_batch_kernel, dim3(blk.block0[blk.n]), dim3(256), 0, st, jobs, blk);
}

// Tiles of one list: per molecule, runs of up to 64 kets x 256 bras; with
// bra and ket lists the same only bras up to the tile's last ket; tiles whose
// largest bound product (first bra x first ket, both lists sorted by
// descending bound) cannot pass thr are dropped unless they hold a diagonal.
std::vector<int4> jred_tiles(const std::vector<int>& bra_seg, const std::vector<int>& ket_seg,
                             const std::vector<double>& bra_bound, const std::vector<double>& ket_bound, int same,
                             double thr)
{
    std::vector<int4> out;
    const int nmol = (int)ket_seg.size() - 1;
    for (int m = 0; m < nmol; ++m) {
        const int ks = ket_seg[m], ke = ket_seg[m + 1], bs = bra_seg[m], be = bra_seg[m + 1];
        for (int k0 = ks; k0 < ke; k0 += 64) {
            const int nk = std::min(64, ke - k0);
            for (int b0 = bs; b0 < be; b0 += JRED_BRAS) {
                if (same && b0 > k0 + nk - 1) break;
                const bool diag = same && b0 <= k0 + nk - 1 && b0 + JRED_BRAS - 1 >= k0;
                if (!diag && !(bra_bound[b0] * ket_bound[k0] > thr)) {
                    if (same) continue;   // the diagonal tile is still ahead
                    break;                // later bra chunks are weaker
                }
                out.push_back(make_int4(k0, nk, b0, std::min(JRED_BRAS, be - b0)));
            }
        }
    }
    return out;
}

JredList jred_list(const ListArgs& a, const ListBras& b, int w, const double* jkbuf, long long nq, int ntiles, int ncd,
                   int n4, const int4* tiles, int ntile)
{
    JredList L;
    L.a = a;
    L.b = b;
    L.jkbuf = jkbuf;
    L.nq = nq;
    L.w = w;
    L.ntiles = ntiles;
    L.ncd = ncd;
    L.n4 = n4;
    L.tiles = tiles;
    L.ntile = ntile;
    L.block0 = 0;
    return L;
}

void jket_reduce_all(const JredList* lists_dev, int nlist, long long nblocks, const MolInfo* mols, double* J,
                     hipStream_t st)
{
    if (nlist > 0 && nblocks > 0)
        hipLaunchKernelGGL(jket_reduce_all_kernel, dim3((unsigned)nblocks), dim3(256), 0, st, lists_dev, nlist, mols, J);
}

void jket_reduce(const JredList& L, const MolInfo* mols, double* J, hipStream_t st)
{
    const long long nblocks = (long long)L.ntile * L.ncd;
    if (nblocks > 0 && L.nq > 0)
        hipLaunchKernelGGL(jket_reduce_kernel, dim3((unsigned)nblocks), dim3(256), 0, st, L, mols, J);
}
