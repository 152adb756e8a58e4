// pychem_hip.hip -- MI355X (gfx950) integral + Fock-build engine.
//
// Device side: Boys function, generated Obara-Saika/HGP ERI classes (s..d,
// one thread per contracted shell quartet, primitive loops inside), one-
// electron S/T/V, Schwarz bounds, J/K digestion of the stored screened ERIs,
// dense scatter.  Host side: the C-ABI declared in include/pychem_hip.h.
//
// Data layout in HBM (per basis handle):
//   pairs   PairHdr[npair]          one per shell pair a<=b, primary shell first
//   prims   PrimPair<real>[nprimpair]  P, P-X1, p, 1/(2p), K = c1 c2 (pi/p)^1.5 e^{-ab/p |AB|^2}, beta,
//           Ks = K sqrt(p) (2/sqrt(pi))^(1/2), pad (96 bytes)
//   per ERI class c: quartets int2[nq_c] (bra pair, ket pair), values real[ncomp_c][nq_c]
//   (structure-of-arrays so that consecutive threads store / load consecutive words)
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <thread>
#include <string>
#include <vector>

#include "../../include/pychem_hip.h"
#include "lists.h"
#include "scf.h"
#include "eri_common.h"
#include "eri_dispatch.h"
#include "mp2.h"
#include "mlp.h"


__global__ void boys_test_kernel(const double* T, int n, int mmax, double* out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double F[17];
    switch (mmax) {
#define BCASE(M) case M: boys_eval<M>(T[i], F); break;
        BCASE(0) BCASE(1) BCASE(2) BCASE(3) BCASE(4) BCASE(5) BCASE(6) BCASE(7) BCASE(8)
#undef BCASE
        default: return;
    }
    for (int m = 0; m <= mmax; ++m) out[(size_t)i * (mmax + 1) + m] = F[m];
}


// Zero fill (used instead of hipMemsetAsync so that a captured graph holds
// only kernel nodes).
__global__ void fill_zero_kernel(double* a, long long n, double* b)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        a[i] = 0.0;
        if (b) b[i] = 0.0;
    }
}

// General (not necessarily symmetric) densities, per molecule block:
// Ds = (Dj + Dj^T)/2 (J depends only on the symmetric part, (ab|cd) = (ab|dc))
// and DkT = Dk^T.  blockIdx.y = molecule.
__global__ void jk_general_prep_kernel(const double* Dj, const double* Dk, double* Ds, double* DkT,
                                       const MolInfo* mols)
{
    const MolInfo mi = mols[blockIdx.y];
    const long long nn = (long long)mi.n * mi.n;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < nn; t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(t / mi.n), j = (int)(t - (long long)i * mi.n);
        const long long u = mi.base + t, w = mi.base + (long long)j * mi.n + i;
        Ds[u] = 0.5 * (Dj[u] + Dj[w]);
        DkT[u] = Dk[w];
    }
}

// General-density finish.  The digestion adds, per stored element v =
// (mn|ls) with its degeneracy factor, K'_ml += Dk_ns v, K'_nl += Dk_ms v,
// K'_ms += Dk_nl v, K'_ns += Dk_ml v: the four permutations of (mn|ls) whose
// exchange index pairs run bra -> ket, each reading the density transposed.
// The other four permutations give the transpose of the same sums over Dk^T.
// So with K1' digested from Dk^T and K2' from Dk: K = -(K1' + K2'^T)/2, and
// J = (J' + J'^T)/2 as for symmetric densities.
__global__ void jk_general_finish_kernel(double* J, double* K, const double* K2, const MolInfo* mols)
{
    const MolInfo mi = mols[blockIdx.y];
    const long long nn = (long long)mi.n * mi.n;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < nn; t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(t / mi.n), j = (int)(t - (long long)i * mi.n);
        if (j < i) continue;
        const long long u = mi.base + t, w = mi.base + (long long)j * mi.n + i;
        const double sj = 0.5 * (J[u] + J[w]);
        J[u] = sj;
        J[w] = sj;
        const double ku = -0.5 * (K[u] + K2[w]), kw = -0.5 * (K[w] + K2[u]);
        K[u] = ku;
        K[w] = kw;
    }
}

// J = (J' + J'^T)/2 ; K = -(K' + K'^T)/2 per molecule block (reference sign
// convention for K).  blockIdx.y = molecule.
__global__ void jk_finish_kernel(double* J, double* K, const MolInfo* mols)
{
    const MolInfo mi = mols[blockIdx.y];
    const long long nn = (long long)mi.n * mi.n;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < nn; t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(t / mi.n), j = (int)(t - (long long)i * mi.n);
        if (j < i) continue;
        const long long u = mi.base + t, w = mi.base + (long long)j * mi.n + i;
        if (J) { const double s = 0.5 * (J[u] + J[w]); J[u] = s; J[w] = s; }
        if (K) { const double s = -0.5 * (K[u] + K[w]); K[u] = s; K[w] = s; }
    }
}

// Schwarz: per pair, max over its final-basis functions (m,n) of
// sqrt((mn|mn)), from the Cartesian diagonal quartet block of that pair
// (Methods/hartree_fock.py:244-254).  Spherical d shells use the rows of
// Data/transform_basis.py:8-12 on xx,xy,xz,yy,yz,zz, with the reference's
// Python 2 integer division: its `-1/2` in the last row is -1.
__constant__ double c_dsph[5][6] = {
    {0.86602540378443864676, 0, 0, -0.86602540378443864676, 0, 0},
    {0, 1, 0, 0, 0, 0},
    {0, 0, 1, 0, 0, 0},
    {0, 0, 0, 0, 1, 0},
    {-1.0, 0, 0, -1.0, 0, 1}};

__global__ void schwarz_extract_kernel(const double* vals, const int* pair_ids, int nq, int n1, int n2,
                                       const PairHdr* pairs, const int* spher, double* bound)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nq) return;
    const int nab = n1 * n2;
    const int pid = pair_ids[q];
    const PairHdr h = pairs[pid];
    const int sp1 = spher ? spher[h.s1] : 0, sp2 = spher ? spher[h.s2] : 0;
    double mx = 0.0;
    if (!sp1 && !sp2) {
        for (int ab = 0; ab < nab; ++ab) {
            const double v = vals[(size_t)(ab * nab + ab) * nq + q];
            const double s = sqrt(v > 0.0 ? v : 0.0);
            mx = s > mx ? s : mx;
        }
    } else {
        const int m1 = sp1 ? 5 : n1, m2 = sp2 ? 5 : n2;
        for (int i = 0; i < m1; ++i)
            for (int j = 0; j < m2; ++j) {
                double acc = 0.0;
                for (int a = 0; a < n1; ++a) {
                    const double ta = sp1 ? c_dsph[i][a] : (a == i ? 1.0 : 0.0);
                    if (ta == 0.0) continue;
                    for (int b = 0; b < n2; ++b) {
                        const double tb = sp2 ? c_dsph[j][b] : (b == j ? 1.0 : 0.0);
                        if (tb == 0.0) continue;
                        for (int c = 0; c < n1; ++c) {
                            const double tc = sp1 ? c_dsph[i][c] : (c == i ? 1.0 : 0.0);
                            if (tc == 0.0) continue;
                            for (int d = 0; d < n2; ++d) {
                                const double td = sp2 ? c_dsph[j][d] : (d == j ? 1.0 : 0.0);
                                if (td == 0.0) continue;
                                acc += ta * tb * tc * td * vals[(size_t)((a * n2 + b) * nab + c * n2 + d) * nq + q];
                            }
                        }
                    }
                }
                const double s = sqrt(acc > 0.0 ? acc : 0.0);
                mx = s > mx ? s : mx;
            }
    }
    bound[pid] = mx;
}

// ==========================================================================
// Host side
// ==========================================================================
static thread_local std::string g_err;
static int fail(const std::string& m)
{
    g_err = m;
    return -1;
}
// error path of the library's other translation units
int pq_set_error(const char* m) { return fail(m); }
#define HIPCHK(x)                                                                       \
    do {                                                                                \
        hipError_t e_ = (x);                                                            \
        if (e_ != hipSuccess) return fail(std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

static inline int ncart_l(int l) { return (l + 1) * (l + 2) / 2; }
static inline int pair_class(int l1, int l2) { return l1 * (l1 + 1) / 2 + l2; }   // l1 >= l2

// Device memory cache.  hipFree synchronises the whole device, and a basis
// owns some hundred buffers, so creating and destroying bases (one per SCF,
// one per element for the atomic guesses) would otherwise stall on every
// buffer.  Released blocks go to a per-device pending list; they are handed
// out again only after one device synchronisation done here, the first time
// an allocation finds no free block that fits, so that no block still read or
// written by queued work on any stream is reused.  Sizes are rounded to 1/8
// of their power of two (waste below 12.5 %); a request takes a cached block
// of at most 5/4 its rounded size.  hipMalloc failing releases the cache and
// retries once.  pq_cache_release() returns everything to the driver; blocks
// still cached at exit are left to the driver.  PQ_DEVICE_CACHE=0 in the
// environment turns the cache off (plain hipMalloc / hipFree per buffer).
namespace {
constexpr int kCacheDevices = 64;
struct DevCache {
    std::mutex mu;
    std::multimap<size_t, void*> avail[kCacheDevices], pending[kCacheDevices];
    size_t held[kCacheDevices] = {};   // bytes cached (avail + pending)
};
DevCache& dev_cache()
{
    static DevCache* c = new DevCache();   // never destroyed: no HIP calls at exit
    return *c;
}
size_t cache_round(size_t b)
{
    if (b <= 512) return 512;
    size_t p = 1;
    while (p * 2 <= b) p *= 2;              // largest power of two <= b
    const size_t g = p >= 4096 ? p / 8 : 512;
    return (b + g - 1) / g * g;
}
void* cache_take(std::multimap<size_t, void*>& m, size_t rb, size_t* got)
{
    auto it = m.lower_bound(rb);
    if (it == m.end() || it->first > rb + rb / 4) return nullptr;
    void* p = it->second;
    *got = it->first;
    m.erase(it);
    return p;
}
bool cache_enabled()
{
    static const bool on = [] {
        const char* e = getenv("PQ_DEVICE_CACHE");
        return !(e && e[0] == '0');
    }();
    return on;
}
void cache_drop_all(DevCache& c, int dev)
{
    for (auto* m : {&c.avail[dev], &c.pending[dev]}) {
        for (auto& kv : *m) (void)hipFree(kv.second);
        m->clear();
    }
    c.held[dev] = 0;
}
}  // namespace

static int dev_alloc(size_t b, void** out, size_t* cap, int* dev_out)
{
    *out = nullptr;
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kCacheDevices) return fail("device memory cache: device index out of range");
    if (!cache_enabled()) {
        void* p = nullptr;
        const hipError_t e = hipMalloc(&p, b);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return fail(std::string("hipMalloc: ") + hipGetErrorString(e));
        }
        *out = p;
        *cap = b;
        *dev_out = dev;
        return 0;
    }
    const size_t rb = cache_round(b);
    DevCache& c = dev_cache();
    std::lock_guard<std::mutex> lk(c.mu);
    size_t got = 0;
    void* p = cache_take(c.avail[dev], rb, &got);
    if (!p && !c.pending[dev].empty()) {
        auto it = c.pending[dev].lower_bound(rb);
        if (it != c.pending[dev].end() && it->first <= rb + rb / 4) {
            HIPCHK(hipDeviceSynchronize());
            c.avail[dev].insert(c.pending[dev].begin(), c.pending[dev].end());
            c.pending[dev].clear();
            p = cache_take(c.avail[dev], rb, &got);
        }
    }
    if (p) {
        c.held[dev] -= got;
        *out = p;
        *cap = got;
        *dev_out = dev;
        return 0;
    }
    hipError_t e = hipMalloc(&p, rb);
    if (e == hipErrorOutOfMemory && c.held[dev]) {
        (void)hipGetLastError();
        HIPCHK(hipDeviceSynchronize());
        cache_drop_all(c, dev);
        e = hipMalloc(&p, rb);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(std::string("hipMalloc: ") + hipGetErrorString(e));
    }
    *out = p;
    *cap = rb;
    *dev_out = dev;
    return 0;
}

static void dev_release(void* p, size_t cap, int dev)
{
    if (!p) return;
    if (!cache_enabled()) {
        (void)hipFree(p);
        return;
    }
    DevCache& c = dev_cache();
    std::lock_guard<std::mutex> lk(c.mu);
    c.pending[dev].insert({cap, p});
    c.held[dev] += cap;
}

// Free every cached block of the current device (synchronises the device).
extern "C" int pq_cache_release(void)
{
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kCacheDevices) return fail("pq_cache_release: device index out of range");
    DevCache& c = dev_cache();
    std::lock_guard<std::mutex> lk(c.mu);
    HIPCHK(hipDeviceSynchronize());
    cache_drop_all(c, dev);
    return 0;
}

// Bytes of device memory the cache holds on the current device.
extern "C" long long pq_cache_bytes(void)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kCacheDevices) return -1;
    DevCache& c = dev_cache();
    std::lock_guard<std::mutex> lk(c.mu);
    return (long long)c.held[dev];
}

// A device buffer that grows on demand (contents are not kept when it grows).
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;   // capacity of the block
    int dev = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { release(); }
    int ensure(size_t b)
    {
        if (b <= bytes && p) return 0;
        release();
        if (b == 0) return 0;
        return dev_alloc(b, &p, &bytes, &dev);
    }
    void release()
    {
        dev_release(p, bytes, dev);
        p = nullptr;
        bytes = 0;
    }
};

struct EriClassStore {
    DevBuf q, vals, items, items32, kets, jkbuf;   // items, items32: class level, in store64
    DevBuf order;                                  // the ERI kernels' quartet order (list_order_batch)
    const int4* jtiles = nullptr;   // the list's ket J reduction tiles (in the basis's d_jtiles)
    int njtile = 0;
    // per bra of the class's bra list (see lists.h)
    DevBuf j0, cnt, np, qs, nit, its;
    int nitems = 0;
    int jk_run = 0;            // J/K work-item length (0: automatic)
    int jk_grid = 0;           // J/K blocks launched (0: one per item)
    int nq = 0;
    int ncomp = 0;
    int is32 = 0;              // values stored as float
    long long nprimq = 0;      // primitive quartets (kept primitive pairs)
};

struct pq_basis {
    int nshell = 0, natom = 0, ncart = 0, npair = 0, nprimpair = 0;
    int nmol = 1, nmax = 0;                 // molecules; largest per-molecule ncart
    long long mat_total = 0;                // packed matrix elements, sum of n_m^2
    std::vector<MolInfo> mols;
    std::vector<int> shell_mol;
    std::vector<int> l, nprim, cart_off;    // cart_off: local to the shell's molecule
    std::vector<double> center, atoms;
    std::vector<PairHdr> pairs;
    // pair id of two shells of one molecule (both orders): per molecule a
    // table over its own shells, [mol_pair_off + (s1 - shell0) * ns + (s2 - shell0)]
    std::vector<int> pair_local;
    std::vector<long long> mol_pair_off;
    std::vector<int> mol_shell0, mol_nshell;
    std::vector<std::vector<int>> class_pairs;   // pair ids per pair class
    int class_nmax[6] = {};                      // most primitive pairs of a pair of the class
    std::vector<double> bound;              // per pair Schwarz bound
    int have_bound = 0;
    // two-electron operator of the class kernels: 0 Coulomb, 1 electron
    // scattering at momentum transfer op_S (pq_eri_set_operator)
    int op = 0;
    double op_S = 0.0;
    // per pair class: pair ids sorted by (molecule, bound desc), molecule
    // segment starts, cumulative primitive-pair counts (device)
    // per pair class: sorted pair ids, molecule segments, cumulative
    // primitive-pair counts and sorted bounds, all in one device buffer
    // (d_sortpack, one upload of hsortpack per plan)
    DevBuf d_sortpack, d_total;
    const int* p_sorted[6] = {};
    const int* p_seg[6] = {};
    const long long* p_npcum[6] = {};
    const unsigned* p_rec[6] = {};
    const double* p_sbound[6] = {};
    std::vector<char> hsortpack;
    std::vector<int> hseg[6], hsorted[6];    // host copies of what the device lists read
    std::vector<double> hsbound[6];
    std::vector<long long> hnpcum[6];
    // batched list construction: job tables (device) and the host copies of
    // every upload of the current plan (kept until the next plan)
    DevBuf d_jobs, d_scans, d_jtiles;
    DevBuf d_order_cnt;                     // list_order_batch counts and cursors
    int eri_order = 1;                      // ERI kernels visit quartets by descending primitive work
    std::vector<std::vector<ListJob>> hjobs;
    std::vector<std::vector<ScanJob>> hscans;
    std::vector<int4> hjtiles_all;
    // every tiled list's ket J reduction, launched once per J/K call
    DevBuf d_jred;
    DevBuf d_jkgen;          // pq_jk_general scratch: symmetrised Dj, Dk^T, J2', K2'
    std::vector<JredList> hjred;
    // ket J reductions, in d_jred launch group by launch group: lists and
    // blocks before group g
    int jred_list0[JK_NGROUP + 1] = {};
    long long jred_block0[JK_NGROUP + 1] = {};
    int nsorted[6] = {};
    DevBuf d_pairbase, d_pairtab;           // packed function pairs of the MP2 transform (ensure_pair_table)
    int npacked = 0;
    DevBuf d_pairs, d_prims, d_atoms, d_cart_off, d_bound, d_tmp_list, d_spher, d_mols;
    int any_spher = 0;
    EriClassStore store64[ERI_NCLASS], store32[ERI_NCLASS];
    double threshold = 1e-8, threshold32 = 0.0;
    // optional live timing (hipEvents on the caller's stream)
    int timing = 0;
    hipEvent_t ev_cls[2 * ERI_NCLASS][2] = {};
    int ev_cls_used[2 * ERI_NCLASS] = {};
    hipEvent_t ev_jk[2] = {};
    int ev_jk_used = 0;
    hipEvent_t ev_pass[2] = {};   // whole ERI pass on the caller's stream
    int ev_pass_used = 0;
    // per-class J/K digestion times (timing on), on the device: per class the
    // current call's first block start and last block end, then the sum of
    // the spans and the number of calls, in ticks of the realtime clock
    DevBuf d_jkclock;
    hipGraphExec_t graph_exec = nullptr;
    // Class launches fan out over side streams (default priority); with the
    // caller's stream, four streams fill the process's four hardware queues.
    // J/K: jk_nstreams streams, the caller's one of them (C20H42: 1.18 ms on
    // one, 1.12 on four).  Schwarz and ERI passes: eri_nstreams side
    // streams beside the caller's, which runs the classes that use scratch.
    int jk_nstreams = 4;
    int eri_nstreams = 3;
    hipStream_t jk_side[4] = {};
    hipEvent_t ev_fork = nullptr, ev_join[4] = {};
};

// The ERI kernels of a class visit its quartets by descending primitive work
// (list_order_batch) when a quartet has at most this many output components:
// measured on C10H22/6-31G*, the ERI pass went from 2.40 to 2.00 ms, the
// classes with narrow outputs gaining most; the wide classes ((dd|dp),
// (dp|dp), (dd|pp), (dd|ds): 216 components and more) lost a few per cent,
// their scattered stores costing more than the divergence saved.
#define ORDER_MAX_NCOMP 200
static inline bool uses_order(const pq_basis* b, const EriClassStore& s)
{
    return b->eri_order && s.nq > 0 && s.ncomp <= ORDER_MAX_NCOMP;
}
// The quartet order the ERI kernels follow for a list (NULL: list order).
static inline const int* order_of(const pq_basis* b, const EriClassStore& s)
{
    return uses_order(b, s) ? (const int*)s.order.p : nullptr;
}

static int ensure_jk_streams(pq_basis* b)
{
    if (b->ev_fork) return 0;
    for (int k = 0; k < 4; ++k) {
        HIPCHK(hipStreamCreateWithFlags(&b->jk_side[k], hipStreamNonBlocking));
        HIPCHK(hipEventCreateWithFlags(&b->ev_join[k], hipEventDisableTiming));
    }
    HIPCHK(hipEventCreateWithFlags(&b->ev_fork, hipEventDisableTiming));
    return 0;
}

static int ensure_events(pq_basis* b)
{
    if (b->ev_jk[0]) return 0;
    for (int i = 0; i < 2 * ERI_NCLASS; ++i)
        for (int k = 0; k < 2; ++k) HIPCHK(hipEventCreate(&b->ev_cls[i][k]));
    HIPCHK(hipEventCreate(&b->ev_jk[0]));
    HIPCHK(hipEventCreate(&b->ev_jk[1]));
    HIPCHK(hipEventCreate(&b->ev_pass[0]));
    HIPCHK(hipEventCreate(&b->ev_pass[1]));
    return 0;
}

// Per class (a block of one wave, a lane per slot): the call's span (set = 0:
// empty it; 1: add it to the sums; 2: clear everything).  The sums lie behind
// the slots.
#define JK_CLOCK_SUMS (2 * JK_CLOCK_SLOTS * JK_CLOCK_CLASSES)
static_assert(ERI_NCLASS <= JK_CLOCK_CLASSES && JK_CLOCK_SLOTS == 64, "one wave per class");
__global__ void __launch_bounds__(64) jk_clock_kernel(unsigned long long* clock, int set)
{
    const int c = blockIdx.x;
    unsigned long long* at = clock + jk_clock_at(threadIdx.x, c);
    unsigned long long lo = at[0], hi = at[1];
    at[0] = ~0ULL;
    at[1] = 0;
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long l = __shfl_xor(lo, o, 64), h = __shfl_xor(hi, o, 64);
        lo = l < lo ? l : lo;
        hi = h > hi ? h : hi;
    }
    if (threadIdx.x) return;
    unsigned long long* sum = clock + JK_CLOCK_SUMS + 2 * c;
    if (set == 2) sum[0] = sum[1] = 0;
    if (set == 1 && hi > lo) {
        sum[0] += hi - lo;
        sum[1] += 1;
    }
}

static void jk_clock_set(pq_basis* b, int set, hipStream_t st)
{
    if (b->timing && b->d_jkclock.p)
        hipLaunchKernelGGL(jk_clock_kernel, dim3(ERI_NCLASS), dim3(64), 0, st, (unsigned long long*)b->d_jkclock.p, set);
}

extern "C" const char* pq_last_error(void) { return g_err.c_str(); }

extern "C" int pq_version(void) { return 1; }

extern "C" int pq_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

extern "C" int pq_boys(int n, const double* T_dev, int mmax, double* out_dev, void* stream)
{
    if (mmax < 0 || mmax > 8) return fail("pq_boys: mmax must be in 0..8");
    if (n <= 0) return 0;
    hipLaunchKernelGGL(boys_test_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, T_dev, n, mmax,
                       out_dev);
    HIPCHK(hipGetLastError());
    return 0;
}

extern "C" void pq_basis_destroy(pq_basis* b);

// Batched basis: nmol molecules, shells and atoms grouped by molecule
// (shell_mol / atom_mol non-decreasing).  Pairs and quartets never mix
// molecules; matrices are packed per-molecule blocks.
// Pair id of shells sa, sb, or -1 when they belong to different molecules.
static int pair_id(const pq_basis* b, int sa, int sb)
{
    const int m = b->shell_mol[sa];
    if (b->shell_mol[sb] != m) return -1;
    const int s0 = b->mol_shell0[m], ns = b->mol_nshell[m];
    return b->pair_local[(size_t)(b->mol_pair_off[m] + (long long)(sa - s0) * ns + (sb - s0))];
}

// Host loops over independent items on up to eight threads (one for fewer
// than 256 items); blocks of 64 items are handed out in order.
template <typename F>
static void host_parallel_for(int n, F f)
{
    const int hw = (int)std::thread::hardware_concurrency();
    const int nt = n < 256 ? 1 : std::max(1, std::min(8, hw));
    if (nt == 1) {
        for (int i = 0; i < n; ++i) f(i);
        return;
    }
    std::atomic<int> next(0);
    auto work = [&]() {
        for (;;) {
            const int i0 = next.fetch_add(64);
            if (i0 >= n) break;
            const int i1 = std::min(n, i0 + 64);
            for (int i = i0; i < i1; ++i) f(i);
        }
    };
    std::vector<std::thread> th;
    for (int t = 1; t < nt; ++t) th.emplace_back(work);
    work();
    for (auto& x : th) x.join();
}

// Pinned host staging of the primitive-pair upload (a pageable copy of the
// ~10 MB of C20H42's records took about a millisecond): grown on demand,
// held until the process ends, one basis construction at a time.
static std::mutex g_prim_stage_mu;
static void* g_prim_stage = nullptr;
static size_t g_prim_stage_bytes = 0;
static void* prim_stage(size_t bytes)
{
    if (bytes > g_prim_stage_bytes) {
        if (g_prim_stage) hipHostFree(g_prim_stage);
        g_prim_stage = nullptr;
        g_prim_stage_bytes = 0;
        const size_t want = std::max(bytes, (size_t)1 << 20);
        if (hipHostMalloc(&g_prim_stage, want, hipHostMallocDefault) != hipSuccess) return nullptr;
        g_prim_stage_bytes = want;
    }
    return g_prim_stage;
}

extern "C" int pq_basis_create_batch(int nmol, int nshell, const int* l, const int* nprim, const int* prim_off,
                                     const double* center, const double* exps, const double* cc,
                                     const int* shell_mol, int natom, const double* atom_xyz, const double* atom_z,
                                     const int* atom_mol, pq_basis** out)
{
    if (!out) return fail("pq_basis_create: null output");
    *out = nullptr;
    if (nshell <= 0 || nmol <= 0) return fail("pq_basis_create: nshell and nmol must be positive");
    for (int s = 0; s < nshell; ++s) {
        if (l[s] < 0 || l[s] > 2) return fail("pq_basis_create: only s, p, d shells are supported");
        if (nprim[s] <= 0 || nprim[s] > 64) return fail("pq_basis_create: bad primitive count");
        const int m = shell_mol ? shell_mol[s] : 0;
        if (m < 0 || m >= nmol || (s > 0 && shell_mol && shell_mol[s] < shell_mol[s - 1]))
            return fail("pq_basis_create: shells must be grouped by molecule");
    }
    for (int a = 0; a < natom; ++a) {
        const int m = atom_mol ? atom_mol[a] : 0;
        if (m < 0 || m >= nmol || (a > 0 && atom_mol && atom_mol[a] < atom_mol[a - 1]))
            return fail("pq_basis_create: atoms must be grouped by molecule");
    }
    pq_basis* b = new pq_basis();
    b->nshell = nshell;
    b->natom = natom;
    b->nmol = nmol;
    b->l.assign(l, l + nshell);
    b->nprim.assign(nprim, nprim + nshell);
    b->center.assign(center, center + 3 * nshell);
    b->shell_mol.resize(nshell);
    for (int s = 0; s < nshell; ++s) b->shell_mol[s] = shell_mol ? shell_mol[s] : 0;
    b->cart_off.resize(nshell);
    b->mols.assign(nmol, MolInfo{0, 0, 0, 0, 0});
    for (int s = 0; s < nshell; ++s) {
        MolInfo& mi = b->mols[b->shell_mol[s]];
        b->cart_off[s] = mi.n;
        mi.n += ncart_l(l[s]);
    }
    for (int m = 0; m < nmol; ++m) { b->mols[m].atom_lo = natom; b->mols[m].atom_hi = 0; }
    for (int a = 0; a < natom; ++a) {
        MolInfo& mi = b->mols[atom_mol ? atom_mol[a] : 0];
        mi.atom_lo = std::min(mi.atom_lo, a);
        mi.atom_hi = std::max(mi.atom_hi, a + 1);
    }
    long long base = 0;
    b->ncart = 0;
    for (int m = 0; m < nmol; ++m) {
        MolInfo& mi = b->mols[m];
        if (mi.atom_hi <= mi.atom_lo) { mi.atom_lo = 0; mi.atom_hi = 0; }
        mi.base = base;
        base += (long long)mi.n * mi.n;
        b->ncart += mi.n;
        b->nmax = std::max(b->nmax, mi.n);
    }
    b->mat_total = base;
    b->atoms.resize(4 * (size_t)std::max(natom, 1));
    for (int a = 0; a < natom; ++a) {
        for (int i = 0; i < 3; ++i) b->atoms[4 * a + i] = atom_xyz[3 * a + i];
        b->atoms[4 * a + 3] = atom_z[a];
    }
    // shell pairs a <= b within a molecule, primary = larger l (first on ties);
    // primitive-pair quantities as Methods/c_ints/shellpair_quantities.c:28-33
    b->mol_shell0.assign(nmol, 0);
    b->mol_nshell.assign(nmol, 0);
    b->mol_pair_off.assign(nmol, 0);
    for (int s = nshell - 1; s >= 0; --s) {
        b->mol_shell0[b->shell_mol[s]] = s;
        b->mol_nshell[b->shell_mol[s]] += 1;
    }
    {
        long long tot = 0;
        for (int m = 0; m < nmol; ++m) {
            b->mol_pair_off[m] = tot;
            tot += (long long)b->mol_nshell[m] * b->mol_nshell[m];
        }
        b->pair_local.assign((size_t)tot, -1);
    }
    b->class_pairs.assign(6, {});
    const double PI = 3.14159265358979323846;
    {
        long long np = 0, npp = 0;   // upper bounds: every pair of one molecule
        std::vector<long long> ps(nmol, 0), pn(nmol, 0);
        for (int s = 0; s < nshell; ++s) {
            ps[b->shell_mol[s]] += nprim[s];
            pn[b->shell_mol[s]] += 1;
        }
        for (int m = 0; m < nmol; ++m) {
            np += pn[m] * (pn[m] + 1) / 2;
            npp += ps[m] * ps[m];
        }
        b->pairs.reserve((size_t)np);
        (void)npp;
    }
    // Shell pairs in (sa, sb) order; then, over the pairs in parallel, the
    // kept primitive pairs of each (pass 1: overlap factors and counts),
    // their offsets, and the records written in place (pass 2) into pinned
    // host memory for the upload.  The output does not depend on the thread
    // count.
    std::vector<int2> plist;
    plist.reserve(b->pairs.capacity());
    for (int sa = 0; sa < nshell; ++sa)
        for (int sb = sa; sb < nshell; ++sb) {
            if (b->shell_mol[sb] != b->shell_mol[sa]) break;   // grouped: later shells are other molecules
            plist.push_back(make_int2(sa, sb));
        }
    const int npl = (int)plist.size();
    std::vector<long long> kofs(npl + 1, 0);   // overlap-factor slots per pair (all primitive pairs)
    for (int t = 0; t < npl; ++t) kofs[t + 1] = kofs[t] + (long long)nprim[plist[t].x] * nprim[plist[t].y];
    std::vector<double> Kv((size_t)std::max(1LL, kofs[npl]));
    std::vector<int> kept(npl + 1, 0);
    b->pairs.resize(npl);
    auto primary = [&](int t, int& s1, int& s2) {
        s1 = plist[t].x;
        s2 = plist[t].y;
        if (l[s2] > l[s1]) std::swap(s1, s2);
    };
    host_parallel_for(npl, [&](int t) {
        int s1, s2;
        primary(t, s1, s2);
        double ab2 = 0.0;
        for (int i = 0; i < 3; ++i) {
            const double d = center[3 * s1 + i] - center[3 * s2 + i];
            ab2 += d * d;
        }
        double* K = Kv.data() + kofs[t];
        int n = 0;
        for (int i1 = 0; i1 < nprim[s1]; ++i1)
            for (int i2 = 0; i2 < nprim[s2]; ++i2) {
                const double a1 = exps[prim_off[s1] + i1], a2 = exps[prim_off[s2] + i2];
                const double p = a1 + a2, sig = 1.0 / p;
                const double q = PI * sig;   // (pi / p)^(3/2) = q sqrt(q)
                const double k = cc[prim_off[s1] + i1] * cc[prim_off[s2] + i2] * (q * sqrt(q)) *
                                 exp(-a1 * a2 * sig * ab2);
                K[i1 * nprim[s2] + i2] = k;
                // primitive pairs whose overlap factor underflows contribute nothing
                if (!(fabs(k) < 1e-30)) ++n;
            }
        kept[t] = n;
    });
    std::vector<long long> pofs(npl + 1, 0);
    for (int t = 0; t < npl; ++t) pofs[t + 1] = pofs[t] + kept[t];
    const long long nprims = pofs[npl];
    if (nprims > 0x7fffffffLL) { pq_basis_destroy(b); return fail("pq_basis_create: too many primitive pairs"); }
    std::unique_lock<std::mutex> stage_lock(g_prim_stage_mu);
    PrimPair<double>* stage = (PrimPair<double>*)prim_stage(sizeof(PrimPair<double>) * (size_t)std::max(1LL, nprims));
    if (!stage) { pq_basis_destroy(b); return fail("pq_basis_create: pinned staging allocation failed"); }
    host_parallel_for(npl, [&](int t) {
        int s1, s2;
        primary(t, s1, s2);
        PairHdr& h = b->pairs[t];
        h.s1 = s1;
        h.s2 = s2;
        h.pcls = pair_class(l[s1], l[s2]);
        h.mol = b->shell_mol[plist[t].x];
        for (int i = 0; i < 3; ++i) h.ab[i] = center[3 * s1 + i] - center[3 * s2 + i];
        h.off = (int)pofs[t];
        h.n = kept[t];
        const double* K = Kv.data() + kofs[t];
        PrimPair<double>* out = stage + pofs[t];
        for (int i1 = 0; i1 < nprim[s1]; ++i1)
            for (int i2 = 0; i2 < nprim[s2]; ++i2) {
                const double k = K[i1 * nprim[s2] + i2];
                if (fabs(k) < 1e-30) continue;
                const double a1 = exps[prim_off[s1] + i1], a2 = exps[prim_off[s2] + i2];
                const double p = a1 + a2, sig = 1.0 / p;
                PrimPair<double> pp;
                pp.Px = (a1 * center[3 * s1] + a2 * center[3 * s2]) * sig;
                pp.Py = (a1 * center[3 * s1 + 1] + a2 * center[3 * s2 + 1]) * sig;
                pp.Pz = (a1 * center[3 * s1 + 2] + a2 * center[3 * s2 + 2]) * sig;
                pp.PAx = pp.Px - center[3 * s1];
                pp.PAy = pp.Py - center[3 * s1 + 1];
                pp.PAz = pp.Pz - center[3 * s1 + 2];
                pp.p = p;
                pp.inv2p = 0.5 * sig;
                pp.K = k;
                pp.beta = a2;
                pp.Ks = k * sqrt(p) * 1.0622519320271968;   // (2/sqrt(pi))^(1/2)
                pp.pad = 0.0;
                *out++ = pp;
            }
    });
    for (int t = 0; t < npl; ++t) {
        const int sa = plist[t].x, sb = plist[t].y;
        const int m = b->shell_mol[sa], s0 = b->mol_shell0[m], ns = b->mol_nshell[m];
        b->pair_local[(size_t)(b->mol_pair_off[m] + (long long)(sa - s0) * ns + (sb - s0))] = t;
        b->pair_local[(size_t)(b->mol_pair_off[m] + (long long)(sb - s0) * ns + (sa - s0))] = t;
        b->class_pairs[b->pairs[t].pcls].push_back(t);
        b->class_nmax[b->pairs[t].pcls] = std::max(b->class_nmax[b->pairs[t].pcls], b->pairs[t].n);
    }
    b->npair = (int)b->pairs.size();
    b->nprimpair = (int)nprims;
    int rc = 0;
    rc |= b->d_pairs.ensure(sizeof(PairHdr) * b->pairs.size());
    rc |= b->d_prims.ensure(sizeof(PrimPair<double>) * std::max<size_t>(1, (size_t)nprims));
    rc |= b->d_atoms.ensure(sizeof(double) * b->atoms.size());
    rc |= b->d_cart_off.ensure(sizeof(int) * nshell);
    rc |= b->d_bound.ensure(sizeof(double) * b->pairs.size());
    rc |= b->d_mols.ensure(sizeof(MolInfo) * nmol);
    if (rc) { pq_basis_destroy(b); return -1; }
    hipError_t e = hipSuccess;
    e = hipMemcpy(b->d_pairs.p, b->pairs.data(), sizeof(PairHdr) * b->pairs.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && nprims > 0)
        e = hipMemcpy(b->d_prims.p, stage, sizeof(PrimPair<double>) * (size_t)nprims, hipMemcpyHostToDevice);
    stage_lock.unlock();
    if (e == hipSuccess) e = hipMemcpy(b->d_atoms.p, b->atoms.data(), sizeof(double) * b->atoms.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(b->d_cart_off.p, b->cart_off.data(), sizeof(int) * nshell, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(b->d_mols.p, b->mols.data(), sizeof(MolInfo) * nmol, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        pq_basis_destroy(b);
        return fail(std::string("pq_basis_create: copy failed: ") + hipGetErrorString(e));
    }
    for (int c = 0; c < ERI_NCLASS; ++c) {
        b->store64[c].ncomp = b->store32[c].ncomp = eri_class_table[c][4];
        b->store32[c].is32 = 1;
    }
    *out = b;
    return 0;
}

extern "C" int pq_basis_create(int nshell, const int* l, const int* nprim, const int* prim_off, const double* center,
                               const double* exps, const double* cc, int natom, const double* atom_xyz,
                               const double* atom_z, pq_basis** out)
{
    return pq_basis_create_batch(1, nshell, l, nprim, prim_off, center, exps, cc, nullptr, natom, atom_xyz, atom_z,
                                 nullptr, out);
}

extern "C" void pq_basis_destroy(pq_basis* b)
{
    if (!b) return;
    for (int c = 0; c < ERI_NCLASS; ++c) {
        b->store64[c].q.release(); b->store64[c].vals.release(); b->store64[c].items.release();
        b->store32[c].q.release(); b->store32[c].vals.release(); b->store32[c].items.release();
        for (int w = 0; w < 2; ++w) {
            EriClassStore& t = w ? b->store32[c] : b->store64[c];
            t.kets.release(); t.jkbuf.release(); t.j0.release(); t.cnt.release(); t.np.release();
            t.qs.release(); t.nit.release(); t.its.release();
        }
    }
    b->d_sortpack.release();
    b->d_pairs.release(); b->d_prims.release(); b->d_atoms.release();
    b->d_cart_off.release(); b->d_bound.release(); b->d_tmp_list.release(); b->d_spher.release();
    b->d_mols.release(); b->d_total.release(); b->d_jred.release(); b->d_jkgen.release();
    if (b->graph_exec) (void)hipGraphExecDestroy(b->graph_exec);
    if (b->ev_jk[0]) {
        for (int i = 0; i < 2 * ERI_NCLASS; ++i)
            for (int k = 0; k < 2; ++k) (void)hipEventDestroy(b->ev_cls[i][k]);
        (void)hipEventDestroy(b->ev_jk[0]);
        (void)hipEventDestroy(b->ev_jk[1]);
        (void)hipEventDestroy(b->ev_pass[0]);
        (void)hipEventDestroy(b->ev_pass[1]);
    }
    if (b->ev_fork) {
        for (int k = 0; k < 4; ++k) {
            (void)hipStreamDestroy(b->jk_side[k]);
            (void)hipEventDestroy(b->ev_join[k]);
        }
        (void)hipEventDestroy(b->ev_fork);
    }
    delete b;
}

extern "C" int pq_basis_set_spherical(pq_basis* b, const int* spher)
{
    if (!b || !spher) return fail("pq_basis_set_spherical: null argument");
    int any = 0;
    for (int s = 0; s < b->nshell; ++s) {
        if (spher[s] && b->l[s] != 2) return fail("pq_basis_set_spherical: only d shells have a spherical form here");
        any |= spher[s] ? 1 : 0;
    }
    if (b->d_spher.ensure(sizeof(int) * b->nshell)) return -1;
    HIPCHK(hipMemcpy(b->d_spher.p, spher, sizeof(int) * b->nshell, hipMemcpyHostToDevice));
    b->any_spher = any;
    b->have_bound = 0;
    return 0;
}

extern "C" int pq_basis_info(const pq_basis* b, long long* info)
{
    if (!b || !info) return fail("pq_basis_info: null argument");
    info[0] = b->ncart;
    info[1] = b->nshell;
    info[2] = b->npair;
    info[3] = b->nprimpair;
    info[4] = b->nmol;
    info[5] = b->mat_total;
    info[6] = b->nmax;
    return 0;
}

// Per molecule: base (packed offset), n (Cartesian functions), atom range.
extern "C" int pq_basis_molecules(const pq_basis* b, long long* base, int* n, int* atom_lo, int* atom_hi)
{
    if (!b) return fail("pq_basis_molecules: null basis");
    for (int m = 0; m < b->nmol; ++m) {
        if (base) base[m] = b->mols[m].base;
        if (n) n[m] = b->mols[m].n;
        if (atom_lo) atom_lo[m] = b->mols[m].atom_lo;
        if (atom_hi) atom_hi[m] = b->mols[m].atom_hi;
    }
    return 0;
}

extern "C" int pq_one_electron(pq_basis* b, double* S, double* T, double* V, void* stream)
{
    if (!b || !S || !T || !V) return fail("pq_one_electron: null argument");
    hipStream_t st = (hipStream_t)stream;
    std::vector<int> all;
    std::vector<int> offs(7, 0);
    for (int c = 0; c < 6; ++c) {
        offs[c] = (int)all.size();
        all.insert(all.end(), b->class_pairs[c].begin(), b->class_pairs[c].end());
    }
    offs[6] = (int)all.size();
    if (b->d_tmp_list.ensure(sizeof(int) * std::max<size_t>(1, all.size()))) return -1;
    HIPCHK(hipMemcpyAsync(b->d_tmp_list.p, all.data(), sizeof(int) * all.size(), hipMemcpyHostToDevice, st));
    // G lanes per shell pair split the nuclear attraction over the atoms of
    // the pair's molecule: the most atoms of any molecule, rounded up to a
    // power of two, at most 32
    int amax = 1;
    for (const MolInfo& mi : b->mols) amax = std::max(amax, mi.atom_hi - mi.atom_lo);
    int G = 1;
    while (G < amax && G < 32) G <<= 1;
    OneeFusedArgs f = {};
    f.G = G;
    f.block0[0] = 0;
    for (int c = 0; c < 6; ++c) {
        OneeArgs& a = f.cls[c];
        a.pair_list = (const int*)b->d_tmp_list.p + offs[c];
        a.pairs = (const PairHdr*)b->d_pairs.p;
        a.prims = (const PrimPair<double>*)b->d_prims.p;
        a.atoms = (const double*)b->d_atoms.p;
        a.cart_off = (const int*)b->d_cart_off.p;
        a.mols = (const MolInfo*)b->d_mols.p;
        a.S = S; a.T = T; a.V = V;
        a.npair = offs[c + 1] - offs[c];
        f.block0[c + 1] = f.block0[c] + (int)(((long long)a.npair * G + 127) / 128);
    }
    onee_fused_run(f, st);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

static int class_of_pair_classes(int X, int Y)
{
    for (int c = 0; c < ERI_NCLASS; ++c)
        if (eri_class_table[c][5] == X && eri_class_table[c][6] == Y) return c;
    return -1;
}

// Launch one class over a quartet list already on the device.
template <typename real>
static int run_class(pq_basis* b, int cls, const int2* dq, int nq, real* dout, hipStream_t st,
                     const int* order = nullptr)
{
    if (nq <= 0) return 0;
    EriArgs<real> a;
    a.quartets = dq;
    a.pairs = (const PairHdr*)b->d_pairs.p;
    a.prims = (const PrimPair<double>*)b->d_prims.p;
    a.out = dout;
    a.nq = nq;
    a.order = order;
    if (b->op == 1) {
        if (sizeof(real) != sizeof(double)) return fail("scattering integrals are computed in FP64 only");
        EriArgs<double> d = *(const EriArgs<double>*)&a;
        d.scatt_S = b->op_S;
        eri_table_s[cls](d, st);
    } else {
        eri_launch<real>(cls, a, st);
    }
    HIPCHK(hipGetLastError());
    return 0;
}

// Scratch bytes per lane of the kernel run_class launches for class cls.
static size_t class_scratch(const pq_basis* b, int cls, bool fp32)
{
    if (b->op == 1) return eri_scratch_table_s[cls]();
    return fp32 ? eri_scratch_table_f[cls]() : eri_scratch_table_d[cls]();
}

extern "C" int pq_schwarz(pq_basis* b, double* pair_bound_host, void* stream)
{
    if (!b) return fail("pq_schwarz: null basis");
    hipStream_t st = (hipStream_t)stream;
    // one upload and one scratch area for the six diagonal classes (P|P)
    size_t nq_all = 0, nv_all = 0;
    for (int X = 0; X < 6; ++X) {
        const size_t n = b->class_pairs[X].size();
        nq_all += n;
        nv_all += n * eri_class_table[class_of_pair_classes(X, X)][4];
    }
    std::vector<int2> hq;
    std::vector<int> hids;
    hq.reserve(nq_all);
    hids.reserve(nq_all);
    for (int X = 0; X < 6; ++X)
        for (int id : b->class_pairs[X]) {
            hq.push_back(make_int2(id, id));
            hids.push_back(id);
        }
    DevBuf dq, dv, dids;
    if (dq.ensure(sizeof(int2) * std::max<size_t>(1, nq_all)) || dv.ensure(sizeof(double) * std::max<size_t>(1, nv_all)) ||
        dids.ensure(sizeof(int) * std::max<size_t>(1, nq_all)))
        return -1;
    if (nq_all) {
        HIPCHK(hipMemcpyAsync(dq.p, hq.data(), sizeof(int2) * nq_all, hipMemcpyHostToDevice, st));
        HIPCHK(hipMemcpyAsync(dids.p, hids.data(), sizeof(int) * nq_all, hipMemcpyHostToDevice, st));
    }
    // the diagonal classes on the side streams, those whose kernels use
    // scratch on the caller's; each class's bounds are extracted on the stream
    // that computed it
    const int ns = std::min(4, std::max(1, b->eri_nstreams));
    if (ns > 1) {
        if (ensure_jk_streams(b)) return -1;
        HIPCHK(hipEventRecord(b->ev_fork, st));
        for (int k = 0; k < ns; ++k) HIPCHK(hipStreamWaitEvent(b->jk_side[k], b->ev_fork, 0));
    }
    auto extract = [&](int cls, int n, size_t oq, size_t ov, hipStream_t sk) {
        const int l1 = eri_class_table[cls][0], l2 = eri_class_table[cls][1];
        hipLaunchKernelGGL(schwarz_extract_kernel, dim3((n + 127) / 128), dim3(128), 0, sk,
                           (const double*)((double*)dv.p + ov), (const int*)dids.p + oq, n, ncart_l(l1), ncart_l(l2),
                           (const PairHdr*)b->d_pairs.p, b->any_spher ? (const int*)b->d_spher.p : (const int*)nullptr,
                           (double*)b->d_bound.p);
    };
    int side = 0;
    size_t oq = 0, ov = 0;
    for (int X = 0; X < 6; ++X) {
        const int n = (int)b->class_pairs[X].size();
        if (!n) continue;
        const int cls = class_of_pair_classes(X, X);
        double* v = (double*)dv.p + ov;
        hipStream_t sk = (ns > 1 && class_scratch(b, cls, false) == 0) ? b->jk_side[side++ % ns] : st;
        if (run_class<double>(b, cls, (const int2*)dq.p + oq, n, v, sk)) return -1;
        extract(cls, n, oq, ov, sk);
        HIPCHK(hipGetLastError());
        oq += n;
        ov += (size_t)n * eri_class_table[cls][4];
    }
    if (ns > 1)
        for (int k = 0; k < ns; ++k) {
            HIPCHK(hipEventRecord(b->ev_join[k], b->jk_side[k]));
            HIPCHK(hipStreamWaitEvent(st, b->ev_join[k], 0));
        }
    HIPCHK(hipStreamSynchronize(st));   // hq, hids and the scratch go out of scope
    dq.release(); dv.release(); dids.release();
    b->bound.resize(b->npair);
    HIPCHK(hipMemcpy(b->bound.data(), b->d_bound.p, sizeof(double) * b->npair, hipMemcpyDeviceToHost));
    b->have_bound = 1;
    if (pair_bound_host) {
        for (int sa = 0; sa < b->nshell; ++sa)
            for (int sb = 0; sb < b->nshell; ++sb)
            {
                const int id = pair_id(b, sa, sb);
                pair_bound_host[(size_t)sa * b->nshell + sb] = id < 0 ? 0.0 : b->bound[id];
            }
    }
    return 0;
}

// Sort every pair class by (molecule, descending bound) on the host (a few
// thousand pairs) and upload the sorted ids, molecule segments and cumulative
// primitive-pair counts that the device list builder reads.
static int upload_sorted_pairs(pq_basis* b, hipStream_t st)
{
    // each pair class sorted by molecule ascending, then bound descending,
    // ties in id order: a stable LSD radix sort on the complemented IEEE bits
    // of the bounds (non-negative doubles order as their bit patterns), byte
    // passes that every key shares skipped, then a stable counting pass on
    // the molecule.  A comparison sort took ~2.5x as long for the 21k pairs of
    // a 20-carbon alkane.
    auto sort_class = [&](int X) {
        const std::vector<int>& ids = b->class_pairs[X];
        const size_t n = ids.size();
        std::vector<uint64_t> key(n), key2(n);
        std::vector<int> id(ids), id2(n);
        for (size_t k = 0; k < n; ++k) {
            uint64_t u;
            memcpy(&u, &b->bound[ids[k]], sizeof(u));
            key[k] = ~u;
        }
        for (int pass = 0; pass < 8; ++pass) {
            const int sh = 8 * pass;
            size_t cnt[257] = {0};
            for (size_t k = 0; k < n; ++k) cnt[((key[k] >> sh) & 255) + 1]++;
            bool shared = false;
            for (int d = 1; d <= 256; ++d) shared = shared || cnt[d] == n;
            if (shared) continue;
            for (int d = 0; d < 256; ++d) cnt[d + 1] += cnt[d];
            for (size_t k = 0; k < n; ++k) {
                const size_t o = cnt[(key[k] >> sh) & 255]++;
                key2[o] = key[k];
                id2[o] = id[k];
            }
            key.swap(key2);
            id.swap(id2);
        }
        if (b->nmol > 1) {
            std::vector<size_t> cnt(b->nmol + 1, 0);
            for (size_t k = 0; k < n; ++k) cnt[b->pairs[id[k]].mol + 1]++;
            for (int m = 0; m < b->nmol; ++m) cnt[m + 1] += cnt[m];
            for (size_t k = 0; k < n; ++k) id2[cnt[b->pairs[id[k]].mol]++] = id[k];
            id.swap(id2);
        }
        b->hsorted[X] = std::move(id);
    };
    for (int X = 0; X < 6; ++X) sort_class(X);
    for (int X = 0; X < 6; ++X) {
        std::vector<int> sorted = std::move(b->hsorted[X]);
        std::vector<int> seg(b->nmol + 1, 0);
        for (int id : sorted) seg[b->pairs[id].mol + 1]++;
        for (int m = 0; m < b->nmol; ++m) seg[m + 1] += seg[m];
        std::vector<long long> npcum(sorted.size() + 1, 0);
        for (size_t k = 0; k < sorted.size(); ++k) npcum[k + 1] = npcum[k] + b->pairs[sorted[k]].n;
        std::vector<double> sb(std::max<size_t>(1, sorted.size()), 0.0);
        for (size_t k = 0; k < sorted.size(); ++k) sb[k] = b->bound[sorted[k]];
        b->nsorted[X] = (int)sorted.size();
        b->hsorted[X] = std::move(sorted);
        b->hnpcum[X] = std::move(npcum);
        b->hseg[X] = std::move(seg);
        b->hsbound[X] = std::move(sb);
    }
    // one upload of every class's arrays (separate copies from pageable
    // memory cost ~20 us of host time each, 24 per plan); 256-byte sections
    size_t off[6][5], total = 0;
    auto take = [&](size_t bytes) {
        const size_t o = total;
        total += (std::max<size_t>(bytes, 1) + 255) / 256 * 256;
        return o;
    };
    for (int X = 0; X < 6; ++X) {
        off[X][0] = take(sizeof(int) * b->hsorted[X].size());
        off[X][1] = take(sizeof(int) * b->hseg[X].size());
        off[X][2] = take(sizeof(long long) * b->hnpcum[X].size());
        off[X][3] = take(sizeof(double) * b->hsbound[X].size());
        off[X][4] = take(sizeof(unsigned) * b->hsorted[X].size());
    }
    if (b->d_sortpack.ensure(total)) return -1;
    // the host pack lives in the handle until the next plan, so the
    // asynchronous upload needs no wait here
    b->hsortpack.assign(total, 0);
    char* h = b->hsortpack.data();
    char* d = (char*)b->d_sortpack.p;
    for (int X = 0; X < 6; ++X) {
        memcpy(h + off[X][0], b->hsorted[X].data(), sizeof(int) * b->hsorted[X].size());
        memcpy(h + off[X][1], b->hseg[X].data(), sizeof(int) * b->hseg[X].size());
        memcpy(h + off[X][2], b->hnpcum[X].data(), sizeof(long long) * b->hnpcum[X].size());
        memcpy(h + off[X][3], b->hsbound[X].data(), sizeof(double) * b->hsbound[X].size());
        unsigned* rec = (unsigned*)(h + off[X][4]);
        for (size_t k = 0; k < b->hsorted[X].size(); ++k) {
            const PairHdr& p = b->pairs[b->hsorted[X][k]];
            rec[k] = (unsigned)b->cart_off[p.s1] | ((unsigned)b->cart_off[p.s2] << 15) | (p.s1 == p.s2 ? 1u << 30 : 0u);
        }
        b->p_sorted[X] = (const int*)(d + off[X][0]);
        b->p_rec[X] = (const unsigned*)(d + off[X][4]);
        b->p_seg[X] = (const int*)(d + off[X][1]);
        b->p_npcum[X] = (const long long*)(d + off[X][2]);
        b->p_sbound[X] = (const double*)(d + off[X][3]);
    }
    HIPCHK(hipMemcpyAsync(d, h, total, hipMemcpyHostToDevice, st));
    return 0;
}

static ListArgs list_args(const pq_basis* b, int c)
{
    const int X = eri_class_table[c][5], Y = eri_class_table[c][6];
    ListArgs a;
    a.bra = b->p_sorted[X];
    a.ket = b->p_sorted[Y];
    a.bra_seg = b->p_seg[X];
    a.ket_seg = b->p_seg[Y];
    a.ket_npcum = b->p_npcum[Y];
    a.ket_rec = b->p_rec[Y];
    a.bound = (const double*)b->d_bound.p;
    a.bra_bound = b->p_sbound[X];
    a.pairs = (const PairHdr*)b->d_pairs.p;
    a.cart_off = (const int*)b->d_cart_off.p;
    a.thr = b->threshold;
    a.thr32 = b->threshold32;
    a.nb = b->nsorted[X];
    a.nk = b->nsorted[Y];
    a.same = X == Y;
    return a;
}

static ListBras list_bras(EriClassStore& s)
{
    ListBras r;
    r.j0 = (int*)s.j0.p;
    r.cnt = (long long*)s.cnt.p;
    r.np = (long long*)s.np.p;
    r.qs = (long long*)s.qs.p;
    r.nit = (long long*)s.nit.p;
    r.its = (long long*)s.its.p;
    return r;
}

// J/K work items of a class on the device (kept with the FP64 store): per bra
// pair, its FP64 kets then its FP32 kets, cut into pieces of at most `run`
// quartets.  Automatic length: every item stages and flushes TA + TB rows of
// Dk and K' of n elements each, so its ERI values (run * ncomp) should
// outweigh one of those row sets 64 times over (PQ_JK_RUN_SCALE), within
// 64..1024.  The staging and flush per item cost more than the parallelism
// of more, shorter items gains: whole J/K of C10H22 / C20H42 (6-31G*) at
// scale 4 with at least 512 items per class was 12 % / 25 % slower than the
// autotuned lengths; at 16, 0.348 / 1.278 ms; at 32, 64, 128 and 256,
// 0.331-0.333 / 1.241-1.249 ms.
static long long item_run(const pq_basis* b, int c)
{
    const EriClassStore& s = b->store64[c];
    long long run = s.jk_run;
    if (run <= 0) {
        static const long long scale = [] {
            const char* e = getenv("PQ_JK_RUN_SCALE");
            return e ? std::max(1LL, atoll(e)) : 64LL;
        }();
        const long long rows = jk_tile_table[c][3] / 2;
        run = (scale * rows * b->nmax + s.ncomp - 1) / s.ncomp;
        run = std::max(64LL, std::min(1024LL, (run + 63) / 64 * 64));
    }
    return run;
}

// Items per bra and their scan; the class's item count lands in *total.
static void items_count(pq_basis* b, int c, long long* total, hipStream_t st)
{
    const ListBras l64 = list_bras(b->store64[c]), l32 = list_bras(b->store32[c]);
    const int nb = list_args(b, c).nb;
    list_items_count(l64, b->store32[c].nq ? &l32 : nullptr, nb, item_run(b, c), st);
    list_scan(l64.nit, l64.its, nb, total, st);
}

static int items_fill(pq_basis* b, int c, long long nitems, hipStream_t st)
{
    EriClassStore& s = b->store64[c];
    if (nitems > 0x7fffffffLL) return fail("J/K work items exceed 2^31");
    s.nitems = (int)nitems;
    const bool f32 = b->store32[c].nq > 0;
    if (s.items.ensure(sizeof(JkItem) * std::max(1, s.nitems)) ||
        (f32 && s.items32.ensure(sizeof(int2) * std::max(1, s.nitems))))
        return -1;
    const ListBras l32 = list_bras(b->store32[c]);
    list_items_fill(list_args(b, c), list_bras(s), f32 ? &l32 : nullptr, nitems, item_run(b, c), (JkItem*)s.items.p,
                    (int2*)s.items32.p, st);
    HIPCHK(hipGetLastError());
    return 0;
}

// One class's items (synchronises `st` to learn the count).
static int build_items(pq_basis* b, int c, hipStream_t st)
{
    b->store64[c].nitems = 0;
    if (!b->store64[c].nq && !b->store32[c].nq) return 0;
    items_count(b, c, (long long*)b->d_total.p, st);
    long long nitems = 0;
    HIPCHK(hipMemcpyAsync(&nitems, b->d_total.p, sizeof(long long), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return items_fill(b, c, nitems, st);
}

// The tiled kernel packs offsets into 15 bits and keeps 2 (TA + TB) rows of
// the largest molecule in LDS, all 160 KiB of a CU if need be: C30H62 (n = 574,
// 83 KB for the nine-row tiles) 3.06 ms per build, 10.9 ms when those classes
// went one thread per quartet from 64 KiB on.
static inline bool jk_tile_fits(const pq_basis* b, int cls)
{
    return b->nmax < 32768 && sizeof(double) * (size_t)jk_tile_table[cls][3] * b->nmax <= 163840;
}

// The two-electron operator of the class kernels (Methods/_c_ints.c:236-239
// dispatches on ints_type): 0 the Coulomb operator, 1 the electron-scattering
// operator at momentum transfer grid_value (Methods/c_ints/
// two_electron_scattering.c).  The Schwarz bounds are taken again with the
// new operator at the next plan, as the reference's evaluate_2e_ints does
// (Methods/hartree_fock.py:244-254 with its ints_type); stored integrals need
// a new pq_eri_plan / pq_eri_compute.
extern "C" int pq_eri_set_operator(pq_basis* b, int ints_type, double grid_value)
{
    if (!b) return fail("pq_eri_set_operator: null basis");
    if (ints_type != 0 && ints_type != 1) return fail("pq_eri_set_operator: ints_type must be 0 or 1");
    if (ints_type == 1 && !(grid_value >= 0.0)) return fail("pq_eri_set_operator: grid_value must be >= 0");
    if (b->op != ints_type || (ints_type == 1 && b->op_S != grid_value)) b->have_bound = 0;
    b->op = ints_type;
    b->op_S = ints_type == 1 ? grid_value : 0.0;
    return 0;
}

extern "C" int pq_eri_plan(pq_basis* b, double threshold, double fp32_threshold, void* stream)
{
    if (!b) return fail("pq_eri_plan: null basis");
    if (b->op == 1 && fp32_threshold > 0.0) return fail("pq_eri_plan: scattering integrals are FP64 only");
    hipStream_t st = (hipStream_t)stream;
    if (!b->have_bound && pq_schwarz(b, nullptr, stream)) return -1;
    b->threshold = threshold;
    b->threshold32 = fp32_threshold;
    // Screened unique quartet lists, built on the device (lists.h): for
    // classes X != Y every (bra, ket) of a molecule with Q_bra Q_ket > thr;
    // for X == Y ket rank >= bra rank; diagonal quartets (P|P) always kept
    // (the reference stores them from its bounds pass,
    // Methods/hartree_fock.py:244-273).  Quartets with bound product below
    // thr32 (when > 0) go to the FP32 list.
    if (upload_sorted_pairs(b, st)) return -1;
    if (b->d_total.ensure(sizeof(long long) * 4 * ERI_NCLASS)) return -1;
    long long* dtot = (long long*)b->d_total.p;
    // one launch per phase over every class (lists.h: batched construction);
    // each upload's host copy stays in the handle until the next plan
    b->hjobs.clear();
    b->hscans.clear();
    if (b->d_jobs.ensure(sizeof(ListJob) * ERI_NCLASS) || b->d_scans.ensure(sizeof(ScanJob) * 4 * ERI_NCLASS))
        return -1;
    auto upload_jobs = [&](const std::vector<ListJob>& v) -> int {
        HIPCHK(hipMemcpyAsync(b->d_jobs.p, v.data(), sizeof(ListJob) * v.size(), hipMemcpyHostToDevice, st));
        return 0;
    };
    auto upload_scans = [&](const std::vector<ScanJob>& v) -> int {
        HIPCHK(hipMemcpyAsync(b->d_scans.p, v.data(), sizeof(ScanJob) * v.size(), hipMemcpyHostToDevice, st));
        return 0;
    };
    // counts per bra, then their scans (totals: quartets and primitive
    // quartets of both lists per class)
    b->hjobs.emplace_back(ERI_NCLASS);
    {
        std::vector<ListJob>& jobs = b->hjobs.back();
        ListBlocks blk = {};
        blk.n = ERI_NCLASS;
        for (int c = 0; c < ERI_NCLASS; ++c) {
            ListArgs a = list_args(b, c);
            const size_t nb = (size_t)std::max(1, a.nb);
            for (int w = 0; w < 2; ++w) {
                EriClassStore& s = w ? b->store32[c] : b->store64[c];
                if (s.j0.ensure(sizeof(int) * nb) || s.cnt.ensure(8 * nb) || s.np.ensure(8 * nb) ||
                    s.qs.ensure(8 * nb) || s.nit.ensure(8 * nb) || s.its.ensure(8 * nb))
                    return -1;
            }
            if (a.nb == 0 || a.nk == 0) a.nb = 0;   // nothing kept: zero totals
            jobs[c] = ListJob{};
            jobs[c].a = a;
            jobs[c].b64 = list_bras(b->store64[c]);
            jobs[c].b32 = list_bras(b->store32[c]);
            blk.block0[c + 1] = blk.block0[c] + (a.nb + 255) / 256;
        }
        if (upload_jobs(jobs)) return -1;
        list_count_batch((const ListJob*)b->d_jobs.p, blk, st);
        b->hscans.emplace_back();
        std::vector<ScanJob>& sc = b->hscans.back();
        for (int c = 0; c < ERI_NCLASS; ++c) {
            const ListBras& l64 = jobs[c].b64;
            const ListBras& l32 = jobs[c].b32;
            const int n = jobs[c].a.nb;
            sc.push_back({l64.cnt, l64.qs, n, dtot + 4 * c + 0});
            sc.push_back({l32.cnt, l32.qs, n, dtot + 4 * c + 1});
            sc.push_back({l64.np, l64.nit, n, dtot + 4 * c + 2});   // nit as scratch: only the totals are kept
            sc.push_back({l32.np, l32.nit, n, dtot + 4 * c + 3});
        }
        if (upload_scans(sc)) return -1;
        list_scan_batch((const ScanJob*)b->d_scans.p, (int)sc.size(), st);
    }
    HIPCHK(hipGetLastError());
    std::vector<long long> tot(4 * ERI_NCLASS);
    HIPCHK(hipMemcpyAsync(tot.data(), dtot, sizeof(long long) * tot.size(), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    // the lists themselves, then the work items' counts per bra and scans
    {
        std::vector<ListJob> next = b->hjobs.back();   // the next phase's table: a new host copy
        b->hjobs.push_back(std::move(next));
    }
    static const int order_env = [] {
        const char* e = getenv("PQ_ERI_ORDER");
        return e ? atoi(e) : 1;
    }();
    b->eri_order = order_env != 0;
    ListBlocks fill_blocks = {};
    fill_blocks.n = 2 * ERI_NCLASS;
    if (b->d_order_cnt.ensure(sizeof(int) * 2 * ORD_NB * fill_blocks.n)) return -1;
    {
        std::vector<ListJob>& jobs = b->hjobs.back();
        for (int c = 0; c < ERI_NCLASS; ++c) {
            const int ncd = ncart_l(eri_class_table[c][2]) * ncart_l(eri_class_table[c][3]);
            for (int w = 0; w < 2; ++w) {
                EriClassStore& s = w ? b->store32[c] : b->store64[c];
                const long long nq = tot[4 * c + w];
                if (nq > 0x7fffffffLL) return fail("pq_eri_plan: more than 2^31 quartets in one class");
                s.nq = (int)nq;
                s.nprimq = tot[4 * c + 2 + w];
                s.nitems = 0;
                jobs[c].nq[w] = s.nq;
                jobs[c].q[w] = nullptr;
                jobs[c].k[w] = nullptr;
                jobs[c].ord[w] = nullptr;
                jobs[c].bk[w] = nullptr;
                if (s.nq) {
                    const size_t vb = (size_t)s.nq * s.ncomp * (w ? sizeof(float) : sizeof(double));
                    const size_t jb =
                        jk_tile_fits(b, c) ? sizeof(double) * (size_t)s.nq * jk_tile_table[c][2] * ncd : 0;
                    if (s.q.ensure(sizeof(int2) * s.nq) || s.vals.ensure(vb) ||
                        s.kets.ensure(sizeof(unsigned) * s.nq) || s.jkbuf.ensure(jb) ||
                        (uses_order(b, s) && s.order.ensure((sizeof(int) + 1) * s.nq)))   // order, then buckets
                        return -1;
                    jobs[c].q[w] = (int2*)s.q.p;
                    jobs[c].k[w] = (unsigned*)s.kets.p;
                    if (uses_order(b, s)) {
                        jobs[c].ord[w] = (int*)s.order.p;
                        jobs[c].bk[w] = (unsigned char*)(jobs[c].ord[w] + s.nq);
                    }
                }
                fill_blocks.block0[2 * c + w + 1] =
                    fill_blocks.block0[2 * c + w] + (int)((nq + 256 * ORD_PT - 1) / (256 * ORD_PT));
            }
        }
        if (upload_jobs(jobs)) return -1;
        list_fill_batch((const ListJob*)b->d_jobs.p, fill_blocks, (int*)b->d_order_cnt.p, st);
    }
    {
        std::vector<ListJob> next = b->hjobs.back();   // the next phase's table: a new host copy
        b->hjobs.push_back(std::move(next));
    }
    {
        std::vector<ListJob>& jobs = b->hjobs.back();
        ListBlocks ib = {};
        ib.n = ERI_NCLASS;
        b->hscans.emplace_back();
        std::vector<ScanJob>& sc = b->hscans.back();
        for (int c = 0; c < ERI_NCLASS; ++c) {
            const bool any = b->store64[c].nq || b->store32[c].nq;
            jobs[c].nb_items = any ? list_args(b, c).nb : 0;
            jobs[c].run = item_run(b, c);
            jobs[c].has32 = b->store32[c].nq > 0;
            ib.block0[c + 1] = ib.block0[c] + (jobs[c].nb_items + 255) / 256;
            sc.push_back({jobs[c].b64.nit, jobs[c].b64.its, jobs[c].nb_items, dtot + c});
        }
        if (upload_jobs(jobs)) return -1;
        list_items_count_batch((const ListJob*)b->d_jobs.p, ib, st);
        if (upload_scans(sc)) return -1;
        list_scan_batch((const ScanJob*)b->d_scans.p, (int)sc.size(), st);
    }
    HIPCHK(hipGetLastError());
    // every class's item count in one transfer, then the items
    std::vector<long long> nit(ERI_NCLASS, 0);
    HIPCHK(hipMemcpyAsync(nit.data(), dtot, sizeof(long long) * nit.size(), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    {
        std::vector<ListJob> next = b->hjobs.back();   // the next phase's table: a new host copy
        b->hjobs.push_back(std::move(next));
    }
    {
        std::vector<ListJob>& jobs = b->hjobs.back();
        ListBlocks tb = {};
        tb.n = ERI_NCLASS;
        for (int c = 0; c < ERI_NCLASS; ++c) {
            EriClassStore& s = b->store64[c];
            s.nitems = b->store32[c].nitems = 0;
            jobs[c].nitems = 0;
            jobs[c].items = nullptr;
            jobs[c].items32 = nullptr;
            if (jobs[c].nb_items > 0) {
                if (nit[c] > 0x7fffffffLL) return fail("J/K work items exceed 2^31");
                s.nitems = (int)nit[c];
                const bool f32 = b->store32[c].nq > 0;
                if (s.items.ensure(sizeof(JkItem) * std::max(1, s.nitems)) ||
                    (f32 && s.items32.ensure(sizeof(int2) * std::max(1, s.nitems))))
                    return -1;
                jobs[c].nitems = s.nitems;
                jobs[c].items = (JkItem*)s.items.p;
                jobs[c].items32 = f32 ? (int2*)s.items32.p : nullptr;
            }
            tb.block0[c + 1] = tb.block0[c] + (int)((jobs[c].nitems + 255) / 256);
        }
        if (upload_jobs(jobs)) return -1;
        list_items_fill_batch((const ListJob*)b->d_jobs.p, tb, st);
        // the ERI kernels' quartet order (the table still holds every list's
        // buckets and order buffer), queued after the plan's last host wait
        if (b->eri_order)
            list_order_batch((const ListJob*)b->d_jobs.p, fill_blocks, (const int*)b->d_order_cnt.p,
                             (int*)b->d_order_cnt.p + ORD_NB * fill_blocks.n, st);
    }
    HIPCHK(hipGetLastError());
    // table of the ket J reductions of every tiled list; every list's tiles
    // in one buffer and one upload (host copy kept in the handle)
    std::vector<JredList> jr;
    std::vector<size_t> toff;
    std::vector<int4>& all = b->hjtiles_all;
    all.clear();
    long long blocks = 0;
    std::vector<int> tiled;   // classes by launch group
    for (int g = 0; g < JK_NGROUP; ++g)
        for (int c = 0; c < ERI_NCLASS; ++c)
            if (jk_group_table[c] == g && jk_tile_fits(b, c)) tiled.push_back(c);
    for (int g = 0; g <= JK_NGROUP; ++g) b->jred_list0[g] = b->jred_block0[g] = 0;
    for (int c : tiled) {
        const int n3 = ncart_l(eri_class_table[c][2]), n4 = ncart_l(eri_class_table[c][3]);
        for (int w = 0; w < 2; ++w) {
            EriClassStore& s = w ? b->store32[c] : b->store64[c];
            s.jtiles = nullptr;
            s.njtile = 0;
            if (!s.nq) continue;
            const int X = eri_class_table[c][5], Y = eri_class_table[c][6];
            const std::vector<int4> tl =
                jred_tiles(b->hseg[X], b->hseg[Y], b->hsbound[X], b->hsbound[Y], X == Y, b->threshold);
            toff.push_back(all.size());
            all.insert(all.end(), tl.begin(), tl.end());
            s.njtile = (int)tl.size();
            JredList L = jred_list(list_args(b, c), list_bras(s), w, (const double*)s.jkbuf.p, s.nq,
                                   jk_tile_table[c][2], n3 * n4, n4, nullptr, s.njtile);
            L.block0 = blocks;
            blocks += (long long)L.ntile * L.ncd;
            jr.push_back(L);
        }
        for (int g = jk_group_table[c] + 1; g <= JK_NGROUP; ++g) {
            b->jred_list0[g] = (int)jr.size();
            b->jred_block0[g] = blocks;
        }
    }
    if (b->d_jtiles.ensure(sizeof(int4) * std::max<size_t>(1, all.size()))) return -1;
    if (!all.empty())
        HIPCHK(hipMemcpyAsync(b->d_jtiles.p, all.data(), sizeof(int4) * all.size(), hipMemcpyHostToDevice, st));
    {
        size_t k = 0;
        for (int c : tiled) {
            for (int w = 0; w < 2; ++w) {
                EriClassStore& s = w ? b->store32[c] : b->store64[c];
                if (!s.nq) continue;
                s.jtiles = (const int4*)b->d_jtiles.p + toff[k];
                jr[k].tiles = s.jtiles;
                ++k;
            }
        }
    }
    if (blocks > 0x7fffffffLL) return fail("pq_eri_plan: ket J reduction grid too large");
    if (b->d_jred.ensure(sizeof(JredList) * std::max<size_t>(1, jr.size()))) return -1;
    b->hjred = std::move(jr);   // kept in the handle: no wait for the upload
    if (!b->hjred.empty())
        HIPCHK(hipMemcpyAsync(b->d_jred.p, b->hjred.data(), sizeof(JredList) * b->hjred.size(), hipMemcpyHostToDevice,
                              st));
    HIPCHK(hipGetLastError());
    return 0;
}

// All class kernels over the planned lists (the ERI-generation pass).
// Each class is one launch: its FP64 and FP32 lists (a mixed-precision plan)
// together, the FP64 blocks first.  The launches fork from `st` onto the
// side streams (the longest expected launch first, each to the least-loaded
// stream) and join back, so that the classes overlap.  Kernels that spill
// (per-lane scratch: the runtime sizes scratch per hardware queue for a full
// device of waves) stay on `st`, the one queue that always carried them.
extern "C" int pq_eri_compute(pq_basis* b, void* stream)
{
    if (!b) return fail("pq_eri_compute: null basis");
    hipStream_t st = (hipStream_t)stream;
    if (b->timing && ensure_events(b)) return -1;
    // A launch lasts about as long as its deepest quartet's chain of dependent
    // instructions, some 8 cycles each (a lane runs all of a quartet's
    // primitives: 1296 of (ss|ss) or 81 of (pp|pp) in 6-31G* are 0.4 and
    // 0.17 ms, however few such quartets there are), plus its share of the
    // chip, 4 cycles per wave instruction and SIMD.  By work alone the deep
    // classes with little of it came last and the pass ended in their chains:
    // C14H30 1.72 ms, in this order 1.58.
    std::vector<std::pair<double, int>> order;
    for (int c = 0; c < ERI_NCLASS; ++c) {
        const double body = 1.5 * eri_body_lines[c] + 50.0;
        const int deepest = b->class_nmax[eri_class_table[c][5]] * b->class_nmax[eri_class_table[c][6]];
        double cost = 0.0;
        for (int w = 0; w < 2; ++w) {
            EriClassStore& s = w ? b->store32[c] : b->store64[c];
            b->ev_cls_used[2 * c + w] = 0;
            if (s.nq)
                cost += 8.0 * (body * deepest + 20.0 * s.ncomp) +
                        4.0 / (64 * 1024) * (body * s.nprimq + (200.0 + 8.0 * s.ncomp) * s.nq);
        }
        if (cost > 0.0) order.push_back({cost, c});
    }
    std::sort(order.begin(), order.end(), [](const std::pair<double, int>& u, const std::pair<double, int>& v) {
        return u.first > v.first;
    });
    const int ns = std::min(4, std::max(1, b->eri_nstreams));
    if (b->timing) HIPCHK(hipEventRecord(b->ev_pass[0], st));
    if (ns > 1) {
        if (ensure_jk_streams(b)) return -1;
        HIPCHK(hipEventRecord(b->ev_fork, st));
        for (int k = 0; k < ns; ++k) HIPCHK(hipStreamWaitEvent(b->jk_side[k], b->ev_fork, 0));
    }
    auto args_d = [&](int c) {
        EriClassStore& s = b->store64[c];
        return EriArgs<double>{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p, (const PrimPair<double>*)b->d_prims.p,
                               (double*)s.vals.p, s.nq, order_of(b, s)};
    };
    auto args_f = [&](int c) {
        EriClassStore& s = b->store32[c];
        return EriArgs<float>{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p, (const PrimPair<double>*)b->d_prims.p,
                              (float*)s.vals.p, s.nq, order_of(b, s)};
    };
    auto mark = [&](int c, int k, hipStream_t sk) -> int {   // timing events of both lists of class c
        if (!b->timing) return 0;
        for (int w = 0; w < 2; ++w)
            if ((w ? b->store32[c] : b->store64[c]).nq) {
                HIPCHK(hipEventRecord(b->ev_cls[2 * c + w][k], sk));
                if (k) b->ev_cls_used[2 * c + w] = 1;
            }
        return 0;
    };
    double load[4] = {0.0, 0.0, 0.0, 0.0};
    for (const auto& o : order) {
        const int c = o.second;
        int k = 0;
        for (int t = 1; t < ns; ++t)
            if (load[t] < load[k]) k = t;
        const bool u64 = b->store64[c].nq > 0, u32 = b->store32[c].nq > 0;
        const bool spills = (u64 && u32) ? eri_scratch_table_mix[c]() > 0 : class_scratch(b, c, !u64) > 0;
        if (!spills) load[k] += o.first;
        hipStream_t sk = (ns > 1 && !spills) ? b->jk_side[k] : st;
        if (mark(c, 0, sk)) return -1;
        if (u64 && u32) {
            eri_table_mix[c](args_d(c), args_f(c), sk);
            HIPCHK(hipGetLastError());
        } else if (u64) {
            if (run_class<double>(b, c, (const int2*)b->store64[c].q.p, b->store64[c].nq, (double*)b->store64[c].vals.p,
                                  sk, order_of(b, b->store64[c])))
                return -1;
        } else {
            if (run_class<float>(b, c, (const int2*)b->store32[c].q.p, b->store32[c].nq, (float*)b->store32[c].vals.p,
                                 sk, order_of(b, b->store32[c])))
                return -1;
        }
        if (mark(c, 1, sk)) return -1;
    }
    if (ns > 1)
        for (int k = 0; k < ns; ++k) {
            HIPCHK(hipEventRecord(b->ev_join[k], b->jk_side[k]));
            HIPCHK(hipStreamWaitEvent(st, b->ev_join[k], 0));
        }
    if (b->timing) {
        HIPCHK(hipEventRecord(b->ev_pass[1], st));
        b->ev_pass_used = 1;
    }
    HIPCHK(hipGetLastError());
    return 0;
}

extern "C" int pq_eri_build(pq_basis* b, double threshold, double fp32_threshold, void* stream)
{
    if (pq_eri_plan(b, threshold, fp32_threshold, stream)) return -1;
    return pq_eri_compute(b, stream);
}

extern "C" int pq_eri_recompute(pq_basis* b, void* stream) { return pq_eri_compute(b, stream); }

// Per-class J/K digestion times summed over the calls made with timing on
// (pq_jk, pq_jk_general, the J/K of pq_scf_run): from the start of a class's
// first block to the end of its last, by the GPU's realtime clock (the classes
// of a call share launches); calls counted and the classes' work items; reset
// != 0 clears the sums afterwards.  Waits for the device.
extern "C" int pq_jk_class_times(pq_basis* b, double* sum_ms, long long* launches, long long* nitems, int reset)
{
    if (!b) return fail("pq_jk_class_times: null basis");
    unsigned long long h[2 * ERI_NCLASS] = {};
    double ms_per_tick = 0.0;
    if (b->d_jkclock.p) {
        int dev = 0, khz = 0;
        HIPCHK(hipGetDevice(&dev));
        HIPCHK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
        if (khz > 0) ms_per_tick = 1.0 / khz;
        HIPCHK(hipDeviceSynchronize());
        HIPCHK(hipMemcpy(h, (unsigned long long*)b->d_jkclock.p + JK_CLOCK_SUMS, sizeof(h), hipMemcpyDeviceToHost));
    }
    for (int c = 0; c < ERI_NCLASS; ++c) {
        if (sum_ms) sum_ms[c] = (double)h[2 * c] * ms_per_tick;
        if (launches) launches[c] = (long long)h[2 * c + 1];
        if (nitems) nitems[c] = b->store64[c].nitems;
    }
    if (reset && b->d_jkclock.p) {
        hipLaunchKernelGGL(jk_clock_kernel, dim3(ERI_NCLASS), dim3(64), 0, nullptr, (unsigned long long*)b->d_jkclock.p, 2);
        HIPCHK(hipDeviceSynchronize());
    }
    return 0;
}

extern "C" int pq_set_timing(pq_basis* b, int on)
{
    if (!b) return fail("pq_set_timing: null basis");
    b->timing = on ? 1 : 0;
    if (!b->timing) return 0;
    if (ensure_events(b)) return -1;
    if (!b->d_jkclock.p) {
        if (b->d_jkclock.ensure(sizeof(unsigned long long) * (JK_CLOCK_SUMS + 2 * ERI_NCLASS))) return -1;
        hipLaunchKernelGGL(jk_clock_kernel, dim3(ERI_NCLASS), dim3(64), 0, nullptr, (unsigned long long*)b->d_jkclock.p, 2);
        HIPCHK(hipDeviceSynchronize());
    }
    return 0;
}

// Elapsed ms of the last timed ERI pass per class (slot 2c = FP64 list,
// 2c+1 = FP32 list; -1 when not launched; classes overlap on the side
// streams), of the whole pass on the caller's stream, and of the last pq_jk.
extern "C" int pq_get_timings(pq_basis* b, double* eri_ms, double* jk_ms, double* eri_pass_ms)
{
    if (!b) return fail("pq_get_timings: null basis");
    if (!b->timing) return fail("pq_get_timings: timing not enabled");
    if (eri_ms)
        for (int i = 0; i < 2 * ERI_NCLASS; ++i) {
            eri_ms[i] = -1.0;
            if (!b->ev_cls_used[i]) continue;
            HIPCHK(hipEventSynchronize(b->ev_cls[i][1]));
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, b->ev_cls[i][0], b->ev_cls[i][1]));
            eri_ms[i] = ms;
        }
    if (eri_pass_ms) {
        *eri_pass_ms = -1.0;
        if (b->ev_pass_used) {
            HIPCHK(hipEventSynchronize(b->ev_pass[1]));
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, b->ev_pass[0], b->ev_pass[1]));
            *eri_pass_ms = ms;
        }
    }
    if (jk_ms) {
        *jk_ms = -1.0;
        if (b->ev_jk_used) {
            HIPCHK(hipEventSynchronize(b->ev_jk[1]));
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, b->ev_jk[0], b->ev_jk[1]));
            *jk_ms = ms;
        }
    }
    return 0;
}

// Recompute one stored class (w = 0: FP64 list, 1: FP32 list).
extern "C" int pq_eri_run_class(pq_basis* b, int cls, int w, void* stream)
{
    if (!b) return fail("pq_eri_run_class: null basis");
    if (cls < 0 || cls >= ERI_NCLASS || w < 0 || w > 1) return fail("pq_eri_run_class: bad class");
    hipStream_t st = (hipStream_t)stream;
    if (w) {
        EriClassStore& t = b->store32[cls];
        return t.nq ? run_class<float>(b, cls, (const int2*)t.q.p, t.nq, (float*)t.vals.p, st, order_of(b, t))
                    : 0;
    }
    EriClassStore& s = b->store64[cls];
    return s.nq ? run_class<double>(b, cls, (const int2*)s.q.p, s.nq, (double*)s.vals.p, st, order_of(b, s))
                : 0;
}

extern "C" int pq_eri_stats(const pq_basis* b, long long* stats, int nstats)
{
    // per class c: stats[c*6 + ...] = {nq64, nq32, ncomp, nprimq64, nprimq32, class id}
    if (!b || !stats) return fail("pq_eri_stats: null argument");
    if (nstats < ERI_NCLASS * 6) return fail("pq_eri_stats: need ERI_NCLASS*6 entries");
    for (int c = 0; c < ERI_NCLASS; ++c) {
        stats[c * 6 + 0] = b->store64[c].nq;
        stats[c * 6 + 1] = b->store32[c].nq;
        stats[c * 6 + 2] = b->store64[c].ncomp;
        stats[c * 6 + 3] = b->store64[c].nprimq;
        stats[c * 6 + 4] = b->store32[c].nprimq;
        stats[c * 6 + 5] = eri_class_table[c][0] * 1000 + eri_class_table[c][1] * 100 + eri_class_table[c][2] * 10 +
                           eri_class_table[c][3];
    }
    return 0;
}

extern "C" int pq_eri_nclass(void) { return ERI_NCLASS; }

// One class into J', K'.  part: 1 = tiled digestion kernel, 2 = ket J
// reductions, 3 = both.  lists: bit 0 the FP64 list, bit 1 the FP32 list; the
// tiled kernel digests both in one launch.
// One class's entry of a group launch (lists: 1 FP64, 2 FP32, 3 both).
// Returns its blocks; 0 when it has nothing to digest.
static int jk_class_args(pq_basis* b, int c, int lists, JkClassArgs& a)
{
    const EriClassStore& s64 = b->store64[c];
    const EriClassStore& s32 = b->store32[c];
    const bool u64 = (lists & 1) && s64.nq, u32 = (lists & 2) && s32.nq;
    if ((!u64 && !u32) || s64.nitems <= 0) return 0;
    a.items = (const JkItem*)s64.items.p;
    a.items32 = u32 ? (const int2*)s64.items32.p : (const int2*)nullptr;
    a.l64 = JkTileList<double>{(const unsigned*)s64.kets.p, (const double*)s64.vals.p, (double*)s64.jkbuf.p, s64.nq};
    a.l32 = JkTileList<float>{(const unsigned*)s32.kets.p, (const float*)s32.vals.p, (double*)s32.jkbuf.p, s32.nq};
    a.nitems = s64.nitems;
    const int tuned = s64.jk_grid > 0 ? s64.jk_grid : s32.jk_grid;
    a.grid = (tuned > 0 && tuned < a.nitems) ? tuned : a.nitems;
    a.cls = c;
    return a.grid * jk_tile_table[c][2];
}

// Work units of a class (quartets, or (quartet, ket row) pairs where the
// kernel splits the rows).
static double jk_class_units(const pq_basis* b, int c, int lists)
{
    const int n3 = ncart_l(eri_class_table[c][2]), n4 = ncart_l(eri_class_table[c][3]);
    const double units = (n3 * n4 >= 3) ? (double)n3 : 1.0;
    return units * (double)(((lists & 1) ? b->store64[c].nq : 0) + ((lists & 2) ? b->store32[c].nq : 0));
}

// The listed classes in one launch of group kernel `group`: threads per block
// from the mean work units per item.
static int jk_group_launch(pq_basis* b, int group, const int* classes, int nc, int lists, const double* Dj,
                           const double* Dk, double* J, double* K, hipStream_t st)
{
    JkGroupArgs g;
    g.n = 0;
    long long blocks = 0;
    double units = 0.0, items = 0.0;
    size_t rows = 0;
    for (int k = 0; k < nc; ++k) {
        const int c = classes[k];
        JkClassArgs& a = g.c[g.n];
        const int nb = jk_class_args(b, c, lists, a);
        if (!nb) continue;
        a.block0 = (int)blocks;
        blocks += nb;
        if (blocks > 0x7fffffffLL) return fail("J/K digestion grid too large");
        units += jk_class_units(b, c, lists);
        items += a.nitems;
        rows = std::max(rows, (size_t)jk_tile_table[c][3]);
        ++g.n;
    }
    if (!g.n) return 0;
    g.mols = (const MolInfo*)b->d_mols.p;
    g.Dj = Dj;
    g.Dk = Dk;
    g.J = J;
    g.K = K;
    g.clock = b->timing ? (unsigned long long*)b->d_jkclock.p : nullptr;
    const double mean = units / std::max(1.0, items);
    const int block = mean > 160.0 ? 256 : (mean > 80.0 ? 128 : 64);
    jk_group_run[group](g, (int)blocks, block, sizeof(double) * rows * b->nmax, st);
    HIPCHK(hipGetLastError());
    return 0;
}

// A class too wide for the tiled kernels' LDS rows, one thread per quartet.
static int jk_launch_untiled(pq_basis* b, int c, const double* Dj, const double* Dk, double* J, double* K,
                             hipStream_t st, int lists)
{
    const EriClassStore& s64 = b->store64[c];
    const EriClassStore& s32 = b->store32[c];
    const MolInfo* dm = (const MolInfo*)b->d_mols.p;
    if ((lists & 1) && s64.nq) {
        JkArgs<double> a{(const int2*)s64.q.p, (const PairHdr*)b->d_pairs.p, (const int*)b->d_cart_off.p, dm,
                         (const double*)s64.vals.p, Dj, Dk, J, K, s64.nq, b->nmax};
        jk_launch<double>(c, a, st);
    }
    if ((lists & 2) && s32.nq) {
        JkArgs<float> a{(const int2*)s32.q.p, (const PairHdr*)b->d_pairs.p, (const int*)b->d_cart_off.p, dm,
                        (const float*)s32.vals.p, Dj, Dk, J, K, s32.nq, b->nmax};
        jk_launch<float>(c, a, st);
    }
    HIPCHK(hipGetLastError());
    return 0;
}

// One class alone: part 1 the digestion, 2 the ket J reduction of its tiled
// lists, 3 both.
static int jk_launch_class(pq_basis* b, int c, const double* Dj, const double* Dk, double* J, double* K,
                           hipStream_t st, int part = 3, int lists = 3)
{
    if (!jk_tile_fits(b, c)) return jk_launch_untiled(b, c, Dj, Dk, J, K, st, lists);
    if ((part & 1) && jk_group_launch(b, jk_group_table[c], &c, 1, lists, Dj, Dk, J, K, st)) return -1;
    if (part & 2) {
        const int n3 = ncart_l(eri_class_table[c][2]), n4 = ncart_l(eri_class_table[c][3]);
        for (int w = 0; w < 2; ++w) {
            EriClassStore& s = w ? b->store32[c] : b->store64[c];
            if (!((lists >> w) & 1) || !s.nq) continue;
            jket_reduce(jred_list(list_args(b, c), list_bras(s), w, (const double*)s.jkbuf.p, s.nq,
                                  jk_tile_table[c][2], n3 * n4, n4, s.jtiles, s.njtile),
                        (const MolInfo*)b->d_mols.p, J, st);
        }
    }
    HIPCHK(hipGetLastError());
    return 0;
}

// Zero J', K'; digest every stored class; add the ket J values of all tiled
// lists in one reduction launch; symmetrise.  The classes go in one launch per
// register / LDS group (jk_group_table; one launch per class, 21 of them, was
// bound by the host: C10H22 387 us, CH3OH 152 us per build; one kernel over
// every class spilled 2.4 KB a lane), the groups over jk_nstreams streams:
// forked from `st` onto side streams (most stored bytes first, each
// to the least-loaded stream) and joined back before the reduction.  (Each
// class's reduction launched behind its digestion on the side stream instead
// was slower: the many small reduction launches queue behind the digestion
// kernels.)
static void jk_reduce_groups(pq_basis* b, int g0, int g1, double* J, hipStream_t st)
{
    jket_reduce_all((const JredList*)b->d_jred.p + b->jred_list0[g0], b->jred_list0[g1] - b->jred_list0[g0],
                    b->jred_block0[g1] - b->jred_block0[g0], (const MolInfo*)b->d_mols.p, J, st);
}

static int jk_digest_all(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K, hipStream_t st,
                         bool single_stream, bool reduce)
{
    // classes by stored bytes per block, so that the longest blocks start first
    int order[ERI_NCLASS], nc = 0;
    double bytes[ERI_NCLASS] = {}, per[ERI_NCLASS] = {};
    long long blocks = 0;
    bool untiled = false;
    for (int c = 0; c < ERI_NCLASS; ++c) {
        for (int w = 0; w < 2; ++w) {
            const EriClassStore& s = w ? b->store32[c] : b->store64[c];
            bytes[c] += (double)s.nq * s.ncomp * (w ? 4.0 : 8.0) + 16.0 * s.nq;
        }
        if (!(bytes[c] > 0.0)) continue;
        if (!jk_tile_fits(b, c)) {
            untiled = true;
            continue;
        }
        JkClassArgs a;
        const int nb = jk_class_args(b, c, 3, a);
        per[c] = bytes[c] / std::max(1, nb);
        blocks += nb;
        int k = nc++;
        for (; k > 0 && per[order[k - 1]] < per[c]; --k) order[k] = order[k - 1];
        order[k] = c;
    }
    jk_clock_set(b, 0, st);
    if (untiled)
        for (int c = 0; c < ERI_NCLASS; ++c)
            if (bytes[c] > 0.0 && !jk_tile_fits(b, c) && jk_launch_untiled(b, c, Dj, Dk, J, K, st, 3)) return -1;
    int in[JK_NGROUP][ERI_NCLASS], ng[JK_NGROUP] = {};
    double gb[JK_NGROUP] = {};
    int gorder[JK_NGROUP], n = 0;
    for (int k = 0; k < nc; ++k) {
        const int c = order[k], g = jk_group_table[c];
        in[g][ng[g]++] = c;
        gb[g] += bytes[c];
    }
    for (int g = 0; g < JK_NGROUP; ++g) {
        if (!ng[g]) continue;
        int k = n++;
        for (; k > 0 && gb[gorder[k - 1]] < gb[g]; --k) gorder[k] = gorder[k - 1];
        gorder[k] = g;
    }
    // The caller's stream is one of the ns streams (its first group starts
    // behind the zero fill with no cross-stream wait), side streams the rest.
    // Below 400 MB of stored integrals every group goes on the caller's
    // stream: the fork and join cost more than the overlap of the groups'
    // ends gains (CH3OH 99 us on four streams, 52 on one; C7H15OH, 150 MB, two
    // digestions, 458 / 441; C10H22, 0.55 GB, 309 / 315; C14H30 613 / 654).
    const bool small = gb[0] + gb[1] + gb[2] + gb[3] < 400e6;
    const int ns = single_stream || small ? 1 : std::min(n, std::min(4, std::max(1, b->jk_nstreams)));
    // From 1 GB on a group's ket J values are summed behind it on its stream,
    // while other groups still run and its values may still lie in the
    // Infinity Cache (C20H42, 2.9 GB: 1143 us with one launch for all behind
    // the join, 1117 so); below, the launches cost more (C10H22 285 / 291).
    const bool behind = ns > 1 && gb[0] + gb[1] + gb[2] + gb[3] >= 1e9;
    if (ns > 1) {
        if (ensure_jk_streams(b)) return -1;
        HIPCHK(hipEventRecord(b->ev_fork, st));
        for (int k = 1; k < ns; ++k) HIPCHK(hipStreamWaitEvent(b->jk_side[k - 1], b->ev_fork, 0));
    }
    double load[4] = {0.0, 0.0, 0.0, 0.0};
    for (int q = 0; q < n; ++q) {
        const int g = gorder[q];
        int k = 0;
        for (int t = 1; t < ns; ++t)
            if (load[t] < load[k]) k = t;
        load[k] += gb[g];
        hipStream_t sk = k > 0 ? b->jk_side[k - 1] : st;
        if (jk_group_launch(b, g, in[g], ng[g], 3, Dj, Dk, J, K, sk)) return -1;
        if (reduce && behind) jk_reduce_groups(b, g, g + 1, J, sk);
    }
    for (int k = 1; k < ns; ++k) {
        HIPCHK(hipEventRecord(b->ev_join[k - 1], b->jk_side[k - 1]));
        HIPCHK(hipStreamWaitEvent(st, b->ev_join[k - 1], 0));
    }
    if (reduce && !behind) jk_reduce_groups(b, 0, JK_NGROUP, J, st);
    jk_clock_set(b, 1, st);
    return 0;
}

static void jk_zero(pq_basis* b, double* J, double* K, hipStream_t st)
{
    const long long tot = b->mat_total;
    long long blocks = (tot + 255) / 256;
    blocks = blocks > 4096 ? 4096 : (blocks < 1 ? 1 : blocks);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)blocks), dim3(256), 0, st, J, tot, K);
}

static int jk_launch_all(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K, hipStream_t st)
{
    const MolInfo* dm = (const MolInfo*)b->d_mols.p;
    jk_zero(b, J, K, st);
    if (jk_digest_all(b, Dj, Dk, J, K, st, false, true)) return -1;
    int gx = (int)((b->nmax * (long long)b->nmax + 255) / 256);
    gx = gx < 1 ? 1 : (gx > 64 ? 64 : gx);
    hipLaunchKernelGGL(jk_finish_kernel, dim3(gx, b->nmol), dim3(256), 0, st, J, K, dm);
    HIPCHK(hipGetLastError());
    return 0;
}

// Number of streams the J/K class launches spread over (1..4).
extern "C" int pq_jk_set_streams(pq_basis* b, int nstreams)
{
    if (!b || nstreams < 1 || nstreams > 4) return fail("pq_jk_set_streams: need a basis and 1..4 streams");
    b->jk_nstreams = nstreams;
    return 0;
}

// Tunables of one class's J/K digestion: work-item length (run_len, 0 =
// automatic) and blocks launched (grid, 0 = one per item; smaller = persistent).
extern "C" int pq_jk_set_params(pq_basis* b, int cls, int run_len, int grid, void* stream)
{
    if (!b || cls < 0 || cls >= ERI_NCLASS) return fail("pq_jk_set_params: bad class");
    hipStream_t st = (hipStream_t)stream;
    for (int w = 0; w < 2; ++w) {
        EriClassStore& s = w ? b->store32[cls] : b->store64[cls];
        s.jk_run = run_len;
        s.jk_grid = grid;
    }
    if (build_items(b, cls, st)) return -1;
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

// Digest one FP64 class into J', K' (no zero fill, no symmetrisation): timing
// unit for the autotuner and the roofline.  part: 1 = tiled digestion kernel
// only, 2 = ket J reduction only (reads what part 1 stored), 3 = both.
// Returns the number of work items in *nitems.
extern "C" int pq_jk_class(pq_basis* b, int cls, int part, const double* Dj, const double* Dk, double* J, double* K,
                           int* nitems, void* stream)
{
    if (!b || cls < 0 || cls >= ERI_NCLASS || !Dj || !Dk || !J || !K) return fail("pq_jk_class: bad argument");
    if (part < 1 || part > 3) return fail("pq_jk_class: part must be 1, 2 or 3");
    hipStream_t st = (hipStream_t)stream;
    if (!jk_tile_fits(b, cls)) return fail("pq_jk_class: LDS rows too large for this basis");
    EriClassStore& s = b->store64[cls];
    if (nitems) *nitems = s.nitems;
    return jk_launch_class(b, cls, Dj, Dk, J, K, st, part, 1);
}

extern "C" int pq_jk(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K, void* stream)
{
    if (!b || !Dj || !Dk || !J || !K) return fail("pq_jk: null argument");
    hipStream_t st = (hipStream_t)stream;
    if (b->timing) {
        if (ensure_events(b)) return -1;
        HIPCHK(hipEventRecord(b->ev_jk[0], st));
    }
    if (jk_launch_all(b, Dj, Dk, J, K, st)) return -1;
    if (b->timing) {
        HIPCHK(hipEventRecord(b->ev_jk[1], st));
        b->ev_jk_used = 1;
    }
    return 0;
}

// J/K for densities that need not be symmetric (the co-densities of NOCI).
// Two digestions over the stored integrals: Dk into a scratch K2' (with the
// symmetrised Dj into a scratch J2'), then Dk^T into K' with the symmetrised
// Dj into J' (the ket J reduction reads what this last digestion stored);
// then the general finish.  scratch: 4 mat_total doubles (Ds, Dk^T, J2',
// K2').  single_stream: every launch on `st`, classes in index order (no
// side-stream fork, no host containers, no timing events).
static int jk_general_run(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K, double* scratch,
                          bool single_stream, hipStream_t st)
{
    const long long tot = b->mat_total;
    double* Ds = scratch;
    double* DkT = Ds + tot;
    double* J2 = DkT + tot;
    double* K2 = J2 + tot;
    const MolInfo* dm = (const MolInfo*)b->d_mols.p;
    int gx = (int)((b->nmax * (long long)b->nmax + 255) / 256);
    gx = gx < 1 ? 1 : (gx > 64 ? 64 : gx);
    hipLaunchKernelGGL(jk_general_prep_kernel, dim3(gx, b->nmol), dim3(256), 0, st, Dj, Dk, Ds, DkT, dm);
    for (int pass = 0; pass < 2; ++pass) {
        double* Jp = pass ? J : J2;
        double* Kp = pass ? K : K2;
        const double* Dkp = pass ? (const double*)DkT : Dk;
        jk_zero(b, Jp, Kp, st);
        if (jk_digest_all(b, Ds, Dkp, Jp, Kp, st, single_stream, pass == 1)) return -1;   // J is the second pass's
    }
    hipLaunchKernelGGL(jk_general_finish_kernel, dim3(gx, b->nmol), dim3(256), 0, st, J, K, K2, dm);
    HIPCHK(hipGetLastError());
    return 0;
}

extern "C" int pq_jk_general(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K, void* stream)
{
    if (!b || !Dj || !Dk || !J || !K) return fail("pq_jk_general: null argument");
    hipStream_t st = (hipStream_t)stream;
    if (b->d_jkgen.ensure(sizeof(double) * 4 * (size_t)b->mat_total)) return -1;
    if (b->timing) {
        if (ensure_events(b)) return -1;
        HIPCHK(hipEventRecord(b->ev_jk[0], st));
    }
    if (jk_general_run(b, Dj, Dk, J, K, (double*)b->d_jkgen.p, false, st)) return -1;
    if (b->timing) {
        HIPCHK(hipEventRecord(b->ev_jk[1], st));
        b->ev_jk_used = 1;
    }
    return 0;
}

// ---------------------------------------------------------------------------
// pq_jk_general without allocation.  Its four scratch matrices live in a
// file-scope device array, one copy per GPU for the life of the process.  In
// host code `scratch` names a host-side stand-in, not device memory: the
// device address of each GPU's copy comes from hipGetSymbolAddress, taken
// once per device (with that device current) on the first call there, and
// only that address is handed to kernels.  Calls that overlap on one GPU
// share the array and race; each call overwrites all it reads (the
// symmetrised density and Dk^T by the prep kernel, J2'/K2' by the zero fill).
#define PQ_JKGEN_STATIC_ELEMS (1 << 19)     // packed matrix elements: n <= 724 for one molecule
#define PQ_MAX_GPUS 64
static __device__ __align__(256) double scratch[4 * (size_t)PQ_JKGEN_STATIC_ELEMS];
static double* g_scratch_dev[PQ_MAX_GPUS];
static std::mutex g_scratch_mu;

static double* static_scratch_of_current_device()
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= PQ_MAX_GPUS) {
        fail("pq_jk_general_noalloc: no current device in range");
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            fail(std::string("pq_jk_general_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_dev[dev] = (double*)p;
    }
    return g_scratch_dev[dev];
}

extern "C" int pq_jk_general_noalloc(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K,
                                     void* stream)
{
    if (!b || !Dj || !Dk || !J || !K) return fail("pq_jk_general_noalloc: null argument");
    if (b->mat_total > PQ_JKGEN_STATIC_ELEMS)
        return fail("pq_jk_general_noalloc: " + std::to_string(b->mat_total) +
                    " packed matrix elements exceed the static scratch's " + std::to_string(PQ_JKGEN_STATIC_ELEMS) +
                    " (use pq_jk_general)");
    double* sc = static_scratch_of_current_device();
    if (!sc) return -1;
    return jk_general_run(b, Dj, Dk, J, K, sc, true, (hipStream_t)stream);
}

// J/K captured once into a HIP graph (kernel nodes only) for fixed device
// buffers, then replayed: the per-iteration Fock build of batched SCF.
extern "C" int pq_jk_graph_create(pq_basis* b, const double* Dj, const double* Dk, double* J, double* K)
{
    if (!b || !Dj || !Dk || !J || !K) return fail("pq_jk_graph_create: null argument");
    if (b->graph_exec) { (void)hipGraphExecDestroy(b->graph_exec); b->graph_exec = nullptr; }
    // side streams and their events must exist before the capture begins
    if (b->jk_nstreams > 1 && ensure_jk_streams(b)) return -1;
    hipStream_t cs;
    HIPCHK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    hipGraph_t g;
    HIPCHK(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
    const int rc = jk_launch_all(b, Dj, Dk, J, K, cs);
    hipError_t e = hipStreamEndCapture(cs, &g);
    if (rc || e != hipSuccess) {
        const std::string why = rc ? g_err : std::string(hipGetErrorString(e));
        (void)hipStreamDestroy(cs);
        return fail("pq_jk_graph_create: capture failed: " + why);
    }
    e = hipGraphInstantiate(&b->graph_exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    (void)hipStreamDestroy(cs);
    if (e != hipSuccess) return fail(std::string("pq_jk_graph_create: instantiate: ") + hipGetErrorString(e));
    return 0;
}

extern "C" int pq_jk_graph_launch(pq_basis* b, void* stream)
{
    if (!b || !b->graph_exec) return fail("pq_jk_graph_launch: no graph");
    HIPCHK(hipGraphLaunch(b->graph_exec, (hipStream_t)stream));
    return 0;
}

extern "C" int pq_eri_dense(pq_basis* b, double* out, void* stream)
{
    if (!b || !out) return fail("pq_eri_dense: null argument");
    if (b->nmol != 1) return fail("pq_eri_dense: single-molecule basis only");
    hipStream_t st = (hipStream_t)stream;
    const size_t n = b->ncart;
    HIPCHK(hipMemsetAsync(out, 0, sizeof(double) * n * n * n * n, st));
    for (int c = 0; c < ERI_NCLASS; ++c) {
        for (int w = 0; w < 2; ++w) {
            EriClassStore& s = w ? b->store32[c] : b->store64[c];
            if (!s.nq) continue;
            if (w) {
                ScatterArgs<float> a{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p, (const int*)b->d_cart_off.p,
                                     (const float*)s.vals.p, out, s.nq, (int)n, 0, (int)n};
                scatter_launch<float>(c, a, st);
            } else {
                ScatterArgs<double> a{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p, (const int*)b->d_cart_off.p,
                                      (const double*)s.vals.p, out, s.nq, (int)n, 0, (int)n};
                scatter_launch<double>(c, a, st);
            }
        }
    }
    HIPCHK(hipGetLastError());
    return 0;
}

// Arbitrary shell quartets -> Cartesian normalised blocks in caller shell
// order, packed one after another into out_host (Level-B two_electron).
extern "C" int pq_eri_blocks(pq_basis* b, int n, const int* shells, double* out_host, void* stream)
{
    if (!b || (n > 0 && (!shells || !out_host))) return fail("pq_eri_blocks: null argument");
    hipStream_t st = (hipStream_t)stream;
    // group by class in canonical orientation
    struct Item { int cls, idx, P, Q, swapq; };
    std::vector<Item> items(n);
    std::vector<size_t> out_off(n + 1, 0);
    for (int i = 0; i < n; ++i) {
        const int* s = shells + 4 * i;
        for (int k = 0; k < 4; ++k)
            if (s[k] < 0 || s[k] >= b->nshell) return fail("pq_eri_blocks: shell index out of range");
        int P = pair_id(b, s[0], s[1]);
        int Q = pair_id(b, s[2], s[3]);
        if (P < 0 || Q < 0 || b->pairs[P].mol != b->pairs[Q].mol)
            return fail("pq_eri_blocks: shells of one quartet must belong to one molecule");
        int X = b->pairs[P].pcls, Y = b->pairs[Q].pcls;
        int swapq = 0;
        if (Y > X) { std::swap(P, Q); std::swap(X, Y); swapq = 1; }
        items[i] = {class_of_pair_classes(X, Y), i, P, Q, swapq};
        out_off[i + 1] = out_off[i] + (size_t)ncart_l(b->l[s[0]]) * ncart_l(b->l[s[1]]) * ncart_l(b->l[s[2]]) *
                                          ncart_l(b->l[s[3]]);
    }
    for (int c = 0; c < ERI_NCLASS; ++c) {
        std::vector<int2> hq;
        std::vector<int> which;
        for (int i = 0; i < n; ++i)
            if (items[i].cls == c) { hq.push_back(make_int2(items[i].P, items[i].Q)); which.push_back(i); }
        if (hq.empty()) continue;
        const int m = (int)hq.size(), ncomp = eri_class_table[c][4];
        DevBuf dq, dv;
        if (dq.ensure(sizeof(int2) * m) || dv.ensure(sizeof(double) * (size_t)m * ncomp)) return -1;
        HIPCHK(hipMemcpyAsync(dq.p, hq.data(), sizeof(int2) * m, hipMemcpyHostToDevice, st));
        if (run_class<double>(b, c, (const int2*)dq.p, m, (double*)dv.p, st)) return -1;
        std::vector<double> hv((size_t)m * ncomp);
        HIPCHK(hipMemcpyAsync(hv.data(), dv.p, sizeof(double) * hv.size(), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        const int l1 = eri_class_table[c][0], l2 = eri_class_table[c][1], l3 = eri_class_table[c][2],
                  l4 = eri_class_table[c][3];
        const int n1 = ncart_l(l1), n2 = ncart_l(l2), n3 = ncart_l(l3), n4 = ncart_l(l4);
        for (int k = 0; k < m; ++k) {
            const Item& it = items[which[k]];
            const int* s = shells + 4 * it.idx;
            // canonical block [c1][c2][c3][c4] with pair shells (pairs[P].s1, .s2 | pairs[Q].s1, .s2)
            const PairHdr& hp = b->pairs[it.P];
            const PairHdr& hq2 = b->pairs[it.Q];
            // map caller position -> canonical slot
            int want[4] = {s[0], s[1], s[2], s[3]};
            int can[4] = {hp.s1, hp.s2, hq2.s1, hq2.s2};
            // caller pair order (0,1 | 2,3); canonical may have swapped pairs and/or shells within pairs
            int pos[4];   // pos[k] = canonical index of caller slot k
            {
                int cb[2] = {it.swapq ? 2 : 0, it.swapq ? 0 : 2};   // canonical pair base for caller bra/ket
                for (int pk = 0; pk < 2; ++pk) {
                    const int base = cb[pk];
                    const int c0 = can[base], c1 = can[base + 1];
                    const int w0 = want[2 * pk], w1 = want[2 * pk + 1];
                    if (c0 == w0 && c1 == w1) { pos[2 * pk] = base; pos[2 * pk + 1] = base + 1; }
                    else { pos[2 * pk] = base + 1; pos[2 * pk + 1] = base; }
                    (void)c1; (void)w1;
                }
            }
            const int nn[4] = {n1, n2, n3, n4};
            const int cw[4] = {ncart_l(b->l[s[0]]), ncart_l(b->l[s[1]]), ncart_l(b->l[s[2]]), ncart_l(b->l[s[3]])};
            double* dst = out_host + out_off[it.idx];
            int idx[4];
            for (idx[0] = 0; idx[0] < cw[0]; ++idx[0])
                for (idx[1] = 0; idx[1] < cw[1]; ++idx[1])
                    for (idx[2] = 0; idx[2] < cw[2]; ++idx[2])
                        for (idx[3] = 0; idx[3] < cw[3]; ++idx[3]) {
                            int ci[4];
                            for (int t = 0; t < 4; ++t) ci[pos[t]] = idx[t];
                            const size_t comp = ((size_t)(ci[0] * nn[1] + ci[1]) * nn[2] + ci[2]) * nn[3] + ci[3];
                            dst[((idx[0] * cw[1] + idx[1]) * cw[2] + idx[2]) * cw[3] + idx[3]] = hv[comp * m + k];
                        }
        }
    }
    return 0;
}

// --------------------------------------------------------------------------
// MP2 AO->MO transform
// --------------------------------------------------------------------------
static int eri_dense_slab(pq_basis* b, int l0, int lc, double* out, hipStream_t st)
{
    const size_t n = b->ncart;
    HIPCHK(hipMemsetAsync(out, 0, sizeof(double) * n * n * (size_t)lc * n, st));
    for (int c = 0; c < ERI_NCLASS; ++c) {
        for (int w = 0; w < 2; ++w) {
            EriClassStore& s = w ? b->store32[c] : b->store64[c];
            if (!s.nq) continue;
            if (w) {
                ScatterArgs<float> a{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p, (const int*)b->d_cart_off.p,
                                     (const float*)s.vals.p, out, s.nq, (int)n, l0, lc};
                scatter_launch<float>(c, a, st);
            } else {
                ScatterArgs<double> a{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p, (const int*)b->d_cart_off.p,
                                      (const double*)s.vals.p, out, s.nq, (int)n, l0, lc};
                scatter_launch<double>(c, a, st);
            }
        }
    }
    HIPCHK(hipGetLastError());
    return 0;
}

extern "C" int pq_eri_dense_slab(pq_basis* b, int l0, int lc, double* out, void* stream)
{
    if (!b || !out) return fail("pq_eri_dense_slab: null argument");
    if (b->nmol != 1) return fail("pq_eri_dense_slab: single-molecule basis only");
    if (l0 < 0 || lc <= 0 || l0 + lc > b->ncart) return fail("pq_eri_dense_slab: slab out of range");
    return eri_dense_slab(b, l0, lc, out, (hipStream_t)stream);
}

extern "C" int pq_gemm_f64(int ta, int tb, int M, int N, int K, double alpha, const double* A, long long lda,
                           long long sA, const double* B, long long ldb, long long sB, double beta, double* C,
                           long long ldc, long long sC, int batch, void* stream)
{
    if (!A || !B || !C) return fail("pq_gemm_f64: null argument");
    if (M < 0 || N < 0 || K <= 0 || batch < 0) return fail("pq_gemm_f64: bad sizes");
    GemmF64Args g{A, B, C, lda, ldb, ldc, sA, sB, sC, M, N, K, ta, tb, alpha, beta};
    if (long_gemm_f64(long_gemm_of(g), batch, (hipStream_t)stream)) return fail("pq_gemm_f64: launch failed");
    return 0;
}

extern "C" int pq_gemm_bf16x3(int ta, int tb, int M, int N, int K, double alpha, const double* A, long long lda,
                              long long sA, const double* B, long long ldb, long long sB, double beta, double* C,
                              long long ldc, long long sC, int batch, void* stream)
{
    if (!A || !B || !C) return fail("pq_gemm_bf16x3: null argument");
    if (M < 0 || N < 0 || K <= 0 || batch < 0) return fail("pq_gemm_bf16x3: bad sizes");
    GemmF64Args g{A, B, C, lda, ldb, ldc, sA, sB, sC, M, N, K, ta, tb, alpha, beta};
    if (long_gemm_bf16x3(long_gemm_of(g), batch, (hipStream_t)stream)) return fail("pq_gemm_bf16x3: launch failed");
    return 0;
}

// The packed function pairs of a single-molecule basis: first index of every
// shell pair (its functions are neighbours) and the n x n table of indices,
// with PQ_TABPAD rows of zeros behind it, which the products read ahead.
// Built once per basis.
__global__ void pair_table_kernel(const PairHdr* pairs, const int* l, const int* cart_off, const int* base, int npair,
                                  int n, int* tab)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= npair) return;
    const PairHdr h = pairs[t];
    const int l1 = l[h.s1], l2 = l[h.s2];
    const int n1 = (l1 + 1) * (l1 + 2) / 2, n2 = (l2 + 1) * (l2 + 2) / 2;
    const bool same = h.s1 == h.s2;
    for (int i = 0; i < n1; ++i)
        for (int j = 0; j < (same ? i + 1 : n2); ++j) {
            const int p = base[t] + pair_component(same, n2, i, j);
            const int m = cart_off[h.s1] + i, k = cart_off[h.s2] + j;
            tab[(size_t)m * n + k] = p;
            tab[(size_t)k * n + m] = p;
        }
}

static int ensure_pair_table(pq_basis* b, hipStream_t st)
{
    if (b->npacked > 0) return 0;
    const int n = b->ncart;
    std::vector<int> host(b->npair + b->nshell);
    int at = 0;
    for (int t = 0; t < b->npair; ++t) {
        host[t] = at;
        const int n1 = ncart_l(b->l[b->pairs[t].s1]), n2 = ncart_l(b->l[b->pairs[t].s2]);
        at += b->pairs[t].s1 == b->pairs[t].s2 ? n1 * (n1 + 1) / 2 : n1 * n2;
    }
    for (int s = 0; s < b->nshell; ++s) host[b->npair + s] = b->l[s];
    if (b->d_pairbase.ensure(sizeof(int) * host.size()) || b->d_pairtab.ensure(sizeof(int) * (size_t)(n + PQ_TABPAD) * n))
        return -1;
    HIPCHK(hipMemcpyAsync(b->d_pairbase.p, host.data(), sizeof(int) * host.size(), hipMemcpyHostToDevice, st));
    HIPCHK(hipStreamSynchronize(st));   // the host array ends with this call
    const int* base = (const int*)b->d_pairbase.p;
    HIPCHK(hipMemsetAsync((int*)b->d_pairtab.p + (size_t)n * n, 0, sizeof(int) * (size_t)PQ_TABPAD * n, st));
    hipLaunchKernelGGL(pair_table_kernel, dim3((b->npair + 127) / 128), dim3(128), 0, st, (const PairHdr*)b->d_pairs.p,
                       base + b->npair, (const int*)b->d_cart_off.p, base, b->npair, n, (int*)b->d_pairtab.p);
    HIPCHK(hipGetLastError());
    b->npacked = at;
    return 0;
}

// rows [p0, p0 + rows) of the stored integrals' symmetric matrix over packed
// function pairs
static int eri_pair_rows(pq_basis* b, long long p0, long long rows, double* out, hipStream_t st)
{
    HIPCHK(hipMemsetAsync(out, 0, sizeof(double) * (size_t)rows * b->npacked, st));
    for (int c = 0; c < ERI_NCLASS; ++c) {
        const EriClassStore& s = b->store64[c];
        const EriClassStore& f = b->store32[c];
        if (s.nq)
            pairscatter_launch<double>(c, PairScatterArgs<double>{(const int2*)s.q.p, (const PairHdr*)b->d_pairs.p,
                                       (const int*)b->d_pairbase.p, (const double*)s.vals.p, out, p0, rows, b->npacked,
                                       s.nq}, st);
        if (f.nq)
            pairscatter_launch<float>(c, PairScatterArgs<float>{(const int2*)f.q.p, (const PairHdr*)b->d_pairs.p,
                                      (const int*)b->d_pairbase.p, (const float*)f.vals.p, out, p0, rows, b->npacked,
                                      f.nq}, st);
    }
    HIPCHK(hipGetLastError());
    return 0;
}

// The quarter transforms over packed function pairs: (mu nu|lam sig) is kept
// as rows p = (lam sig), lam >= sig, of a matrix symmetric in (mu nu), which
// halves the first two quarters (their flops, their output) and quarters the
// integrals' matrix against the dense tensor; the packed rows are read through
// the n x n index table.  C10H22 (n = 194, o = 41, v = 153), with the energy:
// 22.4 ms over slabs of the dense tensor (scatter 11.0, clear 1.8, products
// 9.0, energy 0.5), 6.1 ms now (scatter 1.7, clear 0.43, products 3.9, energy
// 0.15).
extern "C" int pq_mp2_ovov(pq_basis* b, int o1, int v1, const double* Co1, const double* Cv1, int o2, int v2,
                           const double* Co2, const double* Cv2, double* ovov, long long max_slab_bytes,
                           int precision, void* stream)
{
    if (precision < 0 || precision > 1) return fail("pq_mp2_ovov: precision must be 0 (FP64) or 1 (BF16x3)");
    auto gemm = precision ? long_gemm_bf16x3 : long_gemm_f64;
    if (!b || !Co1 || !Cv1 || !Co2 || !Cv2 || !ovov) return fail("pq_mp2_ovov: null argument");
    if (o1 <= 0 || v1 <= 0 || o2 <= 0 || v2 <= 0) return fail("pq_mp2_ovov: empty orbital space");
    if (b->nmol != 1) return fail("pq_mp2_ovov: single-molecule basis only");
    hipStream_t st = (hipStream_t)stream;
    if (ensure_pair_table(b, st)) return -1;
    const long long n = b->ncart, np = b->npacked;
    long long lc;   // rows p at a time
    if (max_slab_bytes > 0) {
        lc = max_slab_bytes / (8 * np);
    } else {
        // half of the free device memory, less the fixed half-transformed
        // arrays, for the rows and their first quarter (np + o1 n doubles per
        // row): every stored quartet is read and scattered once per slab, so
        // fewer, larger slabs (C20H42: one)
        size_t fr = 0, tot = 0;
        if (hipMemGetInfo(&fr, &tot) != hipSuccess) fr = 8ULL << 30;
        // blocks this library's cache holds count as free: they are reused
        const long long avail = (long long)fr + std::max(0LL, pq_cache_bytes());
        const long long fixed = 8LL * ((long long)o1 * v1 * np + (long long)o1 * v1 * o2 * n);
        const long long budget = std::max(1LL << 30, avail / 2 - fixed);
        lc = budget / (8 * (np + (long long)o1 * n));
    }
    // a slab's columns (rows of p times n) are counted in an int
    lc = std::max(1LL, std::min(std::min(lc, np), ((1LL << 31) - 4096) / n));
    if ((long long)o1 * v1 * std::max(n, (long long)o2) > (1LL << 31) - 4096)
        return fail("pq_mp2_ovov: orbital spaces too large");
    DevBuf rows, t1, t2, t3;
    if (rows.ensure(sizeof(double) * (size_t)(np * lc)) || t1.ensure(sizeof(double) * (size_t)(o1 * n * lc)) ||
        t2.ensure(sizeof(double) * (size_t)((long long)o1 * v1 * np)) ||
        t3.ensure(sizeof(double) * (size_t)((long long)o1 * v1 * o2 * n)))
        return -1;
    const int* tab = (const int*)b->d_pairtab.p;
    int rc = 0;
    for (long long p0 = 0; p0 < np && !rc; p0 += lc) {
        const long long L = std::min(lc, np - p0);
        rc |= eri_pair_rows(b, p0, L, (double*)rows.p, st);
        // (i nu|p) = sum_mu C1[mu][i] (mu nu|p), stored [i][p][nu]
        LongGemm g = {};
        g.alpha = 1.0;
        g.P = Co1; g.ldp = o1; g.M = o1; g.pk = 1;
        g.Q = (const double*)rows.p; g.ldq = np; g.qmode = PQ_QSYM; g.tab = tab; g.cn = (int)n; g.N = (int)(L * n);
        g.C = (double*)t1.p; g.ldc = L * n; g.s1 = n;
        g.K = (int)n;
        rc |= gemm(g, 1, st);
        // (i a|p) = sum_nu C1v[nu][a] (i nu|p), into the full [i][a][p]
        g = LongGemm{};
        g.alpha = 1.0;
        g.P = Cv1; g.ldp = v1; g.M = v1; g.pk = 1;
        g.Q = (const double*)t1.p; g.ldq = n; g.sQ = L * n; g.qmode = PQ_QROW; g.N = (int)L;
        g.C = (double*)t2.p + p0; g.ldc = np; g.sC = (long long)v1 * np;
        g.K = (int)n;
        rc |= gemm(g, o1, st);
    }
    if (!rc) {
        // (i a|j sig) = sum_lam C2[lam][j] (i a|lam sig), stored [i][a][j][sig]
        LongGemm g = {};
        g.alpha = 1.0;
        g.P = Co2; g.ldp = o2; g.M = o2; g.pk = 1;
        g.Q = (const double*)t2.p; g.ldq = np; g.qmode = PQ_QSYM; g.tab = tab; g.cn = (int)n; g.N = (int)(o1 * v1 * n);
        g.C = (double*)t3.p; g.ldc = n; g.s1 = (long long)o2 * n;
        g.K = (int)n;
        rc |= gemm(g, 1, st);
        // (i a|j b) = sum_sig (i a|j sig) C2v[sig][b]
        GemmF64Args gd{(const double*)t3.p, Cv2, ovov, n, v2, v2, 0, 0, 0, o1 * v1 * o2, v2, (int)n, 0, 0, 1.0, 0.0};
        g = long_gemm_of(gd);
        rc |= gemm(g, 1, st);
    }
    hipError_t e = hipStreamSynchronize(st);
    if (rc) return fail("pq_mp2_ovov: kernel launch failed");
    if (e != hipSuccess) return fail(std::string("pq_mp2_ovov: ") + hipGetErrorString(e));
    return 0;
}

// Density projector of the SCF loop by TC2 purification (scf.hip): P =
// projector onto the nocc lowest eigenvectors of the symmetric m x m matrix
// F.  work: 2 m^2 + 4 doubles.  Steps run in chunks of 8 with one host read
// of tr(X - X^2) per chunk; once below tol, one more step.
extern "C" int pq_purify(const double* F, int m, int nocc, double* P, double* work, double tol, int max_steps,
                         int* steps_out, double* idem_out, void* stream)
{
    if (!F || !P || !work) return fail("pq_purify: null argument");
    if (m <= 0 || nocc <= 0 || nocc >= m) return fail("pq_purify: need 0 < nocc < m");
    if (max_steps < 1) return fail("pq_purify: max_steps must be positive");
    if ((uintptr_t)work % 32) return fail("pq_purify: work must be 32-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    Tc2Work w = tc2_work(work, m, max_steps);
    if (tc2_start(F, w, st)) return fail("pq_purify: launch failed");
    // Queue the step count of this thread's previous call on the fast step
    // kernel, 4 more on the early-exit one, then 16 at a time (early-exit):
    // the steps record where to stop and the ones queued past it store
    // nothing, so one host round trip usually suffices.
    static thread_local int usual = 44;
    std::vector<double> h(2 * (size_t)max_steps + 1);
    int queued = 0, stop = 0x7fffffff;
    int chunk = std::min(max_steps, usual);
    for (bool first = true;; first = false) {
        if (tc2_steps(w, nocc, tol, queued, chunk, st, !first)) return fail("pq_purify: launch failed");
        queued += chunk;
        if (first) {
            const int extra = std::min(4, max_steps - queued);
            if (extra > 0 && tc2_steps(w, nocc, tol, queued, extra, st, true)) return fail("pq_purify: launch failed");
            queued += extra;
        }
        HIPCHK(hipMemcpyAsync(h.data(), w.t, sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        memcpy(&stop, &h[2 * (size_t)max_steps], sizeof stop);
        if (stop < queued || queued >= max_steps) break;
        chunk = std::min(16, max_steps - queued);
    }
    if (tc2_finish(w, nocc, queued, P, st)) return fail("pq_purify: launch failed");
    const int last = std::min(stop, queued - 1);
    usual = last + 1;
    if (steps_out) *steps_out = last + 1;
    if (idem_out) *idem_out = last >= 1 ? h[2 * (size_t)(last - 1)] - h[2 * (size_t)(last - 1) + 1] : 1.0;
    return 0;
}

// Scalars of one SCF cycle (energy terms, DIIS overlaps, residual maxima)
// in two launches and one device-to-host copy.
extern "C" long long pq_scf_dots_work(long long n, int nout) { return scf_dots_work(n, nout); }

extern "C" int pq_scf_dots(const double* const* x, const double* const* y, int npair, const double* const* r, int nr,
                           long long n, double* work, double* out_host, void* stream)
{
    if (npair < 0 || npair > SCF_MAXDOT || nr < 0 || nr > 2 || n <= 0 || !work || !out_host)
        return fail("pq_scf_dots: bad argument (npair <= 24, nr <= 2, n > 0)");
    if (npair + nr == 0) return 0;
    ScfDotArgs a = {};
    for (int i = 0; i < npair; ++i) {
        if (!x[i] || !y[i]) return fail("pq_scf_dots: null operand");
        a.x[i] = x[i];
        a.y[i] = y[i];
    }
    for (int j = 0; j < nr; ++j) {
        if (!r[j]) return fail("pq_scf_dots: null operand");
        a.r[j] = r[j];
    }
    a.npair = npair;
    a.nr = nr;
    a.n = n;
    hipStream_t st = (hipStream_t)stream;
    if (scf_dots(a, work, st)) return fail("pq_scf_dots: launch failed");
    const int nout = npair + 2 * nr;
    HIPCHK(hipMemcpyAsync(out_host, work + (size_t)scf_dots_blocks(n) * nout, sizeof(double) * nout,
                          hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

// out = sum_i c_i m_i (k <= 16 device matrices of n elements).
extern "C" int pq_lincomb(const double* const* m, const double* c, int k, long long n, double* out, void* stream)
{
    if (k < 1 || k > SCF_MAXCOMB || n <= 0 || !m || !c || !out) return fail("pq_lincomb: bad argument (1 <= k <= 16)");
    LinCombArgs a = {};
    for (int i = 0; i < k; ++i) {
        if (!m[i]) return fail("pq_lincomb: null matrix");
        a.m[i] = m[i];
        a.c[i] = c[i];
    }
    a.k = k;
    a.n = n;
    if (lincomb(a, out, (hipStream_t)stream)) return fail("pq_lincomb: launch failed");
    return 0;
}

extern "C" int pq_mp2_energy(const double* ovov, const double* eo1, const double* ev1, const double* eo2,
                             const double* ev2, int o1, int v1, int o2, int v2, int mode, double* out_host,
                             void* stream)
{
    if (!ovov || !eo1 || !ev1 || !eo2 || !ev2 || !out_host) return fail("pq_mp2_energy: null argument");
    if (mode < 0 || mode > 2) return fail("pq_mp2_energy: mode must be 0, 1 or 2");
    if (mode != 2 && (o1 != o2 || v1 != v2)) return fail("pq_mp2_energy: modes 0/1 need equal spaces");
    hipStream_t st = (hipStream_t)stream;
    DevBuf acc;
    if (acc.ensure(sizeof(double))) return -1;
    HIPCHK(hipMemsetAsync(acc.p, 0, sizeof(double), st));
    if (mp2_energy_launch(ovov, eo1, ev1, eo2, ev2, o1, v1, o2, v2, mode, (double*)acc.p, st))
        return fail("pq_mp2_energy: launch failed");
    HIPCHK(hipMemcpyAsync(out_host, acc.p, sizeof(double), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    acc.release();
    return 0;
}

// --------------------------------------------------------------------------
// Learned-guess MLP (FP32)
// --------------------------------------------------------------------------
extern "C" int pq_mlp_linear_fwd(const float* X, const float* W, const float* b, float* Z, float* A, int B, int I,
                                 int O, int act, void* stream)
{
    if (!X || !W || !Z) return fail("pq_mlp_linear_fwd: null argument");
    if (act < 0 || act > 1) return fail("pq_mlp_linear_fwd: act must be 0 or 1");
    if (mlp_linear_fwd(X, W, b, Z, A, B, I, O, act, (hipStream_t)stream)) return fail("pq_mlp_linear_fwd: launch failed");
    return 0;
}

extern "C" int pq_mlp_linear_bwd(const float* X, const float* W, const float* A, const float* dA, float* dZ,
                                 float* dX, float* dW, float* db, int B, int I, int O, int act, void* stream)
{
    if (!X || !W || !A || !dA || !dZ || !dW || !db) return fail("pq_mlp_linear_bwd: null argument");
    if (act < 0 || act > 1) return fail("pq_mlp_linear_bwd: act must be 0 or 1");
    if (mlp_linear_bwd(X, W, A, dA, dZ, dX, dW, db, B, I, O, act, (hipStream_t)stream))
        return fail("pq_mlp_linear_bwd: launch failed");
    return 0;
}

extern "C" int pq_mlp_mse(const float* Y, const float* T, const float* mask, float* dY, float* loss_dev, long long n,
                          float inv_norm, void* stream)
{
    if (!Y || !T || !dY || !loss_dev) return fail("pq_mlp_mse: null argument");
    if (mlp_mse(Y, T, mask, dY, loss_dev, n, inv_norm, (hipStream_t)stream)) return fail("pq_mlp_mse: launch failed");
    return 0;
}

extern "C" int pq_mlp_forward(int nlayer, const int* dims, const float* X, const float* const* W,
                              const float* const* b, float* const* A, int B, void* stream)
{
    if (nlayer <= 0 || nlayer > MLP_MAX_LAYERS) return fail("pq_mlp_forward: 1 to 8 layers");
    if (!dims || !X || !W || !b || !A || !A[nlayer - 1]) return fail("pq_mlp_forward: null argument");
    for (int l = 0; l < nlayer; ++l)
        if (!W[l] || !b[l]) return fail("pq_mlp_forward: null argument");
    const int rc = mlp_forward(nlayer, dims, X, W, b, A, B, (hipStream_t)stream);
    if (rc == -2) return fail("pq_mlp_forward: layers wider than 448 need every output buffer");
    if (rc) return fail("pq_mlp_forward: launch failed");
    return 0;
}

extern "C" int pq_mlp_backward(int nlayer, const int* dims, const float* X, const float* const* A,
                               const float* const* W, const float* dY, float* const* dZ, float* const* dW,
                               float* const* db, int B, void* stream)
{
    if (nlayer <= 0 || nlayer > MLP_MAX_LAYERS) return fail("pq_mlp_backward: 1 to 8 layers");
    if (!dims || !X || !A || !W || !dY || !dZ || !dW || !db) return fail("pq_mlp_backward: null argument");
    for (int l = 0; l < nlayer; ++l)
        if (!W[l] || !dW[l] || !db[l] || (l + 1 < nlayer && (!A[l] || !dZ[l])))
            return fail("pq_mlp_backward: null argument");
    if (mlp_backward(nlayer, dims, X, A, W, dY, dZ, dW, db, B, (hipStream_t)stream))
        return fail("pq_mlp_backward: launch failed");
    return 0;
}

extern "C" int pq_mlp_adam(float* p, const float* g, float* m, float* v, long long n, float lr, float b1, float b2,
                           float eps, int step, void* stream)
{
    if (!p || !g || !m || !v) return fail("pq_mlp_adam: null argument");
    if (mlp_adam(1, &p, &g, &m, &v, &n, lr, b1, b2, eps, step, (hipStream_t)stream))
        return fail("pq_mlp_adam: launch failed");
    return 0;
}

extern "C" int pq_mlp_adam_multi(int nt, float* const* p, const float* const* g, float* const* m, float* const* v,
                                 const long long* n, float lr, float b1, float b2, float eps, int step, void* stream)
{
    if (nt <= 0 || nt > MLP_MAX_TENSORS) return fail("pq_mlp_adam_multi: 1 to 16 tensors");
    if (!p || !g || !m || !v || !n) return fail("pq_mlp_adam_multi: null argument");
    for (int t = 0; t < nt; ++t)
        if (!p[t] || !g[t] || !m[t] || !v[t]) return fail("pq_mlp_adam_multi: null argument");
    if (mlp_adam(nt, p, g, m, v, n, lr, b1, b2, eps, step, (hipStream_t)stream))
        return fail("pq_mlp_adam_multi: launch failed");
    return 0;
}
