/* pychem_hip.h -- C ABI of the MI355X integral + Fock-build engine.
 *
 * Drop-in replacement for the reference's `_c_ints` CPython extension
 * (Methods/_c_ints.c:68-81) and the per-class driver loops above it
 * (Methods/integrals.py, Methods/hartree_fock.py).  Where the reference
 * crosses Python->C once per recurrence class of one shell quartet, these
 * entry points are batched and device resident: the basis is uploaded once,
 * integrals stay in HBM, and the SCF loop calls pq_jk once per iteration.
 *
 * Conventions: every function returns 0 on success and a negative value on
 * failure (message via pq_last_error()).  Pointers named *_dev / matrices
 * are device pointers; `stream` is a hipStream_t (NULL = default stream).
 * Matrices are row-major float64 over Cartesian basis functions in the
 * reference's global order (atoms, shells in basis order, components lx desc
 * then ly desc).  Coordinates in bohr.  ERIs in chemists' notation (ab|cd).
 */
#ifndef PYCHEM_HIP_H
#define PYCHEM_HIP_H
#ifdef __cplusplus
extern "C" {
#endif

typedef struct pq_basis pq_basis;

/* Last error message of the calling thread. */
const char* pq_last_error(void);
/* ABI version (1). */
int pq_version(void);
/* Number of visible GPUs. */
int pq_device_count(void);
/* Device memory cache of the library (no reference counterpart: the
 * reference holds its integrals in host memory).  Buffers a basis releases
 * stay cached for the next basis; pq_cache_release frees every cached block
 * of the current device (synchronising it), pq_cache_bytes reports how many
 * bytes are cached there. */
int pq_cache_release(void);
long long pq_cache_bytes(void);

/* Boys function F_m(T), m = 0..mmax (mmax <= 8), out[n][mmax+1].
 * Replaces the interpolation in Methods/c_ints/two_electron_fundamentals.c:60-85
 * and one_electron_fundamentals.c:57-96. */
int pq_boys(int n, const double* T_dev, int mmax, double* out_dev, void* stream);

/* Upload shells (l <= 2) and atoms; builds all shell pairs a <= b with their
 * primitive-pair quantities.  Replaces the per-pair
 * _c_ints.shellpair_quantities call (Methods/_c_ints.c:114-155, called from
 * Util/structures.py:931).  cc = contraction coefficients already scaled by
 * (2 alpha)^((l+1.5)/2) (Util/structures.py:843). */
int pq_basis_create(int nshell, const int* l, const int* nprim, const int* prim_off,
                    const double* center, const double* exps, const double* cc,
                    int natom, const double* atom_xyz, const double* atom_z,
                    pq_basis** out);
/* Many molecules in one handle (no reference counterpart: the reference
 * builds one Molecule at a time, Util/structures.py:319-806).  shell_mol[nshell]
 * and atom_mol[natom] give each shell's and atom's molecule (0..nmol-1,
 * non-decreasing).  Shell pairs, quartets and the one-electron nuclear sum
 * stay inside one molecule; matrices are packed per molecule, molecule m's
 * n_m x n_m block starting at element base_m (pq_basis_molecules).  NULL
 * shell_mol/atom_mol with nmol = 1 is pq_basis_create. */
int pq_basis_create_batch(int nmol, int nshell, const int* l, const int* nprim, const int* prim_off,
                          const double* center, const double* exps, const double* cc, const int* shell_mol,
                          int natom, const double* atom_xyz, const double* atom_z, const int* atom_mol,
                          pq_basis** out);
/* Per molecule m < nmol: packed base offset, Cartesian size n, atom range
 * [atom_lo, atom_hi).  Any output may be NULL. */
int pq_basis_molecules(const pq_basis* b, long long* base, int* n, int* atom_lo, int* atom_hi);
void pq_basis_destroy(pq_basis* b);
/* Mark spherical (5d) shells, spher[nshell] in {0,1} (Util/structures.py:844-849).
 * Only affects Schwarz bounds, which the reference takes in the final basis;
 * all matrices stay Cartesian and the caller applies cart->spherical. */
int pq_basis_set_spherical(pq_basis* b, const int* spher);
/* info[0..6] = ncart, nshell, npair, nprimpair, nmol, packed matrix
 * elements (sum of n_m^2), largest n_m. */
int pq_basis_info(const pq_basis* b, long long* info);

/* Overlap, kinetic and nuclear-attraction matrices (Cartesian, normalised).
 * Replaces integrals.one_electron over all pairs (Methods/integrals.py:220-370)
 * i.e. _c_ints.one_electron_{fundamentals,vrr,hrr,kinetic,contract}
 * (Methods/_c_ints.c:380-644), as used by make_core_matrices
 * (Methods/hartree_fock.py:207-223). */
int pq_one_electron(pq_basis* b, double* S_dev, double* T_dev, double* V_dev, void* stream);

/* Schwarz bounds per shell pair: max over functions of sqrt((mn|mn))
 * (Methods/hartree_fock.py:244-254).  pair_bound_host (nshell*nshell) may be
 * NULL. */
int pq_schwarz(pq_basis* b, double* pair_bound_host, void* stream);

/* The two-electron operator of every later Schwarz pass and ERI build:
 * ints_type 0 the Coulomb operator, 1 the elastic electron-scattering
 * operator at momentum transfer grid_value (>= 0), FP64 only.  Replaces the
 * ints_type / grid_value arguments of _c_ints.two_electron_fundamentals
 * (Methods/_c_ints.c:216-239, Methods/c_ints/two_electron_scattering.c:6-84,
 * spherical_bessel_j.c:5-81).  A change of operator makes the next
 * pq_eri_plan take the Schwarz bounds again with it. */
int pq_eri_set_operator(pq_basis* b, int ints_type, double grid_value);

/* Screened unique ERIs into HBM: quartets with bound product > threshold
 * (plus every diagonal (P|P)), Methods/hartree_fock.py:241-325 with the
 * per-quartet integrals.two_electron (Methods/integrals.py:427-555, i.e.
 * _c_ints.two_electron_{fundamentals,vrr,contract,hrr}, Methods/_c_ints.c:
 * 157-378).  Quartets whose bound product is below fp32_threshold are
 * computed and stored in FP32 (0 disables the split). */
int pq_eri_build(pq_basis* b, double threshold, double fp32_threshold, void* stream);
/* pq_eri_build in two steps: plan (Schwarz if needed, screened class lists,
 * HBM allocation) and compute (all class kernels over the planned lists). */
int pq_eri_plan(pq_basis* b, double threshold, double fp32_threshold, void* stream);
int pq_eri_compute(pq_basis* b, void* stream);
/* Recompute the stored ERIs over the same quartet lists (= pq_eri_compute). */
int pq_eri_recompute(pq_basis* b, void* stream);
/* Live kernel timing with hipEvents on the caller's stream (on != 0). */
int pq_set_timing(pq_basis* b, int on);
/* ms of the last timed ERI pass per class, eri_ms[2*nclass] (slot 2c: FP64
 * list, 2c+1: FP32 list, -1 if not launched; the classes run concurrently on
 * side streams), of the whole pass (eri_pass_ms, on the caller's stream) and
 * of the last pq_jk call.  Outputs may be NULL. */
int pq_get_timings(pq_basis* b, double* eri_ms, double* jk_ms, double* eri_pass_ms);
/* Per-class J/K digestion times summed over the J/K calls made with timing
 * on (pq_jk, pq_jk_general and the J/K of pq_scf_run): from the start of the
 * class's first block to the end of its last, by the GPU's realtime clock (the
 * classes share launches); the number of calls and each class's J/K work
 * items, ERI_NCLASS entries each (any may be NULL); reset != 0 clears the
 * sums.  Waits for the device.  No reference counterpart (measurement). */
int pq_jk_class_times(pq_basis* b, double* sum_ms, long long* launches, long long* nitems, int reset);
/* Recompute one class of the stored ERIs: cls in [0, pq_eri_nclass()),
 * w = 0 for the FP64 list, 1 for the FP32 list. */
int pq_eri_run_class(pq_basis* b, int cls, int w, void* stream);
/* Number of ERI classes (21 for s..d). */
int pq_eri_nclass(void);
/* Per class c: stats[6c..6c+5] = nq_fp64, nq_fp32, components per quartet,
 * primitive quartets fp64, primitive quartets fp32, class code la*1000+lb*100+lc*10+ld. */
int pq_eri_stats(const pq_basis* b, long long* stats, int nstats);

/* J and K from the stored ERIs: J_ab = sum_cd Dj_cd (ab|cd),
 * K_ad = -sum_cb Dk_cb (ab|cd); Dj, Dk symmetric.  Replaces
 * make_coulomb_exchange_matrices (Methods/hartree_fock.py:329-347). */
int pq_jk(pq_basis* b, const double* Dj_dev, const double* Dk_dev, double* J_dev, double* K_dev,
          void* stream);

/* J and K for densities that need not be symmetric: J_ab = sum_cd Dj_cd
 * (ab|cd), K_ad = -sum_cb Dk_cb (ab|cd) as the reference's einsums compute
 * them for any matrix (Methods/hartree_fock.py:345-347), which NOCI calls
 * with non-symmetric co-densities (Methods/noci.py:247,275,291).  Two
 * digestions of the stored integrals (Dk and Dk^T); scratch of four packed
 * matrices from the library's device cache. */
int pq_jk_general(pq_basis* b, const double* Dj_dev, const double* Dk_dev, double* J_dev, double* K_dev,
                  void* stream);

/* pq_jk_general that allocates nothing, for callers that cannot allocate
 * device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  No counterpart in the reference.  The
 * scratch (symmetrised Dj, Dk^T and a second J', K') is a static device array
 * of 4 * 2^19 doubles (16 MiB) that each GPU the library runs on holds until
 * the process ends: a basis whose packed matrices exceed 2^19 elements
 * (n > 724 for one molecule) is rejected with an error.  Every launch goes on
 * `stream` (no side streams, no timing events); the basis's stored integrals
 * and buffers come from pq_eri_plan as for pq_jk.  Calls that overlap on one
 * GPU share the scratch and race; each call overwrites all of it that it
 * reads. */
int pq_jk_general_noalloc(pq_basis* b, const double* Dj_dev, const double* Dk_dev, double* J_dev, double* K_dev,
                          void* stream);

/* Autotuning hooks of the J/K digestion: per class, work-item length
 * (run_len, 0 = automatic) and number of blocks (grid, 0 = one per item,
 * smaller = persistent blocks looping over items); and a single-class digest
 * of the FP64 list into unsymmetrised J', K' (nitems receives the work-item
 * count).  part: 1 = tiled digestion kernel only, 2 = ket-side J reduction
 * only (reads what part 1 stored), 3 = both. */
int pq_jk_set_params(pq_basis* b, int cls, int run_len, int grid, void* stream);
int pq_jk_class(pq_basis* b, int cls, int part, const double* Dj_dev, const double* Dk_dev, double* J_dev,
                double* K_dev, int* nitems, void* stream);
/* Number of streams (1..4, default 4) that pq_jk spreads its launches over when
 * the stored integrals exceed 400 MB (one below): the caller's stream and up to three side streams forked from it and
 * joined back to it (no reference counterpart: the reference digests one
 * quartet at a time on the host). */
int pq_jk_set_streams(pq_basis* b, int nstreams);

/* pq_jk captured once into a HIP graph for fixed device buffers (kernel
 * nodes only), and replayed on `stream`: the per-iteration Fock build of
 * batched SCF without per-kernel launch overhead. */
int pq_jk_graph_create(pq_basis* b, const double* Dj_dev, const double* Dk_dev, double* J_dev, double* K_dev);
int pq_jk_graph_launch(pq_basis* b, void* stream);

/* Dense (ab|cd) tensor [ncart]^4 from the stored ERIs (screened entries
 * zero), the CoulombIntegrals array of Util/structures.py:506 as filled by
 * Methods/hartree_fock.py:266-325. */
int pq_eri_dense(pq_basis* b, double* out_dev, void* stream);

/* Arbitrary shell quartets (shells[4*i .. 4*i+3]) -> Cartesian normalised
 * blocks packed consecutively in out_host, each [nA][nB][nC][nD] in caller
 * order.  The batched form of integrals.two_electron
 * (Methods/integrals.py:427-555) before its spherical transform. */
int pq_eri_blocks(pq_basis* b, int n, const int* shells, double* out_host, void* stream);

/* Slab of the dense ERI tensor: out[mu][nu][lam - l0][sig] for lam in
 * [l0, l0 + lc) (zero where screened).  lc = ncart gives the full tensor. */
int pq_eri_dense_slab(pq_basis* b, int l0, int lc, double* out_dev, void* stream);

/* Batched FP64 matrix-core GEMM: C[b] = alpha op(A[b]) op(B[b]) + beta C[b],
 * op(A)(m,k) = ta ? A[k*lda+m] : A[m*lda+k], op(B)(k,n) = tb ? B[n*ldb+k] :
 * B[k*ldb+n]; batch strides sA, sB, sC in elements.  The dense products of
 * the MP2 transform (Methods/mp2.py:43-69 uses numpy dot). */
int pq_gemm_f64(int ta, int tb, int M, int N, int K, double alpha, const double* A, long long lda,
                long long sA, const double* B, long long ldb, long long sB, double beta, double* C,
                long long ldc, long long sC, int batch, void* stream);
/* pq_gemm_f64's product with split-BF16 matrix-core products: every FP64
 * operand element x is split into hi = bf16(x) and lo = bf16(fp32(x) - hi); a*b = hi*hi + hi*lo + lo*hi, accumulated in FP32,
 * written as FP64 (relative error ~1e-5 per product).  No reference
 * counterpart: the reference's MP2 transform is FP64 numpy. */
int pq_gemm_bf16x3(int ta, int tb, int M, int N, int K, double alpha, const double* A, long long lda,
                   long long sA, const double* B, long long ldb, long long sB, double beta, double* C,
                   long long ldc, long long sC, int batch, void* stream);

/* AO->MO transform (ia|jb) = sum C1_mi C1v_na C2_lj C2v_sb (mn|ls) from the
 * stored ERIs, by quarter transforms over the packed function pairs (lam sig),
 * lam >= sig, in slabs (at most max_slab_bytes of AO integrals at a time, one
 * pair at least; <= 0: slabs sized to half of the free device memory, so that
 * the stored quartets are read as few times as possible).
 * C matrices are row-major over Cartesian AOs: Co1[ncart][o1] etc.
 * ovov_dev is [o1][v1][o2][v2].  precision 0: FP64 matrix-core products;
 * 1: the pq_gemm_bf16x3 products (FP32 accumulation).  Replaces the O(N^6)
 * loops of Methods/mp2.py:37-69 (one call per spin pair: aa, bb, ab). */
int pq_mp2_ovov(pq_basis* b, int o1, int v1, const double* Co1, const double* Cv1, int o2, int v2,
                const double* Co2, const double* Cv2, double* ovov_dev, long long max_slab_bytes,
                int precision, void* stream);

/* Density projector of the device SCF loop: P = projector onto the nocc
 * lowest eigenvectors of the symmetric m x m matrix F (orthonormal basis),
 * by trace-correcting purification (X <- X^2 or 2X - X^2 from the Gershgorin-
 * scaled, symmetrised F; one fused product/trace/branch launch per step).
 * Replaces the per-cycle diagonalisation and occupation of
 * Methods/hartree_fock.py:168-184 (same density; orbitals are diagonalised
 * once at convergence).  work: 4 ld^2 + 2 max_steps + 3 doubles, ld = m
 * rounded up to a multiple of 32, 32-byte aligned.  0 < nocc < m,
 * max_steps >= 1.  Stops once tr(X - X^2) < tol (one more step) or after
 * max_steps; steps_out / idem_out (host, may be NULL) report the steps taken
 * and tr(X - X^2) of the converged input. */
int pq_purify(const double* F_dev, int m, int nocc, double* P_dev, double* work_dev, double tol, int max_steps,
              int* steps_out, double* idem_out, void* stream);

/* Scalars of one device SCF cycle (no reference counterpart: the
 * reference forms them on the host, the energy in Methods/hartree_fock.py:
 * 188-201 and the DIIS overlaps in Methods/hf_extensions/diis.py:62-75):
 * out_host[i] = sum_e x[i][e] y[i][e] for i < npair (<= 24), then max and
 * max-abs of each of the nr (<= 2) arrays r[j], all over n elements; two
 * launches, one copy back.  work: pq_scf_dots_work(n, npair + 2 nr)
 * doubles.  Pointer arrays are host arrays of device pointers. */
long long pq_scf_dots_work(long long n, int nout);
int pq_scf_dots(const double* const* x_dev, const double* const* y_dev, int npair, const double* const* r_dev,
                int nr, long long n, double* work_dev, double* out_host, void* stream);
/* out = sum_i c[i] m[i] over n elements, k <= 16 (the DIIS extrapolation of
 * Methods/hf_extensions/diis.py:108-118 in one launch). */
int pq_lincomb(const double* const* m_dev, const double* c_host, int k, long long n, double* out_dev, void* stream);

/* The whole SCF iteration in one call: the loop of Methods/hartree_fock.py:
 * 79-140 (J/K from pq_jk, Fock matrices, Pulay DIIS as in
 * Methods/hf_extensions/diis.py:14-155, new densities) with the densities
 * from pq_purify and the convergence test on the variational energy
 * E[D] = sum D (H + F[D]) / 2 of each cycle's input density: stop when
 * |E - E_prev| <= conv and max |X^T (S D F - F D S) X| <= sqrt(conv).
 * n = final basis size, X = n x nx orthogonaliser (X^T S X = 1); T = the
 * n x ncart Cartesian-to-final transform, or NULL when ncart == n.  H, S, X,
 * T, Da, Db, Fa, Fb are device matrices (row-major).  Da (and Db when
 * unrestricted) hold the guess on entry and the last input density on
 * exit (after maxiter cycles: the last new density); Fa (Fb) its own Fock
 * matrix (after maxiter cycles: the last extrapolated one).  Restricted:
 * nalpha == nbeta, J from 2 Da, Db / Fb may be NULL or receive copies.
 * DIIS: a residual enters while |max r| < diis_threshold and max |r| >=
 * 1e-14, from cycle diis_start + 1 when use_diis; the oldest vectors are
 * dropped while more than diis_size (restricted <= 15, unrestricted <= 9)
 * are kept or the bordered matrix's condition number exceeds
 * diis_max_cond.  work: pq_scf_work(...) doubles, 256-byte aligned.
 * energies (host, maxiter) receive each cycle's electronic energy, jk_ms
 * (host, 2 maxiter, may be NULL; needs pq_set_timing) each J/K's time;
 * result (host) = [E, dE, cycles (maxiter + 1 when not converged),
 * purification steps].  One host copy of the cycle's scalars and the
 * purification's own step read per cycle.  Returns -2 when a purification
 * does not become idempotent within 200 steps (occupied and virtual levels
 * degenerate at the Fermi level, where the reference's diagonalisation picks
 * an aufbau set): the caller then diagonalises instead. */
long long pq_scf_work(int n, int nx, int ncart, int unrestricted, int diis_size);
int pq_scf_run(pq_basis* b, const double* H_dev, const double* S_dev, const double* X_dev, int n, int nx,
               const double* T_dev, int ncart, int nalpha, int nbeta, int unrestricted, double conv, int maxiter,
               int use_diis, int diis_start, double diis_threshold, double diis_max_cond, int diis_size,
               double* Da_dev, double* Db_dev, double* Fa_dev, double* Fb_dev, double* work_dev, double* energies_host,
               double* jk_ms_host, double* result_host, void* stream);

/* Observer of pq_scf_run's late cycles (no reference counterpart: the
 * reference diagonalises every cycle, Methods/hartree_fock.py:168-177).  For
 * the pq_scf_run calls made afterwards on the calling thread: in a cycle
 * whose energy change |dE| <= threshold, each spin's purification input
 * (the DIIS-extrapolated X^T F X, nx x nx, row-major) is copied into host_a
 * (alpha) / host_b (beta) and fn(user, cycle, spin, dE) is called once the
 * copy is complete; fn returns nonzero to see that spin again in later
 * cycles, 0 to stop.  The caller may start a host diagonalisation of the
 * copy (overlapping the remaining cycles) and refine it to the final Fock
 * matrix.  fn = NULL removes the observer. */
typedef int (*pq_scf_observer_fn)(void* user, int cycle, int spin, double dE);
int pq_scf_set_observer(pq_scf_observer_fn fn, void* user, double threshold, double* host_a, double* host_b);

/* Refinement of approximate eigenvectors (no reference counterpart: the
 * reference diagonalises the Fock matrix with numpy, Methods/hartree_fock.py:
 * 168-177; this replaces that diagonalisation when an approximate
 * eigenbasis of a nearby matrix is at hand, e.g. from pq_scf_set_observer).
 * A (n x n symmetric) and U (n x n, eigenvectors as columns, row-major) are
 * device matrices; U is refined in place by the iteration of Ogita and
 * Aishima (Japan J. Indust. Appl. Math. 35 (2018) 1007-1035) until the
 * largest correction of a separated pair is <= tol or max_iter iterations;
 * pairs still unseparated (splittings below their coupling, degenerate
 * levels) are then joined into clusters whose blocks are diagonalised on
 * the host, and the iteration resumes (three rounds at most); a final step
 * orthonormalises.  lam (device, n) receives the Rayleigh quotients
 * (unsorted, in U's column order).  work: pq_eigh_refine_work(n) doubles,
 * 256-byte aligned.  info (host, 5) = [iterations, last largest correction,
 * pairs not separated (both triangles), max |A U - U diag(lam)|,
 * max |U^T U - I|]: the caller accepts the result from the last two. */
long long pq_eigh_refine_work(int n);
int pq_eigh_refine(const double* A_dev, double* U_dev, int n, int max_iter, double tol, double* lam_dev,
                   double* work_dev, double* info_host, void* stream);

/* Eigenvalues (ascending) and eigenvectors (columns) of `batch` symmetric
 * n x n matrices, A [batch][n][n] row-major on the device, into w
 * [batch][n] and V [batch][n][n]; n <= 90 (each matrix and its rotations are
 * held in LDS by one workgroup, cyclic Jacobi).  Replaces the reference's
 * per-molecule numpy.linalg.eigh of the overlap matrix
 * (Methods/hartree_fock.py:226) for the batched SCF. */
int pq_eigh_batched(const double* A_dev, int batch, int n, double* w_dev, double* V_dev, void* stream);

/* Density projectors of `batch` small symmetric matrices M [batch][m][m]
 * (device, row-major; m <= 90) onto their nocc[b] lowest states (nocc a
 * device int array), by trace-correcting purification with one workgroup
 * per matrix held in LDS: Gershgorin start, X <- X^2 or 2X - X^2 toward
 * nocc, one more step once tr(X - X^2) < tol, at most max_steps steps.
 * P [batch][m][m] receives (X + X^T) / 2, steps [batch] (device) the steps
 * taken (max_steps + 1 when the tolerance was not met).  The batched SCF's
 * replacement of the reference's per-molecule diagonalisation and density
 * (Methods/hartree_fock.py:168-184). */
int pq_purify_batched(const double* M_dev, const int* nocc_dev, int batch, int m, double tol, int max_steps,
                      double* P_dev, int* steps_dev, void* stream);

/* The batched SCF between its matrix products, one workgroup per molecule.
 * Matrices [batch][m][m] (m <= 30000), molecule b's in the leading n[b] x
 * n[b] corner; packed arrays hold the n[b] x n[b] blocks from element base[b]
 * on (base, n: device arrays of batch).  All pointers are device pointers.
 * pack: D <- Dn where !done (Dn NULL: unchanged), Dj = 2 D and Dk = D packed.
 * fock: F = H + J + K, J and K packed.
 * test: E[b] = sum D (H + F) + enuc[b] and iters[b] = it of the molecules not
 *   done; done[b] (and newly[b] = 1) once, for it > 1, E moved by less than
 *   conv and max |R| <= rtol.  flags: [0] set when any is newly done, [1]
 *   counts those not done (both zeroed by the caller).
 * diis: ring slot `newest` of Fbuf, Rbuf [batch][slots][m][m] takes F and R,
 *   G [batch][slots][slots] their products with the last k slots, and Fx is
 *   Pulay's combination of the last k Fock matrices (F itself for k = 1).
 *   flags[2] counts singular systems.  work: pq_batch_diis_work doubles.
 * lift: M += diag(dropped t), t one above the Gershgorin bound of M (at least
 *   1), dropped [batch][m]. */
int pq_batch_pack(int batch, int m, const long long* base, const long long* n, double* D, const double* Dn,
                  const unsigned char* done, double* Dj, double* Dk, void* stream);
int pq_batch_fock(int batch, int m, const long long* base, const long long* n, const double* H, const double* J,
                  const double* K, double* F, void* stream);
int pq_batch_test(int batch, int m, const long long* n, const double* D, const double* H, const double* F,
                  const double* R, const double* enuc, double conv, double rtol, int it, double* E, long long* iters,
                  unsigned char* done, unsigned char* newly, int* flags, void* stream);
long long pq_batch_diis_work(int batch, int k);
int pq_batch_diis(int batch, int m, const double* F, const double* R, double* Fbuf, double* Rbuf, double* G, int slots,
                  int newest, int k, double* Fx, double* work, int* flags, void* stream);
int pq_batch_lift(int batch, int m, double* M, const double* dropped, void* stream);

/* MP2 energy sum over ovov [o1][v1][o2][v2] with D = e_i + e_j - e_a - e_b:
 * mode 0 closed shell sum v(2v - (ib|ja))/D; mode 1 same spin
 * 1/4 sum ((ia|jb) - (ib|ja))^2 / D; mode 2 opposite spin sum v^2 / D
 * (Methods/mp2.py:77-94).  Orbital energies are device arrays. */
int pq_mp2_energy(const double* ovov_dev, const double* eo1, const double* ev1, const double* eo2,
                  const double* ev2, int o1, int v1, int o2, int v2, int mode, double* out_host, void* stream);

/* Learned SCF guess: kernels of a small FP32 multilayer perceptron (no
 * reference counterpart: the reference has only the core guess,
 * Methods/hartree_fock.py:55-57).  X [B x I], W [I x O], b [O], Z/A [B x O];
 * act 0 = identity, 1 = tanh.
 * fwd: Z = X W + b, A = act(Z) (A may be NULL).
 * bwd: dZ = dA act'(Z) (A = act(Z)), dX = dZ W^T (dX may be NULL),
 *      dW = X^T dZ, db = column sums of dZ.
 * mse: loss += sum mask (Y-T)^2 * inv_norm (device scalar), dY = 2 mask (Y-T) inv_norm.
 * adam: one bias-corrected Adam step at step number `step` (>= 1). */
int pq_mlp_linear_fwd(const float* X, const float* W, const float* b, float* Z, float* A, int B, int I, int O,
                      int act, void* stream);
int pq_mlp_linear_bwd(const float* X, const float* W, const float* A, const float* dA, float* dZ, float* dX,
                      float* dW, float* db, int B, int I, int O, int act, void* stream);
int pq_mlp_mse(const float* Y, const float* T, const float* mask, float* dY, float* loss_dev, long long n,
               float inv_norm, void* stream);
int pq_mlp_adam(float* p, const float* g, float* m, float* v, long long n, float lr, float b1, float b2, float eps,
                int step, void* stream);
/* A whole network in one launch (gradients in two): nlayer (<= 8) layers of
 * widths dims[nlayer + 1], hidden layers tanh, the last layer linear; the
 * arrays are host arrays of device pointers, one per layer.
 * forward: A[l] [B x dims[l+1]] receives layer l's output; NULL for a hidden
 * layer that is not wanted (all are needed when a width exceeds 448).
 * backward: A[l] the hidden layers' outputs, dY the gradient of the last
 * layer's output; dZ[l] [B x dims[l+1]] scratch of the hidden layers; dW, db
 * receive the gradients.
 * adam_multi: pq_mlp_adam over nt (<= 16) tensors of n[t] elements. */
int pq_mlp_forward(int nlayer, const int* dims, const float* X, const float* const* W, const float* const* b,
                   float* const* A, int B, void* stream);
int pq_mlp_backward(int nlayer, const int* dims, const float* X, const float* const* A, const float* const* W,
                    const float* dY, float* const* dZ, float* const* dW, float* const* db, int B, void* stream);
int pq_mlp_adam_multi(int nt, float* const* p, const float* const* g, float* const* m, float* const* v,
                      const long long* n, float lr, float b1, float b2, float eps, int step, void* stream);

#ifdef __cplusplus
}
#endif
#endif
