"""Batched RHF for many small molecules of uneven size on one GPU.

All molecules share one engine handle (pq_basis_create_batch): one Schwarz
pass, one ERI pass (21 class launches for the whole batch) and, per SCF
iteration, one J/K digestion replayed from a captured HIP graph.  The host
side works on padded per-molecule tensors [B, nmax, nmax] on the GPU: Fock
assembly, Pulay DIIS (last 8 residuals), batched eigh, densities and energies
for every molecule at once; converged molecules are frozen.

The reference runs one molecule per process and has no batched path; the
per-molecule algorithm is the same RHF as hartree_fock.py (closed shells,
Cartesian basis functions only: a molecule with spherical d shells is
rejected).
"""
import ctypes
import time

import numpy as np
import torch

from . import _lib, structures
from ._lib import check, dptr, iptr
from .engine import EIGH_BATCHED_MAXN, _ptr, _stream, eigh_batched


class BatchEngine:
    """One device handle over many molecules (packed per-molecule matrices)."""

    def __init__(self, mols, device="cuda"):
        if not torch.cuda.is_available():
            raise _lib.HipError("no GPU visible: the HIP engine has no CPU fallback")
        self.mols = mols
        self.device = torch.device(device)
        tabs = [m.shell_layout() for m in mols]
        for m, t in zip(mols, tabs):
            if int(m.NOrbitals) != t["ncart_total"]:
                raise ValueError("batched path expects Cartesian-basis molecules (cartesian_l covering d)")
        l = np.concatenate([t["l"] for t in tabs]).astype(np.int32)
        nprim = np.concatenate([t["nprim"] for t in tabs]).astype(np.int32)
        prim_off = np.zeros(len(l), dtype=np.int32)
        prim_off[1:] = np.cumsum(nprim)[:-1]
        exps = np.concatenate([t["exps"] for t in tabs]).astype(float)
        cc = np.concatenate([t["cc"] for t in tabs]).astype(float)
        shell_mol = np.repeat(np.arange(len(tabs), dtype=np.int32), [t["nshell"] for t in tabs])
        xyz = np.array([a.Coordinates for m in mols for a in m.Atoms], dtype=float).reshape(-1, 3)
        center = np.repeat(xyz, np.concatenate([t["per_atom"] for t in tabs]), axis=0).reshape(-1)
        axyz = xyz.reshape(-1)
        az = np.array([a.NuclearCharge for m in mols for a in m.Atoms], dtype=float)
        amol = np.repeat(np.arange(len(tabs), dtype=np.int32), [m.NAtom for m in mols])
        self._keep = (l, nprim, prim_off, center, exps, cc, shell_mol, axyz, az, amol)
        h = ctypes.c_void_p()
        L = _lib.lib()
        check(L.pq_basis_create_batch(len(mols), len(l), iptr(l), iptr(nprim), iptr(prim_off), dptr(center),
                                      dptr(exps), dptr(cc), iptr(shell_mol), len(az), dptr(axyz), dptr(az),
                                      iptr(amol), ctypes.byref(h)), "pq_basis_create_batch")
        self.h = h
        info = np.zeros(7, dtype=np.int64)
        check(L.pq_basis_info(h, info.ctypes.data_as(_lib.P_ll)), "pq_basis_info")
        self.nmol, self.mat_total, self.nmax = int(info[4]), int(info[5]), int(info[6])
        self.base = np.zeros(self.nmol, dtype=np.int64)
        self.n = np.zeros(self.nmol, dtype=np.int32)
        check(L.pq_basis_molecules(h, self.base.ctypes.data_as(_lib.P_ll), iptr(self.n), None, None),
              "pq_basis_molecules")
        # packed position -> padded flat position [B, nmax, nmax]: the packed
        # matrices are the molecules' n x n blocks back to back (built on the
        # device: the index array is several MB for a large batch)
        nm = self.nmax
        total = int((self.n.astype(np.int64) ** 2).sum())
        nn = torch.as_tensor(self.n.astype(np.int64), device=self.device)
        sizes = nn * nn
        rep = dict(output_size=total)
        mol = torch.repeat_interleave(torch.arange(self.nmol, device=self.device), sizes, **rep)
        k = torch.arange(total, device=self.device) - torch.repeat_interleave(torch.cumsum(sizes, 0) - sizes, sizes, **rep)
        nrow = torch.repeat_interleave(nn, sizes, **rep)
        self.pidx = mol * nm * nm + torch.div(k, nrow, rounding_mode="floor") * nm + k % nrow
        self.n_dev = nn
        self.base_dev = torch.cumsum(sizes, 0) - sizes
        self.graph = False

    def close(self):
        if getattr(self, "h", None):
            _lib.lib().pq_basis_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def to_padded(self, packed):
        out = torch.zeros(self.nmol * self.nmax * self.nmax, dtype=packed.dtype, device=self.device)
        out[self.pidx] = packed
        return out.view(self.nmol, self.nmax, self.nmax)

    def to_packed(self, padded, out=None):
        flat = padded.reshape(-1)[self.pidx]
        if out is None:
            return flat
        out.copy_(flat)
        return out

    def one_electron(self):
        S = torch.empty(self.mat_total, dtype=torch.float64, device=self.device)
        T = torch.empty_like(S)
        V = torch.empty_like(S)
        check(_lib.lib().pq_one_electron(self.h, _ptr(S), _ptr(T), _ptr(V), _stream()), "pq_one_electron")
        return S, T, V

    def build_eri(self, threshold=1e-8, fp32_threshold=0.0):
        check(_lib.lib().pq_eri_build(self.h, float(threshold), float(fp32_threshold), _stream()), "pq_eri_build")

    def stats(self):
        nc = _lib.lib().pq_eri_nclass()
        st = np.zeros(nc * 6, dtype=np.int64)
        check(_lib.lib().pq_eri_stats(self.h, st.ctypes.data_as(_lib.P_ll), nc * 6), "pq_eri_stats")
        return st.reshape(nc, 6)

    def jk_buffers(self):
        """Fixed device buffers used by the captured J/K graph."""
        self.Dj = torch.zeros(self.mat_total, dtype=torch.float64, device=self.device)
        self.Dk = torch.zeros_like(self.Dj)
        self.J = torch.zeros_like(self.Dj)
        self.K = torch.zeros_like(self.Dj)
        torch.cuda.synchronize()
        check(_lib.lib().pq_jk_graph_create(self.h, _ptr(self.Dj), _ptr(self.Dk), _ptr(self.J), _ptr(self.K)),
              "pq_jk_graph_create")
        self.graph = True

    def jk_replay(self):
        check(_lib.lib().pq_jk_graph_launch(self.h, _stream()), "pq_jk_graph_launch")

    # the SCF's steps between its matrix products, one launch each, on padded
    # matrices [nmol, nmax, nmax] (scf_batch.hip)
    def _call(self, name, *args):
        check(getattr(_lib.lib(), name)(self.nmol, self.nmax, *args, _stream()), name)

    def pack(self, D, Dn=None, done=None):
        """D <- Dn where not done; the J/K inputs Dj = 2 D and Dk = D."""
        self._call("pq_batch_pack", _ptr(self.base_dev), _ptr(self.n_dev), _ptr(D),
                   None if Dn is None else _ptr(Dn), None if done is None else _ptr(done), _ptr(self.Dj), _ptr(self.Dk))

    def fock(self, H):
        """H + J + K of the last J/K build."""
        F = torch.empty_like(H)
        self._call("pq_batch_fock", _ptr(self.base_dev), _ptr(self.n_dev), _ptr(H), _ptr(self.J), _ptr(self.K), _ptr(F))
        return F

    def jk_direct(self):
        check(_lib.lib().pq_jk(self.h, _ptr(self.Dj), _ptr(self.Dk), _ptr(self.J), _ptr(self.K), _stream()), "pq_jk")


def _sad_packed(eng, mols):
    """SAD densities, packed (host): a quarter of the padded matrices' bytes
    for 512 molecules of 7 to 61 functions."""
    from .guess import sad_density
    D = np.empty(eng.mat_total)
    layouts = {}   # one SAD matrix per layout (basis, atom labels, Cartesian shells) of this batch
    for m, mol in enumerate(mols):
        key = (mol.Basis, tuple(a.Label for a in mol.Atoms), tuple(mol.CartesianL))
        d = layouts.get(key)
        if d is None:
            d = layouts[key] = np.asarray(sad_density(mol), dtype=float).reshape(-1)
        D[eng.base[m]:eng.base[m] + d.size] = d
    return D


def rhf_batch(mols, conv=1e-8, maxiter=60, threshold=1e-8, guess="SAD", use_graph=True, diis_size=8,
              tune=None, return_density=False):
    """Closed-shell RHF for every molecule in ``mols`` at once.

    Returns dict: energies [B], iterations [B], converged [B], per-molecule
    latency (seconds from start until its convergence), stage timings."""
    t_start = time.perf_counter()
    for m in mols:
        if m.NAlphaElectrons != m.NBetaElectrons:
            raise ValueError("rhf_batch handles closed-shell molecules")
    eng = BatchEngine(mols)
    dev = eng.device
    B, nm = eng.nmol, eng.nmax
    S, T, V = eng.one_electron()
    eng.build_eri(threshold)
    Sp = eng.to_padded(S)
    Hp = eng.to_padded(T + V)
    n_t = eng.n_dev   # on the device since the handle's creation: no copy queued behind the ERI pass
    ar = torch.arange(nm, device=dev)
    valid = (ar[None, :] < n_t[:, None])                                 # [B, nm]
    vmask = (valid[:, :, None] & valid[:, None, :]).to(torch.float64)
    # canonical orthogonaliser per molecule; the pad block of S is 1e3 * I so
    # its eigenvalues separate from the molecular ones and are dropped
    pad_eye = 1e3 * torch.diag_embed((~valid).to(torch.float64))
    if nm <= EIGH_BATCHED_MAXN:
        s, U = eigh_batched(Sp + pad_eye)
    else:
        s, U = torch.linalg.eigh(Sp + pad_eye)
    keep = (s > structures.LINEAR_DEPENDENCE) & (s < 5e2)               # [B, nm] kept columns
    X = U * torch.where(keep, s.clamp_min(1e-300) ** -0.5, torch.zeros_like(s))[:, None, :]
    X = X * valid[:, :, None]
    dropped = (~keep).to(torch.float64)                                  # [B, nm] dropped / pad columns
    # host inputs, prepared while the ERI pass and the eigensolver run; the
    # copies to the device then wait for that work
    nocc_h = np.array([m.NAlphaElectrons for m in mols])
    enuc_h = _nuclear_batch(eng)
    D_h = _sad_packed(eng, mols) if guess == "SAD" else None
    nocc = torch.as_tensor(nocc_h, device=dev).to(torch.int32)
    enuc = torch.as_tensor(enuc_h, dtype=torch.float64, device=dev)
    if guess == "SAD":
        D = 0.5 * eng.to_padded(torch.as_tensor(D_h).to(dev))
    else:
        D = _density(X, Hp, dropped, nocc)
    if tune is not None:
        from . import autotune
        eng.Dj = eng.to_packed(2.0 * D).contiguous()
        eng.Dk = eng.to_packed(D).contiguous()
        eng.J = torch.zeros_like(eng.Dj)
        eng.K = torch.zeros_like(eng.Dj)
        if tune == "search":
            eng.tuned = autotune.tune_jk(eng, eng.Dj, eng.Dk, eng.J, eng.K)
        else:
            autotune.apply(eng, tune)
            eng.tuned = tune
    if use_graph:
        eng.jk_buffers()
    else:
        eng.Dj = torch.zeros(eng.mat_total, dtype=torch.float64, device=dev)
        eng.Dk = torch.zeros_like(eng.Dj)
        eng.J = torch.zeros_like(eng.Dj)
        eng.K = torch.zeros_like(eng.Dj)
    torch.cuda.synchronize()
    t_setup = time.perf_counter() - t_start
    E = torch.zeros(B, dtype=torch.float64, device=dev)
    done = torch.zeros(B, dtype=torch.bool, device=dev)
    newly = torch.zeros_like(done)
    iters = torch.zeros(B, dtype=torch.long, device=dev)
    latency = np.full(B, np.nan)
    # DIIS history in a ring of slots: the stored Fock matrices and residuals
    # and their Gram matrix, the last k slots active
    S_ = diis_size + 1
    Fbuf = torch.zeros((B, S_, nm, nm), dtype=torch.float64, device=dev)
    Rbuf = torch.zeros_like(Fbuf)
    G = torch.zeros((B, S_, S_), dtype=torch.float64, device=dev)
    work = None
    # per cycle: any newly converged, molecules not converged, singular systems
    flags = torch.zeros((max(maxiter, 0) + 1, 3), dtype=torch.int32, device=dev)
    D, Hp, Dn = D.contiguous(), Hp.contiguous(), None
    for it in range(1, maxiter + 1):
        eng.pack(D, Dn, done)
        Dn = None
        if use_graph:
            eng.jk_replay()
        else:
            eng.jk_direct()
        F = eng.fock(Hp)
        # Pulay DIIS on X^T (S D F - F D S) X, batched
        A = Sp @ D @ F
        R = X.transpose(1, 2) @ (A - A.transpose(1, 2)) @ X
        # variational energy of this cycle's input density with its own Fock
        # matrix (the single-molecule device loop's test): |dE| < conv counts
        # once the orbital gradient has settled too, and the molecule keeps
        # the density whose energy passed
        eng._call("pq_batch_test", _ptr(eng.n_dev), _ptr(D), _ptr(Hp), _ptr(F), _ptr(R), _ptr(enuc), float(conv),
                  float(conv) ** 0.5, it, _ptr(E), _ptr(iters), _ptr(done), _ptr(newly), _ptr(flags[it]))
        # one host wait per iteration (the singular systems are the last cycle's)
        (_, _, singular), (any_new, not_done, _) = flags[it - 1:it + 1].tolist()
        if singular:
            raise torch.linalg.LinAlgError("rhf_batch: singular DIIS system")
        if any_new:
            tnow = time.perf_counter() - t_start
            for m in torch.nonzero(newly).flatten().tolist():
                latency[m] = tnow
        if not not_done:
            break
        k = max(1, min(it, diis_size))
        if work is None or k > 64:
            work = torch.empty(max(1, _lib.lib().pq_batch_diis_work(B, k)), dtype=torch.float64, device=dev)
        Fx = torch.empty_like(F)
        eng._call("pq_batch_diis", _ptr(F), _ptr(R), _ptr(Fbuf), _ptr(Rbuf), _ptr(G), S_, (it - 1) % S_, k, _ptr(Fx),
                  _ptr(work), _ptr(flags[it]))
        Dn = _density(X, Fx, dropped, nocc).contiguous()
    if Dn is not None:   # not every molecule converged
        if flags[it, 2].item():
            raise torch.linalg.LinAlgError("rhf_batch: singular DIIS system")
        D = torch.where(done[:, None, None], D, Dn)
    torch.cuda.synchronize()
    total = time.perf_counter() - t_start
    latency[np.isnan(latency)] = total
    out = dict(energies=E.cpu().numpy(), iterations=iters.cpu().numpy(), converged=done.cpu().numpy(),
               latency_s=latency, total_s=total, setup_s=t_setup, nmol=B, stats=eng.stats(),
               tuned=getattr(eng, "tuned", None))
    if return_density:
        Dh = eng.to_packed(D).cpu().numpy()
        out["densities"] = [Dh[eng.base[m]:eng.base[m] + int(eng.n[m]) ** 2].reshape(eng.n[m], eng.n[m]).copy()
                            for m in range(B)]
    eng.close()
    return out


def _density(X, F, dropped, nocc):
    """D = X P X^T with P the projector onto the nocc lowest states of
    X^T F X, by batched trace-correcting purification.  Dropped and pad
    columns (zero rows of X^T F X) are lifted above every molecule's spectrum
    so that they stay empty."""
    from .engine import EIGH_BATCHED_MAXN, purify_batched as purify_lib
    from .hartree_fock import purify_batched
    M = (X.transpose(1, 2) @ F @ X).contiguous()
    check(_lib.lib().pq_batch_lift(M.shape[0], M.shape[1], _ptr(M), _ptr(dropped), _stream()), "pq_batch_lift")
    if M.shape[1] <= EIGH_BATCHED_MAXN:
        P, _ = purify_lib(M, nocc)
    else:
        P = purify_batched(M.contiguous(), nocc)
    return X @ P @ X.transpose(1, 2)


def _nuclear_batch(eng):
    """sum_{i>j} Z_i Z_j / r_ij per molecule (Methods/integrals.py:196-207)
    for every molecule of the handle at once, from its packed atom arrays
    (atoms grouped by molecule), over a [molecule, atom, atom] padding."""
    axyz, az, amol = eng._keep[7].reshape(-1, 3), eng._keep[8], eng._keep[9]
    B = eng.nmol
    counts = np.bincount(amol, minlength=B)
    start = np.zeros(B, dtype=np.int64)
    start[1:] = np.cumsum(counts)[:-1]
    A = int(counts.max()) if len(counts) else 0
    R = np.zeros((B, A, 3))
    Z = np.zeros((B, A))
    slot = np.arange(len(amol)) - start[amol]
    R[amol, slot] = axyz
    Z[amol, slot] = az
    d = np.sqrt(((R[:, :, None, :] - R[:, None, :, :]) ** 2).sum(-1))
    i, j = np.tril_indices(A, -1)
    zz = Z[:, i] * Z[:, j]
    r = d[:, i, j]
    return np.where(zz != 0.0, zz / np.where(r > 0.0, r, 1.0), 0.0).sum(1)


def structures_nuclear(mol):
    from .hartree_fock import nuclear_repulsion
    return nuclear_repulsion(mol)


def config4_molecules(count=512, seed=4, sigma=0.05):
    """512 molecules drawn by numpy.random.default_rng(seed) from
    {H2O, NH3, CH4, C2H6, CH3OH, C3H8} x {STO-3G, 6-31G*}, coordinate jitter
    sigma (Angstrom); 6-31G* with Cartesian d."""
    from . import geometry
    rng = np.random.default_rng(seed)
    names = ["H2O", "NH3", "CH4", "C2H6", "CH3OH", "C3H8"]
    bases = ["STO-3G", "6-31G*"]
    mols = []
    for k in range(count):
        name = names[int(rng.integers(len(names)))]
        basis = bases[int(rng.integers(len(bases)))]
        rows = geometry.small_molecule(name, sigma, int(rng.integers(1 << 30)))
        mols.append(structures.Molecule(rows, basis=basis, cartesian_l=[2]))
    return mols
