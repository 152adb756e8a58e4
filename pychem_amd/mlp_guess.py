"""Learned SCF initial guess: an MLP maps local-geometry descriptors of an
atom pair to that pair's block of the alpha density matrix.

No reference counterpart: the reference starts from the core Hamiltonian
(Methods/hartree_fock.py:55-57).  The network is trained and evaluated with
the library's own FP32 kernels (pq_mlp_forward / _backward, pq_mlp_mse,
pq_mlp_adam_multi); torch only provides device buffers.

Density blocks are not rotation invariant, so each block is learned in a
local frame of its atom pair and rotated back:

* frame of an off-diagonal pair (A, B): e1 along B - A, e2 towards the atom
  nearest to A (other than A, B) orthogonalised against e1, e3 = e1 x e2;
  of a diagonal block (A, A): e1 towards the nearest neighbour, e2 towards
  the second nearest.
* a rotation R (rows e1, e2, e3) acts on the normalised Cartesian functions
  of a shell through M(R) (monomials of R v expanded in monomials of v,
  scaled by the per-component normalisation), and the density block in the
  local frame is D' = M_A^-T D M_B^-1, i.e. D = M_A^T D' M_B.
* descriptors (invariant): pair distance, 16 radial Gaussian features
  (centres 0.5..4 A, Z-weighted, cutoff 4 A) for each of the two atoms, and
  the local coordinates of the frame-defining neighbours.
* one network per (element A, element B, diagonal) type: 3 hidden layers of
  128 tanh units and a linear output of n_A * n_B values, inputs and outputs
  standardised.
"""
import ctypes
import itertools
import math
import os
import time

import numpy as np
import torch

from . import _lib, structures
from ._lib import check

ANG = 1.0 / structures.TO_BOHR
RCUT_PAIR = 6.0          # Angstrom: pairs beyond this start from a zero block
RCUT_ENV = 4.0
MU = np.linspace(0.5, 4.0, 16)
ETA = 1.0 / (2 * 0.25 ** 2)
NFEAT = 1 + 16 + 16 + 4
HIDDEN = 128


# ----------------------------------------------------------------- geometry
def _monomial_expansion(l, R):
    """P[c][c'] with prod_i (sum_j R_ij v_j)^{c_i} = sum_c' P[c][c'] v^{c'}."""
    comps = structures.cart_components(l)
    index = {c: k for k, c in enumerate(comps)}
    P = np.zeros((len(comps), len(comps)))
    for a, c in enumerate(comps):
        # product over axes i of (R_i . v)^{c_i}: expand as a polynomial dict
        poly = {(0, 0, 0): 1.0}
        for i in range(3):
            for _ in range(c[i]):
                new = {}
                for mono, coef in poly.items():
                    for j in range(3):
                        m2 = list(mono)
                        m2[j] += 1
                        m2 = tuple(m2)
                        new[m2] = new.get(m2, 0.0) + coef * R[i, j]
                poly = new
        for mono, coef in poly.items():
            P[a, index[mono]] += coef
    return P


def cart_rotation(l, R):
    """M(R) acting on the normalised Cartesian functions of one shell."""
    if l == 0:
        return np.ones((1, 1))
    comps = structures.cart_components(l)
    N = np.array([(math.gamma(a + 0.5) * math.gamma(b + 0.5) * math.gamma(c + 0.5)) ** -0.5 for a, b, c in comps])
    P = _monomial_expansion(l, R)
    return (N[:, None] * P) / N[None, :]


def atom_rotation(ls, R):
    """Block-diagonal M(R) over an atom's shells (list of l)."""
    blocks = [cart_rotation(l, R) for l in ls]
    n = sum(b.shape[0] for b in blocks)
    M = np.zeros((n, n))
    o = 0
    for b in blocks:
        k = b.shape[0]
        M[o:o + k, o:o + k] = b
        o += k
    return M


def _unit(v):
    return v / np.linalg.norm(v)


def _frame(xyz, a, b):
    """Rows e1, e2, e3 of the local frame, and the frame-defining atoms."""
    d = np.linalg.norm(xyz - xyz[a], axis=1)
    order = [k for k in np.argsort(d) if k != a and k != b]
    if a != b:
        e1 = _unit(xyz[b] - xyz[a])
        refs = order
    else:
        if not order:
            return np.eye(3), []
        e1 = _unit(xyz[order[0]] - xyz[a])
        refs = order[1:]
    e2 = None
    used = []
    for k in refs:
        v = xyz[k] - xyz[a]
        w = v - np.dot(v, e1) * e1
        if np.linalg.norm(w) > 1e-3:
            e2 = _unit(w)
            used.append(k)
            break
    if e2 is None:
        t = np.array([1.0, 0.0, 0.0]) if abs(e1[0]) < 0.9 else np.array([0.0, 1.0, 0.0])
        e2 = _unit(t - np.dot(t, e1) * e1)
    e3 = np.cross(e1, e2)
    if a == b:
        used = [order[0]] + used
    return np.array([e1, e2, e3]), used


def _radial(xyz, Z, a):
    d = np.linalg.norm(xyz - xyz[a], axis=1) * ANG
    m = (d > 1e-8) & (d < RCUT_ENV)
    fc = 0.5 * (np.cos(np.pi * d[m] / RCUT_ENV) + 1.0)
    return (Z[m, None] * fc[:, None] * np.exp(-ETA * (d[m, None] - MU[None, :]) ** 2)).sum(0)


def pair_samples(mol):
    """Yield (type, i, j, features, local->global rotation data) for all atom
    pairs i <= j within RCUT_PAIR (Angstrom)."""
    xyz = np.array([a.Coordinates for a in mol.Atoms])
    Z = np.array([a.NuclearCharge for a in mol.Atoms])
    rad = [_radial(xyz, Z, a) for a in range(len(Z))]
    out = []
    for i in range(len(Z)):
        for j in range(i, len(Z)):
            a, b = (i, j) if Z[i] >= Z[j] else (j, i)
            r = np.linalg.norm(xyz[b] - xyz[a]) * ANG
            if r > RCUT_PAIR:
                continue
            R, used = _frame(xyz, a, b)
            loc = [(R @ (xyz[k] - xyz[a])) * ANG for k in used[:2]]
            while len(loc) < 2:
                loc.append(np.zeros(3))
            f = np.concatenate([[r], rad[a], rad[b], [loc[0][0], loc[0][1], loc[1][0], loc[1][1]]])
            key = (mol.Atoms[a].Label, mol.Atoms[b].Label, a == b)
            out.append((key, a, b, f, R))
    return out


def _atom_functions(mol):
    """Per atom: function indices and shell l list (final = Cartesian basis)."""
    idx = [[] for _ in range(mol.NAtom)]
    ls = [[] for _ in range(mol.NAtom)]
    o = 0
    for at, atom in enumerate(mol.Atoms):
        for cg in atom.Basis:
            idx[at].extend(range(o, o + cg.NAngMom))
            ls[at].append(cg.AngularMomentum)
            o += cg.NAngMom
    return idx, ls


def local_block(D, mol, a, b, R, idx=None, ls=None):
    """D'_{ab} = M_a^-T D_ab M_b^-1 (block of D in the pair's local frame)."""
    if idx is None:
        idx, ls = _atom_functions(mol)
    Ma, Mb = atom_rotation(ls[a], R), atom_rotation(ls[b], R)
    blk = D[np.ix_(idx[a], idx[b])]
    return np.linalg.solve(Ma.T, blk) @ np.linalg.inv(Mb)


# ------------------------------------------------- vectorised pair data
def _d_tables():
    comps = structures.cart_components(2)
    ax = [[i for i in range(3) for _ in range(c[i])] for c in comps]
    I = np.array([a[0] for a in ax])
    J = np.array([a[1] for a in ax])
    index = {c: k for k, c in enumerate(comps)}
    A = np.zeros((9, 6))
    for k in range(3):
        for l in range(3):
            m = [0, 0, 0]
            m[k] += 1
            m[l] += 1
            A[k * 3 + l, index[tuple(m)]] = 1.0
    N = np.array([(math.gamma(a + 0.5) * math.gamma(b + 0.5) * math.gamma(c + 0.5)) ** -0.5 for a, b, c in comps])
    return I, J, A, N


_DTAB = _d_tables()


def rot_d_batch(R):
    """cart_rotation(2, R) for a stack R [P, 3, 3] (numpy or torch)."""
    I, J, A, N = _DTAB
    if isinstance(R, torch.Tensor):
        A_, N_ = torch.as_tensor(A, dtype=R.dtype, device=R.device), torch.as_tensor(N, dtype=R.dtype, device=R.device)
        T = R[:, I, :, None] * R[:, J, None, :]
        P = T.reshape(-1, 6, 9) @ A_
        return N_[:, None] * P / N_[None, :]
    T = R[:, I, :, None] * R[:, J, None, :]
    P = T.reshape(-1, 6, 9) @ A
    return N[:, None] * P / N[None, :]


def atom_rot_batch(ls, R):
    """atom_rotation(ls, R) for a stack R [P, 3, 3]: [P, n, n]."""
    torch_in = isinstance(R, torch.Tensor)
    n = sum((l + 1) * (l + 2) // 2 for l in ls)
    P = R.shape[0]
    if torch_in:
        M = torch.zeros((P, n, n), dtype=R.dtype, device=R.device)
    else:
        M = np.zeros((P, n, n))
    o = 0
    for l in ls:
        k = (l + 1) * (l + 2) // 2
        if l == 0:
            M[:, o, o] = 1.0
        elif l == 1:
            M[:, o:o + 3, o:o + 3] = R
        else:
            M[:, o:o + 6, o:o + 6] = rot_d_batch(R)
        o += k
    return M


def pair_data(mol):
    """All atom pairs (a, b) within RCUT_PAIR, a the heavier atom, grouped
    by type (label_a, label_b, a == b): {type: (a [P], b [P], features
    [P, NFEAT], R [P, 3, 3])}.  Same frames and features as pair_samples,
    computed over all pairs at once."""
    xyz = np.array([at.Coordinates for at in mol.Atoms], dtype=float)
    Z = np.array([at.NuclearCharge for at in mol.Atoms], dtype=float)
    labels = [at.Label for at in mol.Atoms]
    n = len(Z)
    diff = xyz[None, :, :] - xyz[:, None, :]          # [a, k, 3] = x_k - x_a
    dist = np.linalg.norm(diff, axis=2)
    dA = dist * ANG
    env = (dA > 1e-8) & (dA < RCUT_ENV)
    # radial features over the neighbours inside the cutoff only (the cutoff
    # function is zero elsewhere)
    ea, ek = np.nonzero(env)
    de = dA[ea, ek]
    we = Z[ek] * (0.5 * (np.cos(np.pi * de / RCUT_ENV) + 1.0))
    rad = np.zeros((n, len(MU)))
    if len(ea):   # np.nonzero lists ea ascending: one segment per atom
        starts = np.flatnonzero(np.r_[True, ea[1:] != ea[:-1]])
        rad[ea[starts]] = np.add.reduceat(we[:, None] * np.exp(-ETA * (de[:, None] - MU[None, :]) ** 2), starts, axis=0)
    ii, jj = np.triu_indices(n)
    keep = dA[ii, jj] <= RCUT_PAIR
    ii, jj = ii[keep], jj[keep]
    swap = Z[ii] < Z[jj]
    a = np.where(swap, jj, ii)
    b = np.where(swap, ii, jj)
    P = len(a)
    ar = np.arange(n)
    diag = a == b
    # first axis: towards b, or towards the nearest neighbour for (a, a)
    dmask = np.where(ar[None, :] == a[:, None], np.inf, dist[a])
    nn1 = np.argmin(dmask, axis=1) if n > 1 else np.zeros(P, dtype=int)
    tgt = np.where(diag, nn1, b)
    pr = np.arange(P)
    e1 = diff[a, tgt]
    has1 = np.linalg.norm(e1, axis=1) > 0
    e1 = e1 / np.where(has1, np.linalg.norm(e1, axis=1), 1.0)[:, None]
    # second axis: nearest remaining atom with a component normal to e1; the
    # normal part's length from |x_k - x_a|^2 - ((x_k - x_a).e1)^2, the
    # projections as one [P, n] product
    proj = e1 @ xyz.T - (xyz[a] * e1).sum(1)[:, None]
    wn = np.sqrt(np.maximum(dist[a] ** 2 - proj ** 2, 0.0))
    cand = (ar[None, :] != a[:, None]) & (ar[None, :] != b[:, None]) & (wn > 1e-3)
    cand &= ~(diag[:, None] & (ar[None, :] == nn1[:, None]))
    dc = np.where(cand, dist[a], np.inf)
    k2 = np.argmin(dc, axis=1)
    has2 = np.isfinite(dc[pr, k2])
    v2 = diff[a, k2]
    w2 = v2 - (v2 * e1).sum(1, keepdims=True) * e1
    e2 = w2 / np.where(has2, np.linalg.norm(w2, axis=1), 1.0)[:, None]
    t = np.where((np.abs(e1[:, 0]) < 0.9)[:, None], np.array([1.0, 0.0, 0.0]), np.array([0.0, 1.0, 0.0]))
    tf = t - (t * e1).sum(1, keepdims=True) * e1
    tf = tf / np.linalg.norm(tf, axis=1, keepdims=True)
    e2 = np.where(has2[:, None], e2, tf)
    e3 = np.cross(e1, e2)
    R = np.stack([e1, e2, e3], axis=1)
    R = np.where(has1[:, None, None], R, np.eye(3)[None])
    # local coordinates of the frame-defining atoms (nearest neighbour, then e2 atom, for (a, a))
    loc_e2 = np.einsum("pij,pj->pi", R, v2) * ANG
    loc_nn = np.einsum("pij,pj->pi", R, diff[a, nn1]) * ANG
    loc0 = np.where(diag[:, None], np.where(has1[:, None], loc_nn, 0.0), np.where(has2[:, None], loc_e2, 0.0))
    loc1 = np.where((diag & has1 & has2)[:, None], loc_e2, 0.0)
    F = np.concatenate([dA[a, b][:, None], rad[a], rad[b], loc0[:, :2], loc1[:, :2]], axis=1)
    groups = {}
    for p in range(P):
        groups.setdefault((labels[a[p]], labels[b[p]], bool(diag[p])), []).append(p)
    return {key: (a[v], b[v], F[v], R[v]) for key, v in groups.items()}


def _atom_layout(mol):
    """Per atom: first function index and its shells' l list."""
    off, ls = [], []
    o = 0
    for atom in mol.Atoms:
        off.append(o)
        ls.append([cg.AngularMomentum for cg in atom.Basis])
        o += sum(cg.NAngMom for cg in atom.Basis)
    return np.array(off), ls


# ----------------------------------------------------------------- network
def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


# widest layer of the one-launch network kernels (pq_mlp_forward)
FUSED_WIDTH = 448


def _ptrs(tensors):
    """Host array of device pointers (None: NULL)."""
    return (ctypes.c_void_p * len(tensors))(*[None if t is None else t.data_ptr() for t in tensors])


def _dims(dims):
    return (ctypes.c_int * len(dims))(*dims)


class MLP:
    """Input -> 3 x (128, tanh) -> linear output, FP32 on the GPU."""

    def __init__(self, nin, nout, seed=0, device="cuda"):
        g = np.random.default_rng(seed)
        dims = [nin, HIDDEN, HIDDEN, HIDDEN, nout]
        self.dims = dims
        self.W, self.b = [], []
        for i in range(4):
            lim = math.sqrt(6.0 / (dims[i] + dims[i + 1]))
            self.W.append(torch.tensor(g.uniform(-lim, lim, (dims[i], dims[i + 1])), dtype=torch.float32, device=device))
            self.b.append(torch.zeros(dims[i + 1], dtype=torch.float32, device=device))
        self.m = [torch.zeros_like(p) for p in self.W + self.b]
        self.v = [torch.zeros_like(p) for p in self.W + self.b]
        self.step = 0
        self.xmean = self.xstd = self.ymean = self.ystd = None

    def params(self):
        return self.W + self.b

    def forward(self, X, keep=False):
        B, last = X.shape[0], len(self.W) - 1
        wide = max(self.dims) > FUSED_WIDTH      # such layers go one launch each, through buffers of their own
        outs = [torch.empty((B, self.dims[i + 1]), dtype=torch.float32, device=X.device)
                if keep or wide or i == last else None for i in range(last + 1)]
        check(_lib.lib().pq_mlp_forward(last + 1, _dims(self.dims), _ptr(X), _ptrs(self.W), _ptrs(self.b), _ptrs(outs),
                                        B, _stream()), "pq_mlp_forward")
        return (outs[-1], [X] + outs) if keep else outs[-1]

    def backward(self, acts, dY):
        """Gradients of the parameters given dLoss/dY; returns (gW, gb)."""
        n = len(self.W)
        B = acts[0].shape[0]
        gW = [torch.empty_like(w) for w in self.W]
        gb = [torch.empty_like(b) for b in self.b]
        dZ = [torch.empty((B, self.dims[i + 1]), dtype=torch.float32, device=dY.device) for i in range(n - 1)]
        check(_lib.lib().pq_mlp_backward(n, _dims(self.dims), _ptr(acts[0]), _ptrs(acts[1:]), _ptrs(self.W), _ptr(dY),
                                         _ptrs(dZ + [None]), _ptrs(gW), _ptrs(gb), B, _stream()), "pq_mlp_backward")
        return gW, gb

    def loss_grad(self, Y, T):
        L = _lib.lib()
        dY = torch.empty_like(Y)
        loss = torch.zeros(1, dtype=torch.float32, device=Y.device)
        check(L.pq_mlp_mse(_ptr(Y), _ptr(T), None, _ptr(dY), _ptr(loss), Y.numel(), 1.0 / Y.numel(), _stream()),
              "pq_mlp_mse")
        return loss, dY

    def adam(self, gW, gb, lr=1e-3):
        L = _lib.lib()
        self.step += 1
        ps = self.params()
        sizes = (ctypes.c_longlong * len(ps))(*[p.numel() for p in ps])
        check(L.pq_mlp_adam_multi(len(ps), _ptrs(ps), _ptrs(gW + gb), _ptrs(self.m), _ptrs(self.v), sizes, lr, 0.9,
                                  0.999, 1e-8, self.step, _stream()), "pq_mlp_adam_multi")

    def state(self):
        d = {"W%d" % i: w.cpu().numpy() for i, w in enumerate(self.W)}
        d.update({"b%d" % i: b.cpu().numpy() for i, b in enumerate(self.b)})
        d.update(xmean=self.xmean, xstd=self.xstd, ymean=self.ymean, ystd=self.ystd)
        return d

    @classmethod
    def from_state(cls, d, device="cuda"):
        W0 = d["W0"]
        net = cls(W0.shape[0], d["W3"].shape[1], device=device)
        for i in range(4):
            net.W[i] = torch.tensor(d["W%d" % i], device=device)
            net.b[i] = torch.tensor(d["b%d" % i], device=device)
        net.xmean, net.xstd, net.ymean, net.ystd = d["xmean"], d["xstd"], d["ymean"], d["ystd"]
        return net


# ----------------------------------------------------------------- data
def local_blocks(D, mol, groups=None):
    """{type: (features [P, NFEAT], local blocks [P, n_a n_b])} from a density
    D (numpy, final Cartesian basis): D' = M_a(R^T)^T D_ab M_b(R^T)."""
    groups = pair_data(mol) if groups is None else groups
    off, ls = _atom_layout(mol)
    out = {}
    for key, (a, b, F, R) in groups.items():
        la, lb = ls[a[0]], ls[b[0]]
        na, nb = sum((l + 1) * (l + 2) // 2 for l in la), sum((l + 1) * (l + 2) // 2 for l in lb)
        rows = off[a][:, None] + np.arange(na)[None, :]
        cols = off[b][:, None] + np.arange(nb)[None, :]
        blk = D[rows[:, :, None], cols[:, None, :]]
        Rt = np.transpose(R, (0, 2, 1))
        loc = np.transpose(atom_rot_batch(la, Rt), (0, 2, 1)) @ blk @ atom_rot_batch(lb, Rt)
        out[key] = (F, loc.reshape(len(a), -1))
    return out


def collect(mols, densities):
    """Training samples per pair type from converged alpha densities."""
    data = {}
    for mol, D in zip(mols, densities):
        for key, (F, Y) in local_blocks(np.asarray(D), mol).items():
            data.setdefault(key, ([], []))
            data[key][0].append(F)
            data[key][1].append(Y)
    return {k: (np.concatenate(x).astype(np.float32), np.concatenate(y).astype(np.float32))
            for k, (x, y) in data.items()}


def train(data, epochs=200, batch=1024, lr=2e-3, seed=0, time_budget=None, log=None, holdout=0.1):
    """Train one network per pair type on standardised inputs and outputs
    (Adam, learning rate halved every epochs/4), keeping a random fraction
    ``holdout`` of each type's samples out for validation.  Returns
    {type: MLP}, {type: stats}."""
    nets, stats = {}, {}
    t0 = time.perf_counter()
    rng = np.random.default_rng(seed)
    for ti, (key, (X, Y)) in enumerate(sorted(data.items())):
        order = rng.permutation(len(X))
        nval = int(holdout * len(X)) if len(X) >= 20 else 0
        val, tr = order[:nval], order[nval:]
        net = MLP(X.shape[1], Y.shape[1], seed=seed + ti)
        net.xmean, net.xstd = X[tr].mean(0), X[tr].std(0) + 1e-6
        net.ymean, net.ystd = Y[tr].mean(0), Y[tr].std(0) + 1e-6
        Xd = torch.tensor((X - net.xmean) / net.xstd, dtype=torch.float32, device="cuda")
        Yd = torch.tensor((Y - net.ymean) / net.ystd, dtype=torch.float32, device="cuda")
        tr_d = torch.as_tensor(tr, device="cuda")
        n = len(tr)
        g = torch.Generator(device="cpu").manual_seed(seed + ti)
        first = last = None
        for ep in range(epochs):
            perm = tr_d[torch.randperm(n, generator=g).to("cuda")]
            tot = torch.zeros(1, dtype=torch.float32, device="cuda")
            nb = 0
            for s0 in range(0, n, batch):
                ids = perm[s0:s0 + batch]
                xb, yb = Xd[ids].contiguous(), Yd[ids].contiguous()
                out, acts = net.forward(xb, keep=True)
                loss, dY = net.loss_grad(out, yb)
                gW, gb = net.backward(acts, dY)
                net.adam(gW, gb, lr=lr * (0.5 ** (ep / max(1, epochs // 4))))
                tot += loss
                nb += 1
            last = float(tot) / nb
            first = last if first is None else first
            if time_budget and time.perf_counter() - t0 > time_budget * (ti + 1) / len(data):
                break
        vloss = None
        if nval:
            vd = torch.as_tensor(val, device="cuda")
            vout = net.forward(Xd[vd].contiguous())
            vloss = float(((vout - Yd[vd]) ** 2).mean())
        nets[key] = net
        stats["%s-%s%s" % (key[0], key[1], "-diag" if key[2] else "")] = {
            "samples": int(n), "holdout": int(nval), "epochs": ep + 1, "loss_first": first, "loss_last": last,
            "holdout_loss": vloss}
        if log:
            log("type %s: %d samples, %d epochs, loss %.4g -> %.4g, holdout %s"
                % (key, n, ep + 1, first, last, "%.4g" % vloss if vloss is not None else "-"))
    return nets, stats


def assemble_density(mol, blocks, groups=None, device="cuda"):
    """Density (torch float64 on ``device``) from local-frame pair blocks
    {type: [P, n_a n_b]} (torch or numpy): D_ab = M_a(R)^T D'_ab M_b(R), the
    transpose for D_ba, the symmetric part on diagonal blocks.  Types missing
    from ``blocks`` stay zero.  The rotations and the scatter run on the host
    (a few hundred products of at most 15 x 15 matrices: as torch launches
    they cost more than the arithmetic), then one upload."""
    groups = pair_data(mol) if groups is None else groups
    off, ls = _atom_layout(mol)
    n = mol.NOrbitals
    D = np.zeros((n, n))
    for key, (a, b, F, R) in groups.items():
        if key not in blocks:
            continue
        la, lb = ls[a[0]], ls[b[0]]
        na, nb = sum((l + 1) * (l + 2) // 2 for l in la), sum((l + 1) * (l + 2) // 2 for l in lb)
        Y = blocks[key]
        Y = Y.detach().to("cpu", torch.float64).numpy() if isinstance(Y, torch.Tensor) else np.asarray(Y, dtype=float)
        R = R.detach().cpu().numpy() if isinstance(R, torch.Tensor) else np.asarray(R, dtype=float)
        G = np.transpose(atom_rot_batch(la, R), (0, 2, 1)) @ Y.reshape(-1, na, nb) @ atom_rot_batch(lb, R)
        rows = off[a][:, None] + np.arange(na)[None, :]
        cols = off[b][:, None] + np.arange(nb)[None, :]
        if key[2]:
            D[rows[:, :, None], rows[:, None, :]] = 0.5 * (G + np.transpose(G, (0, 2, 1)))
        else:
            D[rows[:, :, None], cols[:, None, :]] = G
            D[cols[:, :, None], rows[:, None, :]] = np.transpose(G, (0, 2, 1))
    return torch.as_tensor(D, device=device)


def predict_density(mol, nets, device="cuda", groups=None):
    """Alpha-density guess from the networks' local-frame blocks (pair types
    without a network stay zero); ``groups`` = pair_data(mol) when the caller
    has it already.  The networks run on the device; their outputs come back
    in one copy for the host assembly."""
    groups = pair_data(mol) if groups is None else groups
    outs = {}
    for key, (a, b, F, R) in groups.items():
        net = nets.get(key)
        if net is None:
            continue
        X = torch.tensor(((F - net.xmean) / net.xstd).astype(np.float32), device=device)
        outs[key] = net.forward(X)
    blocks = {}
    if outs:
        keys = list(outs)
        flat = torch.cat([outs[k].reshape(-1) for k in keys]).cpu().numpy()
        o = 0
        for k in keys:
            m = outs[k].numel()
            net = nets[k]
            y = flat[o:o + m].reshape(outs[k].shape).astype(np.float64)
            blocks[k] = y * np.asarray(net.ystd, dtype=np.float64) + np.asarray(net.ymean, dtype=np.float64)
            o += m
    return assemble_density(mol, blocks, groups, device)


def purify(D, S, nalpha, rounds=2):
    """Scale to tr(DS) = N_alpha, then McWeeny D <- 3 DSD - 2 DSDSD (numpy or
    torch)."""
    tr = (D * S).sum()
    D = D * (nalpha / max(1e-12, float(tr)))
    for _ in range(rounds):
        DS = D @ S
        D = 3.0 * DS @ D - 2.0 * DS @ DS @ D
        D = 0.5 * (D + D.T)
    return D


def guess_density(mol, nets, rounds=2, groups=None):
    """Learned guess for an SCF: predicted alpha density, purified against
    the overlap on the device (needs mol.Overlap)."""
    D = predict_density(mol, nets, groups=groups)
    dc = getattr(mol, "_device_core", None)   # S already on the device (the SCF's copy)
    if dc is not None and dc[0].device == D.device:
        S = dc[0]
    else:
        S = mol.Overlap.to(D.device) if isinstance(mol.Overlap, torch.Tensor) else torch.as_tensor(mol.Overlap, device=D.device)
    return purify(D, S, mol.NAlphaElectrons, rounds)


def save(nets, path, meta=None):
    arrays = {}
    for key, net in nets.items():
        tag = "%s_%s_%d" % (key[0], key[1], int(key[2]))
        for k, v in net.state().items():
            arrays["%s__%s" % (tag, k)] = v
    if meta:
        arrays["__meta__"] = np.frombuffer(__import__("json").dumps(meta).encode(), dtype=np.uint8)
    np.savez(path, **arrays)


def load(path):
    z = np.load(path, allow_pickle=False)
    groups = {}
    for name in z.files:
        if name == "__meta__":
            continue
        tag, k = name.split("__")
        groups.setdefault(tag, {})[k] = z[name]
    nets = {}
    for tag, d in groups.items():
        a, b, diag = tag.split("_")
        nets[(a, b, bool(int(diag)))] = MLP.from_state(d)
    return nets


DEFAULT_WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "data", "mlp_guess_631gs.npz")
_DEFAULT_NETS = None


def default_nets():
    """The shipped networks (6-31G*, Cartesian d), loaded once; None when the
    weights file is absent."""
    global _DEFAULT_NETS
    if _DEFAULT_NETS is None and os.path.exists(DEFAULT_WEIGHTS):
        _DEFAULT_NETS = load(DEFAULT_WEIGHTS)
    return _DEFAULT_NETS


def learned_guess(mol, nets=None):
    """Purified learned alpha density (torch, device) for ``mol``, or None
    when the networks do not cover it (other basis, spherical d, or a pair
    type without a network): the caller then falls back to SAD."""
    nets = default_nets() if nets is None else nets
    if not nets or mol.Basis != "631GS" or 2 not in mol.CartesianL:
        return None
    groups = pair_data(mol)
    if not set(groups) <= set(nets):
        return None
    return guess_density(mol, nets, groups=groups)


def training_molecules(count, seed=5, sigma=0.05):
    """Jittered C1..C8 alkanes and primary alcohols, 6-31G* (Cartesian d)."""
    from . import geometry
    rng = np.random.default_rng(seed)
    mols = []
    for k in range(count):
        n = int(rng.integers(1, 9))
        rows = geometry.alkane(n, sigma, int(rng.integers(1 << 30))) if rng.random() < 0.5 else \
            geometry.alcohol(n, sigma, int(rng.integers(1 << 30)))
        mols.append(structures.Molecule(rows, basis="6-31G*", cartesian_l=[2]))
    return mols
