"""The batched SCF's one-launch steps against their definitions in torch:
sizes around a wave and a block, molecules smaller than the padding, rings that
wrap, DIIS spaces of one up to past the one kept in LDS.

Tolerances: copies are exact; a sum of N products is off by at most (N + 8) u
sum |terms|; an elimination's solution by 8 q u cond(A) of its norm (q
unknowns, partial pivoting on these random systems grows no element tenfold).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _sizes(m, batch, rng):
    n = rng.integers(1, m + 1, batch)
    n[0] = m
    return n.astype(np.int64), np.concatenate([[0], np.cumsum(n * n)[:-1]]).astype(np.int64)


def _call(name, *args):
    import torch
    from pychem_amd import _lib
    from pychem_amd.engine import _ptr, _stream
    _lib.check(getattr(_lib.lib(), name)(*(_ptr(a) if isinstance(a, torch.Tensor) else a for a in args), _stream()), name)


@pytest.mark.parametrize("m,batch", [(1, 1), (7, 3), (16, 5), (33, 2)])
def test_pack_fock_and_convergence(gpu, m, batch):
    import torch
    rng = np.random.default_rng(m)
    n, base = _sizes(m, batch, rng)
    dev = lambda x: torch.as_tensor(np.ascontiguousarray(x), device="cuda")
    inside = np.zeros((batch, m, m))
    for b in range(batch):
        inside[b, :n[b], :n[b]] = 1
    D, Dn, H, R = (rng.normal(size=(batch, m, m)) * inside for _ in range(4))
    done = rng.integers(0, 2, batch).astype(bool)
    total = int((n * n).sum())
    Dj, Dk, Dd = torch.zeros(total, dtype=torch.float64, device="cuda"), torch.zeros(total, dtype=torch.float64, device="cuda"), dev(D)
    nd, bd, dd = dev(n), dev(base), dev(done)
    _call("pq_batch_pack", batch, m, bd, nd, Dd, dev(Dn), dd, Dj, Dk)
    sel = np.where(done[:, None, None], D, Dn)
    assert np.array_equal(Dd.cpu().numpy(), sel)
    packed = np.concatenate([sel[b, :n[b], :n[b]].ravel() for b in range(batch)])
    assert np.array_equal(Dk.cpu().numpy(), packed) and np.array_equal(Dj.cpu().numpy(), 2 * packed)
    _call("pq_batch_pack", batch, m, bd, nd, Dd, None, None, Dj, Dk)
    assert np.array_equal(Dd.cpu().numpy(), sel) and np.array_equal(Dk.cpu().numpy(), packed)
    J, K = rng.normal(size=(2, total))
    F = torch.empty((batch, m, m), dtype=torch.float64, device="cuda")
    _call("pq_batch_fock", batch, m, bd, nd, dev(H), dev(J), dev(K), F)
    Fr = H.copy()
    for b in range(batch):
        s = slice(base[b], base[b] + n[b] ** 2)
        Fr[b, :n[b], :n[b]] = H[b, :n[b], :n[b]] + J[s].reshape(n[b], n[b]) + K[s].reshape(n[b], n[b])
    assert np.array_equal(F.cpu().numpy(), Fr)
    enuc, E0 = rng.normal(size=batch), rng.normal(size=batch)
    ev = (sel * (H + Fr) * inside).sum((1, 2)) + enuc
    tol = (m * m + 8) * U * (np.abs(sel) * np.abs(H + Fr)).sum((1, 2)) + 4 * U * np.abs(enuc)
    E0[::2] = ev[::2] + 1e-3     # these settle, the others moved by more
    R[batch // 2:] *= 1e-9
    R[-1, 0, 0] = np.nan if batch > 3 else 0.0
    E, iters, newly = dev(E0), torch.zeros(batch, dtype=torch.long, device="cuda"), torch.zeros(batch, dtype=torch.bool, device="cuda")
    flags = torch.zeros(3, dtype=torch.int32, device="cuda")
    _call("pq_batch_test", batch, m, nd, dev(sel), dev(H), F, dev(R), dev(enuc), 1e-2, 1e-4, 5, E, iters, dd, newly, flags)
    new = ~done & (np.abs(ev - E0) < 1e-2) & (np.abs(R).max((1, 2)) <= 1e-4)
    assert np.array_equal(newly.cpu().numpy(), new) and np.array_equal(dd.cpu().numpy(), done | new)
    assert (np.abs(E.cpu().numpy() - np.where(done, E0, ev)) <= tol).all()
    assert np.array_equal(iters.cpu().numpy(), np.where(done, 0, 5))
    assert flags.tolist() == [int(new.any()), int((~(done | new)).sum()), 0]


@pytest.mark.parametrize("m,diis,cycles", [(5, 1, 3), (5, 3, 9), (17, 8, 12), (9, 70, 72)])
def test_diis_ring(gpu, m, diis, cycles):
    import torch
    from pychem_amd import _lib
    rng = np.random.default_rng(m + diis)
    batch, S = 3, diis + 1
    z = lambda *s: torch.zeros(s, dtype=torch.float64, device="cuda")
    Fb, Rb, G, Fx = z(batch, S, m, m), z(batch, S, m, m), z(batch, S, S), z(batch, m, m)
    flags = torch.zeros(3, dtype=torch.int32, device="cuda")
    hist = []
    for it in range(1, cycles + 1):
        F, R = rng.normal(size=(2, batch, m, m))
        hist = (hist + [(F, R)])[-diis:]
        k = len(hist)
        work = z(max(1, _lib.lib().pq_batch_diis_work(batch, k)))
        _call("pq_batch_diis", batch, m, torch.as_tensor(F, device="cuda"), torch.as_tensor(R, device="cuda"), Fb, Rb, G, S,
              (it - 1) % S, k, Fx, work, flags)
        out = Fx.cpu().numpy()
        for b in range(batch):
            if k < 2:
                assert np.array_equal(out[b], F[b])
                continue
            r = np.array([h[1][b].ravel() for h in hist])
            g = r @ r.T
            A = np.full((k + 1, k + 1), -1.0)
            A[:k, :k] = g + (1e-14 * g.trace() / k + 1e-300) * np.eye(k)
            A[k, k] = 0.0
            c = np.linalg.solve(A, np.r_[np.zeros(k), -1.0])[:k]
            f = np.array([h[0][b].ravel() for h in hist])
            tol = 16 * (k + 1) * U * np.linalg.cond(A) * np.linalg.norm(c) * np.linalg.norm(f, axis=0)
            tol += 2 * (m * m + 8) * U * np.linalg.cond(A) * np.linalg.norm(f, axis=0)
            assert (np.abs(out[b].ravel() - c @ f) <= tol).all()
    assert flags.tolist() == [0, 0, 0]


@pytest.mark.parametrize("m", [1, 5, 64, 65])
def test_lift(gpu, m):
    import torch
    rng = np.random.default_rng(m)
    M = rng.normal(size=(3, m, m)) - 2.0 * (rng.integers(0, 2, (3, 1, 1)))
    drop = rng.integers(0, 2, (3, m)).astype(float)
    d = np.einsum("bii->bi", M)
    top = np.maximum((d + np.abs(M).sum(2) - np.abs(d)).max(1), 0.0) + 1.0
    ref = M + np.einsum("bi,ij->bij", drop * top[:, None], np.eye(m))
    t = torch.as_tensor(M.copy(), device="cuda")
    _call("pq_batch_lift", 3, m, t, torch.as_tensor(drop, device="cuda"))
    assert (np.abs(t.cpu().numpy() - ref) <= (m + 8) * U * (np.abs(M).sum(2).max((1,), keepdims=True) + 2)[:, :, None]).all()


def _tc2(A, nocc, tol=1e-11, max_steps=200):
    """The purification over the whole matrix: (P, steps)."""
    d = np.diag(A)
    rad = np.abs(A).sum(1) - np.abs(d)
    lo, hi = (d - rad).min(), (d + rad).max()
    X, last, k = (hi * np.eye(len(A)) - A) / (hi - lo), False, 0
    while k < max_steps:
        X2 = X @ X
        t1, t2 = np.trace(X), np.trace(X2)
        X = X2 if abs(t2 - nocc) < abs(2 * t1 - t2 - nocc) else 2 * X - X2
        if last:
            break
        last = t1 - t2 < tol
        k += 1
    return 0.5 * (X + X.T), k + 1 if last else max_steps + 1


@pytest.mark.parametrize("m,coupled", [(5, 0), (16, 15), (17, 16), (33, 17), (48, 48), (61, 7), (90, 65), (90, 90)])
def test_projectors_with_uncoupled_rows(gpu, m, coupled):
    """Trailing rows that couple to nothing, above the rest or among its
    levels, against the same steps over the whole matrix.  The purified X is
    idempotent to 1e-11 before the last squaring and the spectra have a gap of
    1 at the Fermi level: 1e-10."""
    import torch
    from pychem_amd.engine import purify_batched
    rng = np.random.default_rng(m + 100 * coupled)
    A, nocc = np.zeros((4, m, m)), np.zeros(4, dtype=np.int64)
    for b in range(4):
        low = rng.integers(0, m + 1)
        lam = np.concatenate([rng.uniform(-3, -0.5, low), rng.uniform(0.5, 3, m - low)])
        rng.shuffle(lam)
        Q = np.eye(m)
        if coupled:
            Q[:coupled, :coupled] = np.linalg.qr(rng.normal(size=(coupled, coupled)))[0]
        A[b] = (Q * lam) @ Q.T
        A[b] = 0.5 * (A[b] + A[b].T)
        nocc[b] = low
    P, steps = purify_batched(torch.as_tensor(A, device="cuda"), nocc)
    for b in range(4):
        ref, k = _tc2(A[b], nocc[b])
        assert np.abs(P[b].cpu().numpy() - ref).max() < 1e-10
        assert int(steps[b]) == k


@pytest.mark.parametrize("n,coupled", [(1, 0), (5, 0), (16, 2), (17, 16), (61, 7), (64, 64), (65, 63), (90, 89)])
def test_eigenpairs_with_uncoupled_rows(gpu, n, coupled):
    """Trailing rows that couple to nothing, repeated levels among them.  The
    sweeps stop at 1e-15 of the diagonal; each of some 10 sweeps of n rounds
    rounds an element twice: 20 n u of the norm at most, 1e-12 at n = 90."""
    import torch
    from pychem_amd.engine import eigh_batched
    rng = np.random.default_rng(7 * n + coupled)
    A = np.zeros((3, n, n))
    for b in range(3):
        A[b] = np.diag(rng.integers(-3, 4, n).astype(float))
        B = rng.normal(size=(coupled, coupled))
        A[b, :coupled, :coupled] = B + B.T
    w, V = (x.cpu().numpy() for x in eigh_batched(torch.as_tensor(A, device="cuda")))
    ref = np.linalg.eigvalsh(A)
    scale = max(1.0, np.abs(ref).max())
    assert np.abs(w - ref).max() <= 1e-12 * scale
    for b in range(3):
        assert np.abs(A[b] @ V[b] - V[b] * w[b]).max() <= 1e-12 * scale
        assert np.abs(V[b].T @ V[b] - np.eye(n)).max() <= 1e-12
