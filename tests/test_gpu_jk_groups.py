"""The grouped J/K launches: molecules of one atom and one class upward, FP32
lists, one stream and four, persistent blocks, the timed build and the
allocation-free entry against a float64 contraction of the dense integrals.

Tolerance: each matrix element sums at most n^2 products, rounded once per
addition; FP32 lists hold values rounded to 2^-24 of themselves, which the
dense tensor holds as well.
"""
import numpy as np
import pytest

from pychem_amd import geometry, structures

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def _case(rows, basis, cartesian, fp32, seed):
    import torch
    from pychem_amd.engine import Engine
    m = structures.Molecule(rows, basis=basis, cartesian_l=cartesian, multiplicity=1)
    e = Engine(m)
    e.build_eri(1e-8, fp32)
    n = e.ncart
    rng = np.random.default_rng(seed)
    D = rng.normal(size=(2, n, n))
    D = D + D.transpose(0, 2, 1)
    t = torch.empty((n, n, n, n), dtype=torch.float64, device="cuda")
    from pychem_amd import _lib
    from pychem_amd.engine import _ptr, _stream
    _lib.check(_lib.lib().pq_eri_dense(e.h, _ptr(t), _stream()), "pq_eri_dense")
    eri = t.cpu().numpy()
    J = np.einsum("abcd,cd->ab", eri, D[0], optimize=True)
    K = -np.einsum("abcd,cb->ad", eri, D[1], optimize=True)
    Jm = np.einsum("abcd,cd->ab", np.abs(eri), np.abs(D[0]), optimize=True)
    Km = np.einsum("abcd,cb->ad", np.abs(eri), np.abs(D[1]), optimize=True)
    tol = 4 * (n * n + 16) * U
    return e, torch.as_tensor(D, device="cuda"), (J, tol * Jm), (K, tol * Km)


def _jk(e, D, fn="pq_jk"):
    import torch
    from pychem_amd import _lib
    from pychem_amd.engine import _ptr, _stream
    J, K = torch.full_like(D[0], 7.0), torch.full_like(D[0], 7.0)
    _lib.check(getattr(_lib.lib(), fn)(e.h, _ptr(D[0]), _ptr(D[1]), _ptr(J), _ptr(K), _stream()), fn)
    return J.cpu().numpy(), K.cpu().numpy()


ROWS = {"He": [["He", 2.0, 0.0, 0.0, 0.0]], "Ne": [["Ne", 10.0, 0.0, 0.0, 0.0]],
        "H2O": geometry.small_molecule("H2O", 0.05, 3), "CH3OH": geometry.small_molecule("CH3OH", 0.05, 4),
        "C4H10": geometry.alkane(4, 0.05, 5)}


@pytest.mark.parametrize("name,basis,cartesian,fp32", [
    ("He", "STO-3G", [2], 0.0), ("He", "6-31G*", [2], 0.0), ("Ne", "6-31G*", [2], 0.0), ("H2O", "STO-3G", [2], 1e-3),
    ("CH3OH", "6-31G*", [2], 0.0), ("CH3OH", "6-31G*", [2], 1e-2), ("C4H10", "6-31G*", [2], 1e-5),
    ("C4H10", "6-311G*", [2], 0.0)])
def test_builds_against_the_dense_integrals(gpu, name, basis, cartesian, fp32):
    from pychem_amd import _lib
    L = _lib.lib()
    e, D, (J, eJ), (K, eK) = _case(ROWS[name], basis, cartesian, fp32, len(name))

    def check(got):
        assert (np.abs(got[0] - J) <= eJ).all() and (np.abs(got[1] - K) <= eK).all()

    for ns in (1, 4):
        _lib.check(L.pq_jk_set_streams(e.h, ns), "pq_jk_set_streams")
        check(_jk(e, D))
    check(_jk(e, D, "pq_jk_general"))
    check(_jk(e, D, "pq_jk_general_noalloc"))
    for cls in range(L.pq_eri_nclass()):          # short items, three persistent blocks a tile
        _lib.check(L.pq_jk_set_params(e.h, cls, 64, 3, None), "pq_jk_set_params")
    check(_jk(e, D))
    e.set_timing(True)
    e.jk_class_times(reset=True)
    check(_jk(e, D))
    check(_jk(e, D))
    ms, calls, items = e.jk_class_times()
    stored = np.array([s["nq64"] + s["nq32"] > 0 for s in e.stats()])
    assert (calls[stored] == 2).all() and (calls[~stored] == 0).all()
    assert (ms[stored] > 0.0).all() and (ms < 100.0).all() and (items[stored] > 0).all()
    e.close()


def test_rows_beyond_64_kib_of_lds(gpu):
    """Three distant octanes in one molecule (468 functions: 67 KB of rows for
    the nine-row tiles): with a density on one of them its own J block, and
    every octane's K block, are those of the octane alone, to the rounding of
    the same sums in another order."""
    import torch
    from pychem_amd.engine import Engine
    one = geometry.alkane(8, 0.02, 9)
    far = [[r[0], r[1], r[2], r[3] + 200.0 * k, r[4]] for k in range(3) for r in one]
    ms = [structures.Molecule(rows, basis="6-31G*", cartesian_l=[2]) for rows in (one, far)]
    es = [Engine(m) for m in ms]
    for e in es:
        e.build_eri(1e-8)
    n = es[0].ncart
    assert es[1].ncart == 3 * n and 9 * 16 * 3 * n > 65536
    # fragments of the long molecule hold the same atoms in the same order
    rng = np.random.default_rng(8)
    A = rng.normal(size=(n, n))
    D = torch.as_tensor(A + A.T, device="cuda")
    J1, K1 = es[0].jk(D, D)
    Dj, Dk = (torch.zeros((3 * n, 3 * n), dtype=torch.float64, device="cuda") for _ in range(2))
    Dj[:n, :n] = D
    for k in range(3):
        Dk[k * n:(k + 1) * n, k * n:(k + 1) * n] = D
    J3, K3 = es[1].jk(Dj, Dk)
    # translations round the coordinates of two of them (200 A: 2^-53 * 400 bohr)
    assert (J3[:n, :n] - J1).abs().max().item() < 1e-11 * J1.abs().max().item()
    for k in range(3):
        blk = K3[k * n:(k + 1) * n, k * n:(k + 1) * n]
        assert (blk - K1).abs().max().item() < 1e-10 * K1.abs().max().item()
    for e in es:
        e.close()


@pytest.mark.parametrize("fp32", [0.0, 1e-5])
def test_reductions_behind_each_group(gpu, fp32):
    """Above 1 GB of stored integrals the ket sums of a group run behind it on
    its own stream: four streams against one.  A term of J_ab is at most
    Q_ab Q_cd |D_cd| (Schwarz), in any order of n^2 additions."""
    import torch
    from pychem_amd import _lib
    from pychem_amd.engine import Engine
    m = structures.Molecule(geometry.alkane(16, 0.05, 5), basis="6-31G*", cartesian_l=[2], multiplicity=1)
    e = Engine(m)
    e.build_eri(1e-8, fp32)
    n = e.ncart
    assert sum((s["nq64"] * 8 + s["nq32"] * 4) * s["ncomp"] for s in e.stats()) > 1e9 or fp32
    D = np.random.default_rng(9).normal(size=(2, n, n))
    D = torch.as_tensor(D + D.transpose(0, 2, 1), device="cuda")
    L = _lib.lib()
    out = {}
    for ns in (1, 4):
        _lib.check(L.pq_jk_set_streams(e.h, ns), "pq_jk_set_streams")
        out[ns] = _jk(e, D)
    Q = e.schwarz()
    tol = 4 * (n * n + 16) * U * Q.max() * Q.sum() * 36 * float(D.abs().max())
    for a, b in zip(out[1], out[4]):
        assert np.abs(a - b).max() <= tol
    assert np.abs(out[1][0]).max() > 1e3 * tol
