"""The long-side matrix-core products and the packed-pair quarter transforms
at the edges of their tiles: short sides around the 16-row blocks and the
80-row tile, long sides around the 128-column tile and past each other (either
operand can be the long one), K around the 4-, 16- and 32-deep steps; orbital
spaces that differ, FP32 lists, one-row slabs.

Tolerances: a sum of K products in any order is off by at most (K + 2) u
sum |a b|, u = 2^-53; four quarter transforms in a row by their sum.  Split
BF16 operands keep 16 bits (2^-17 per operand rounding lo, and lo lo dropped,
2^-16), plus the FP32 sum.
"""
import ctypes

import numpy as np
import pytest

from pychem_amd import geometry, structures

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.mark.parametrize("shape", [(1, 129, 4), (16, 128, 16), (17, 127, 17), (41, 300, 33), (80, 256, 3), (81, 129, 31),
                                   (161, 97, 32), (300, 15, 50), (128, 128, 1)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("precision", ["fp64", "bf16x3"])
def test_products_at_tile_edges(gpu, shape, ta, tb, precision):
    """Strided operands, batch 2, alpha and beta."""
    import torch
    from pychem_amd import _lib
    from pychem_amd.engine import _ptr, _stream
    M, N, K = shape
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    ra, ca = (K, M) if ta else (M, K)
    rb, cb = (N, K) if tb else (K, N)
    A = torch.as_tensor(rng.normal(size=(2, ra, ca + 3)), device="cuda")
    B = torch.as_tensor(rng.normal(size=(2, rb, cb + 1)), device="cuda")
    C = torch.as_tensor(rng.normal(size=(2, M, N + 5)), device="cuda")
    C0 = C.clone()
    fn = {"fp64": "pq_gemm_f64", "bf16x3": "pq_gemm_bf16x3"}[precision]
    _lib.check(getattr(_lib.lib(), fn)(int(ta), int(tb), M, N, K, 0.5, _ptr(A), ca + 3, ra * (ca + 3), _ptr(B), cb + 1,
                                       rb * (cb + 1), 2.0, _ptr(C), N + 5, M * (N + 5), 2, _stream()), fn)
    a = A[:, :, :ca].transpose(1, 2) if ta else A[:, :, :ca]
    b = B[:, :, :cb].transpose(1, 2) if tb else B[:, :, :cb]
    a, b = a.cpu().numpy(), b.cpu().numpy()
    ref = 0.5 * (a @ b) + 2.0 * C0[:, :, :N].cpu().numpy()
    mag = 0.5 * (np.abs(a) @ np.abs(b)) + 2.0 * np.abs(C0[:, :, :N].cpu().numpy())
    # per product: both operands' rounding (2 x 2^-17), lo lo (2^-16); the FP32 sum of 3 K terms
    tol = (K + 4) * U if precision == "fp64" else 2.0 ** -15 + (3 * K + 4) * 2.0 ** -24
    assert (np.abs(C[:, :, :N].cpu().numpy() - ref) <= tol * mag).all()
    assert torch.equal(C[:, :, N:], C0[:, :, N:])


def _spaces(n, rng):
    Q = np.linalg.qr(rng.normal(size=(n, n)))[0]
    R = np.linalg.qr(rng.normal(size=(n, n)))[0]
    return Q, R


@pytest.mark.parametrize("name,basis,cartesian,fp32", [("H2O", "STO-3G", [2], 0.0), ("CH3OH", "6-31G*", [2], 0.0),
                                                       ("CH3OH", "6-31G*", [], 1e-4), ("NH3", "6-31G*", [2], 1e-3)])
def test_transform_of_two_spaces_and_slabs(gpu, name, basis, cartesian, fp32):
    from pychem_amd.engine import Engine
    m = structures.Molecule(geometry.small_molecule(name, 0.05, 5), basis=basis, cartesian_l=cartesian)
    e = Engine(m)
    e.build_eri(1e-8, fp32)
    n = m.NOrbitals
    Q, R = _spaces(n, np.random.default_rng(n))
    o1, o2, v1, v2 = 3, 2, n - 3, 4
    Co1, Cv1, Co2, Cv2 = (np.ascontiguousarray(x) for x in (Q[:, :o1], Q[:, o1:], R[:, :o2], R[:, n - v2:]))
    eri = e.eri_dense().cpu().numpy()

    def transform(t, a, b, c, d):
        t = np.einsum("mi,mnls->inls", a, t, optimize=True)
        t = np.einsum("na,inls->ials", b, t, optimize=True)
        t = np.einsum("lj,ials->iajs", c, t, optimize=True)
        return np.einsum("sb,iajs->iajb", d, t, optimize=True)

    ref = transform(eri, Co1, Cv1, Co2, Cv2)
    mag = transform(np.abs(eri), *(np.abs(x) for x in (Co1, Cv1, Co2, Cv2)))
    got = e.mp2_ovov(Co1, Cv1, Co2, Cv2).cpu().numpy()
    # both sides round (4 quarters of n terms each, the 5d transform in front)
    assert (np.abs(got - ref) <= 2 * (6 * (n + 12)) * U * mag).all()
    for prec in ("fp64", "bf16x3"):
        whole = e.mp2_ovov(Co1, Cv1, Co2, Cv2, precision=prec)
        for slab in (1, 5 * 8 * n * n):       # one packed row at a time; a few rows, the last slab short
            assert (e.mp2_ovov(Co1, Cv1, Co2, Cv2, max_slab_bytes=slab, precision=prec) == whole).all()
    e.close()


@pytest.mark.parametrize("o,v", [(1, 1), (2, 31), (3, 32), (2, 33), (5, 70)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_energy_tiles(gpu, o, v, mode):
    import torch
    from pychem_amd.engine import mp2_energy
    rng = np.random.default_rng(o * 100 + v)
    o2, v2 = (o, v) if mode != 2 else (o + 1, v + 3)
    ov = rng.normal(size=(o, v, o2, v2))
    eo1, ev1, eo2, ev2 = rng.uniform(-2, -1, o), rng.uniform(0.5, 3, v), rng.uniform(-2, -1, o2), rng.uniform(0.5, 3, v2)
    den = eo1[:, None, None, None] + eo2[None, None, :, None] - ev1[None, :, None, None] - ev2[None, None, None, :]
    x = ov.transpose(0, 3, 2, 1) if mode != 2 else 0.0
    terms = {0: ov * (2 * ov - x), 1: 0.25 * (ov - x) ** 2, 2: ov * ov}[mode] / den
    got = mp2_energy(torch.as_tensor(ov, device="cuda"), eo1, ev1, eo2, ev2, mode)
    assert abs(got - terms.sum()) <= (ov.size + 8) * U * np.abs(terms).sum() * 2
