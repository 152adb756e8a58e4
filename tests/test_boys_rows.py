"""The class kernels' Boys polynomials (gen_eri.boys_lds_table): the rows
staged for each order against F_m from its series in 40 digits, at the grid
points, half-way between them and at the ends of the table.

Tolerance: the table's F values and the coefficients are rounded once each
(2 u of F_m over the row, u = 2^-53, and the row's higher terms add at most a
quarter), economising costs 4e-19, and 1.1e-21 x 9^2 / 0.05 in a derivative.
"""
import decimal
import os

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pychem_amd", "csrc")
U = 2.0 ** -53


def _horner(c, x):
    s = decimal.Decimal(0)
    for v in reversed(c):
        s = s * x + v
    return s


def _boys(m, T):
    with decimal.localcontext() as ctx:
        ctx.prec = 40
        T = decimal.Decimal(T)
        term = decimal.Decimal(1) / (2 * m + 1)
        s = term
        for i in range(1, 300):
            term = term * 2 * T / (2 * m + 2 * i + 1)
            s += term
        return s * (-T).exp()


@pytest.mark.parametrize("L", range(9))
def test_rows_reproduce_the_boys_functions(L, monkeypatch):
    monkeypatch.syspath_prepend(CSRC)
    gen = __import__("gen_eri")
    step, rows = gen.boys_rows(CSRC)
    text = gen.boys_lds_table(L, step, rows)[1]
    vals = [float(v) for v in text.split("{", 1)[1].split("}", 1)[0].replace("\n", " ").split(",") if v.strip()]
    assert len(vals) == 10 * len(rows)
    D = decimal.Decimal
    with decimal.localcontext() as ctx:
        ctx.prec = 40
        for k in (0, 1, 7, 100, 359, 360):
            c = [D(v) for v in vals[10 * k:10 * k + (8 if L == 0 else 9)]]
            for x in (0.0, 0.049, -0.049, 0.05, -0.05):
                T = D(step) * k - D(x)          # the row expands F(T_k - x)
                if T < 0:
                    continue
                poly = _horner(c, D(x))
                m = L - 1 if 0 < L <= gen.BOYS_PAIR_MAX else L
                F = _boys(m, T)
                assert abs(poly - F) <= D(2.5 * U) * F + D("1e-18")
                if m < L:
                    slope = _horner([j * v for j, v in enumerate(c)][1:], D(x))
                    G = _boys(L, T)
                    assert abs(slope - G) <= D(2.5 * U) * G + D("4e-18")
