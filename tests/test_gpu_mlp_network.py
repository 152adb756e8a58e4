"""The one-launch network kernels (pq_mlp_forward, pq_mlp_backward, the batch
split of the weight gradients) against torch in 64 bits, at the edges of their
tiles: rows around a 16-row strip, layer widths around the 16- and 32-column
tiles and the 448-column limit of the strip form.

Tolerances: a running bound of the FP32 rounding, propagated in 64 bits
through the same products with absolute values; a sum of K products in any
order is off by at most (K + 2) u sum |a b| with u = 2^-24, and tanh by a few
ulp.
"""
import numpy as np
import pytest
import torch

from pychem_amd import mlp_guess

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _bounded(net, X, dY):
    """(values, bounds) of the outputs and gradients, 64 bits."""
    W = [w.double() for w in net.W]
    b = [x.double() for x in net.b]
    A, EA = [X.double()], [torch.zeros_like(X, dtype=torch.float64)]
    n = len(W)
    for k in range(n):
        z = A[-1] @ W[k] + b[k]
        K = W[k].shape[0]
        e = EA[-1] @ W[k].abs() + (K + 3) * U * (A[-1].abs() @ W[k].abs() + b[k].abs())
        A.append(torch.tanh(z) if k < n - 1 else z)
        EA.append(e + 8 * U * A[-1].abs() if k < n - 1 else e)
    d, ed = dY.double(), torch.zeros_like(dY, dtype=torch.float64)
    gW, eW, gb, eb = [None] * n, [None] * n, [None] * n, [None] * n
    B = X.shape[0]
    for k in reversed(range(n)):
        if k < n - 1:
            f = 1.0 - A[k + 1] ** 2
            ed = ed * f + d.abs() * (2 * A[k + 1].abs() * EA[k + 1] + 4 * U)
            d = d * f
        gW[k] = A[k].T @ d
        eW[k] = (EA[k].T @ (d.abs() + ed)) + A[k].abs().T @ ed + (B + 2) * U * (A[k].abs().T @ d.abs())
        gb[k] = d.sum(0)
        eb[k] = ed.sum(0) + (B + 2) * U * d.abs().sum(0)
        ed = ed @ W[k].abs().T + (W[k].shape[1] + 3) * U * (d.abs() @ W[k].abs().T)
        d = d @ W[k].T
    return A[1:], EA[1:], gW, eW, gb, eb


def _check(got, want, bound):
    assert got.shape == want.shape
    # the bound is first order in u: twice it covers the higher orders
    assert bool(((got.double() - want).abs() <= 2.0 * bound + 1e-30).all())


@pytest.mark.parametrize("rows,outputs", [(1, 30), (15, 1), (16, 16), (17, 33), (156, 30), (67, 225), (513, 4),
                                          (30, 448), (33, 449)])
def test_network_kernels_within_rounding(gpu, rows, outputs):
    rng = np.random.default_rng(rows * 1000 + outputs)
    net = mlp_guess.MLP(mlp_guess.NFEAT, outputs, seed=outputs)
    for b in net.b:
        b.copy_(torch.as_tensor(rng.normal(0.0, 0.1, b.shape).astype(np.float32)))
    X = torch.as_tensor(rng.normal(size=(rows, mlp_guess.NFEAT)).astype(np.float32), device="cuda")
    dY = torch.as_tensor(rng.normal(size=(rows, outputs)).astype(np.float32), device="cuda")
    out, acts = net.forward(X, keep=True)
    alone = net.forward(X)
    gW, gb = net.backward(acts, dY)
    A, EA, rW, eW, rb, eb = _bounded(net, X, dY)
    assert torch.equal(out, alone) and acts[0] is X and acts[-1] is out
    for got, want, bound in zip(acts[1:] + gW + gb, A + rW + rb, EA + eW + eb):
        _check(got, want, bound)


def test_adam_over_several_tensors_equals_one_at_a_time(gpu):
    from pychem_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(3)
    sizes = [1, 255, 256, 257, 37 * 128]
    base = [[torch.rand(n, generator=g, device="cuda") for n in sizes] for _ in range(4)]
    one = [[t.clone() for t in ts] for ts in base]
    many = [[t.clone() for t in ts] for ts in base]
    L = _lib.lib()
    for p, gr, m, v in zip(*one):
        _lib.check(L.pq_mlp_adam(mlp_guess._ptr(p), mlp_guess._ptr(gr), mlp_guess._ptr(m), mlp_guess._ptr(v), p.numel(),
                                 1e-3, 0.9, 0.999, 1e-8, 3, mlp_guess._stream()), "pq_mlp_adam")
    import ctypes
    n = (ctypes.c_longlong * len(sizes))(*sizes)
    _lib.check(L.pq_mlp_adam_multi(len(sizes), *[mlp_guess._ptrs(ts) for ts in many], n, 1e-3, 0.9, 0.999, 1e-8, 3,
                                   mlp_guess._stream()), "pq_mlp_adam_multi")
    for a, b in zip(one, many):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
    assert not torch.equal(one[0][4], base[0][4])
