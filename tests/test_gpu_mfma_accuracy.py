"""Rounding of the FP64 matrix-unit forms of 4-target gates.

The circuits are computed in extended precision, and again with every multiply-add
rounded to 64 bits in the order of two reference forms: the plain complex product,
and Gauss's three products P1, P2 and P3 with P3 added to -(P1 + P2).  Tiles of 2^12
amplitudes must be no further off than the latter (with a sum of its own for P3 and
Yi = P3 - (P1 + P2) they were, by 2.2%), tiles of 2^13, which take the plain product,
closer to the former than to the latter.  Errors are means over ten circuits, whose
scatter is 0.3%.
"""
import numpy as np
import pytest

from test_emu_kernels import _unitary

pytestmark = pytest.mark.gpu

LD, D = np.longdouble, np.float64


def _fma(acc, a, b):
    """acc + a b rounded to 64 bits (the product to 80 bits, which adds 1/2048 of a rounding)."""
    return (acc.astype(LD) + a.astype(LD) * b.astype(LD)).astype(D)


def _plain(u, x):
    yr, yi = np.zeros(x.shape), np.zeros(x.shape)
    for c in range(u.shape[0]):
        a, b = u[:, c, None], x[None, c]
        yr = _fma(_fma(yr, a.real, b.real), -a.imag, b.imag)
        yi = _fma(_fma(yi, a.real, b.imag), a.imag, b.real)
    return yr + 1j * yi


def _gauss(u, x):
    p1, p2 = np.zeros(x.shape), np.zeros(x.shape)
    for c in range(u.shape[0]):
        a, b = u[:, c, None], x[None, c]
        p1, p2 = _fma(p1, a.real, b.real), _fma(p2, a.imag, b.imag)
    yi = -(p1 + p2)
    for c in range(u.shape[0]):
        a, b = u[:, c, None], x[None, c]
        yi = _fma(yi, a.real + a.imag, b.real + b.imag)
    return (p1 - p2) + 1j * yi


def _circuit(n, ops, product, dtype):
    v = np.zeros(1 << n, dtype)
    v[0] = 1
    for _, (q, u) in ops:
        axes = [n - 1 - t for t in reversed(q)]
        x = np.moveaxis(v.reshape((2,) * n), axes, range(len(q)))
        shape = x.shape
        x = product(u.astype(dtype), x.reshape(1 << len(q), -1)).reshape(shape)
        v = np.moveaxis(x, range(len(q)), axes).reshape(-1)
    return v


def test_matrix_products_of_four_targets_round_no_worse(monkeypatch):
    import __graft_entry__ as ge

    fsa = ge.load_package()
    n = 14
    errors = dict.fromkeys(("plain", "gauss", "12", "13"), 0.0)
    for seed in range(10):
        rng = np.random.default_rng(seed)
        ops = [("manyTargGate", ([int(t) for t in rng.permutation(n)[:4]], _unitary(rng, 16))) for _ in range(30)]
        v = _circuit(n, ops, lambda u, x: u @ x, np.clongdouble)
        out = {"plain": _circuit(n, ops, _plain, complex), "gauss": _circuit(n, ops, _gauss, complex)}
        for bits in ("12", "13"):
            monkeypatch.setenv("FSA_TILE_BITS", bits)
            psi = fsa.StateVector(n)
            psi.init_zero()
            fsa.profile_enable(True)
            fsa.Circuit(ops).apply(psi)
            out[bits] = psi.download()
            ran = fsa.profile_read()
            fsa.profile_enable(False)
            assert any("mfma" in k for k in ran), ran
            psi.close()
        for k, w in out.items():
            errors[k] += float(np.sqrt((np.abs(w - v) ** 2).sum())) / 10
    assert errors["12"] <= errors["gauss"], errors
    assert errors["13"] <= (errors["plain"] + errors["gauss"]) / 2, errors
