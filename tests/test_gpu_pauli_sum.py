"""Grouped Pauli sums on a statevector (k_pauli_groups) against the oracle.

Sizes: states smaller than a workgroup, one workgroup, the last size of the
one-amplitude form (19 qubits) and the first of the eight-amplitude form (20),
whose X/Y masks fall on lanes, on a thread's amplitudes and on the chunk index.
The sums accumulate in FP64: n-term sums of products of magnitude at most 1
keep 1e-12 of sum |c| with a wide margin (each rounding is 1.1e-16).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fsa():
    import __graft_entry__ as ge

    return ge.load_package()


def _strings(rng, n, kind):
    if kind == "ising":            # many terms on one mask, then one mask per qubit
        rows = []
        for q in range(n):
            z = np.zeros(n, np.uint32)
            z[[q, (q + 1) % n]] = 3
            x = np.zeros(n, np.uint32)
            x[q] = 1
            rows += [z, x]
        return np.array(rows)
    if kind == "single":
        p = np.zeros((1, n), np.uint32)
        p[0, n - 1] = 2
        return p
    p = rng.integers(0, 4, (37, n)).astype(np.uint32)
    # the same X/Y mask with real and with imaginary factors, and the identity
    p[1] = p[0]
    q = int(rng.integers(n))
    p[0, q], p[1, q] = 1, 2
    p[2] = 0
    return p


@pytest.mark.parametrize("kind", ["random", "ising", "single"])
@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 13, 19, 20, 21])
def test_pauli_sum_forms(fsa, orc, n, kind):
    if kind == "ising" and n < 2:
        pytest.skip("needs a pair")
    rng = np.random.default_rng(1000 * n + len(kind))
    paulis = _strings(rng, n, kind)
    coeffs = rng.normal(size=len(paulis))
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    v /= np.linalg.norm(v)
    for prec in ("fp64", "fp32"):
        psi, out = fsa.StateVector(n, precision=prec), fsa.StateVector(n, precision=prec)
        psi.upload(v)
        w = psi.download()                                  # what the device holds
        h = orc.sv_applyPauliSum(w, coeffs, paulis)
        scale = np.abs(coeffs).sum()
        e = fsa.statevector_expecPauliSum(psi, coeffs, paulis)
        assert abs(e - np.vdot(w, h)) <= 1e-12 * scale, (n, prec, e)
        assert e.imag == 0
        fsa.statevector_applyPauliSum(psi, coeffs, paulis, out)
        # FP32 results are rounded once (6e-8 relative per amplitude)
        tol = 1e-12 if prec == "fp64" else 1.2e-7
        assert np.linalg.norm(out.download() - h) <= tol * scale
        # psi is an input only
        assert np.array_equal(psi.download(), w)
