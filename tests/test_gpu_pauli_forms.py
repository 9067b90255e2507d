"""The two forms of a Pauli sum on a statevector (pauli_sum_grouped): which one
a size takes, and both against the oracle at the sizes and term counts next to
the lines between them.

Small states and short sums go term by term: by groups, <H> of 1000 Z strings on
4 qubits takes 200 instead of 58 us, H psi of 100 strings on 10 qubits 53
instead of 42.  24 qubits: more chunks than workgroups of <H>, so a workgroup
reuses its LDS copy for the next chunk.  Sums accumulate in FP64: 1e-12 of
sum |c| leaves a wide margin (each rounding is 1.1e-16), an FP32 result is
rounded once more (6e-8 relative per amplitude).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fsa():
    import __graft_entry__ as ge

    return ge.load_package()


def _sum(rng, n, terms):
    """Strings of weight 1-4 (the first on the lowest, the second on the highest qubit) and the identity."""
    paulis = np.zeros((terms, n), np.uint32)
    for t in range(terms):
        w = int(rng.integers(1, min(n, 4) + 1))
        paulis[t, rng.choice(n, w, replace=False)] = rng.integers(1, 4, w)
    paulis[0, 0] = 1
    if terms > 1:
        paulis[1, n - 1] = 2
    if terms > 2:
        paulis[2] = 0
    return rng.normal(size=terms), paulis


def _run(fsa, name, call):
    fsa.profile_enable(True)
    out = call()
    ran = [k for k in fsa.profile_read() if k.startswith("pauli_")]
    fsa.profile_enable(False)
    assert ran == [name], ran
    return out


@pytest.mark.parametrize("n,terms,expec,apply64,apply32", [
    (4, 1000, "terms", "terms", "terms"),
    (13, 100, "terms", "terms", "terms"),
    (19, 40, "terms", "terms", "terms"),
    (20, 1, "terms", "terms", "terms"),
    (20, 2, "groups", "terms", "terms"),
    (21, 64, "groups", "terms", "terms"),
    (22, 47, "groups", "terms", "terms"),
    (22, 48, "groups", "terms", "groups"),
    (22, 64, "groups", "groups", "groups"),
    (24, 5, "groups", "terms", "terms"),
])
def test_form_of_a_pauli_sum(fsa, orc, n, terms, expec, apply64, apply32):
    rng = np.random.default_rng(100 * n + terms)
    coeffs, paulis = _sum(rng, n, terms)
    scale = np.abs(coeffs).sum()
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    v /= np.linalg.norm(v)
    for prec, apply, tol in (("fp64", apply64, 1e-12), ("fp32", apply32, 1.2e-7)):
        psi, out = fsa.StateVector(n, precision=prec), fsa.StateVector(n, precision=prec)
        psi.upload(v)
        w = psi.download()                                  # what the device holds
        h = orc.sv_applyPauliSum(w, coeffs, paulis)
        e = _run(fsa, "pauli_expec_" + expec, lambda: fsa.statevector_expecPauliSum(psi, coeffs, paulis))
        assert abs(e - np.vdot(w, h)) <= 1e-12 * scale and e.imag == 0, (prec, e)
        _run(fsa, "pauli_apply_" + apply, lambda: fsa.statevector_applyPauliSum(psi, coeffs, paulis, out))
        assert np.linalg.norm(out.download() - h) <= tol * scale, prec
        psi.close()
        out.close()
