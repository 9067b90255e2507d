"""The two forms of a Pauli sum on a statevector (by_groups in circuit.cpp): which one
a size takes, and both against the oracle at the sizes and term counts next to
the lines between them.

Small states and short sums of scattered strings go term by term: by groups,
<H> of 1000 Z strings on 4 qubits takes 200 instead of 58 us, H psi of 16 strings
on 23 qubits FP64 170 instead of 129.  24 qubits: more chunks than workgroups of
<H>, so a workgroup reuses its LDS copy for the next chunk.  Sums accumulate in
FP64: 1e-12 of sum |c| leaves a wide margin (each rounding is 1.1e-16), an FP32
result is rounded once more (6e-8 relative per amplitude).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fsa():
    import __graft_entry__ as ge

    return ge.load_package()


def _sum(rng, n, terms, kind):
    """far: strings of weight 1-4 with X or Y on a qubit above the lowest 11, all masks different
    there; near: X and Y on the lowest 11 only, and the identity; z: Z strings; one: X on the highest qubit."""
    paulis = np.zeros((terms, n), np.uint32)
    for t in range(terms):
        if kind == "far":
            # the 2^(n-11) masks above the chunk, from 1 on
            for b in range(n - 11):
                if ((t + 1) >> b) & 1:
                    paulis[t, 11 + b] = rng.integers(1, 3)
            paulis[t, rng.integers(11)] = rng.integers(1, 4)
        elif kind == "near":
            w = int(rng.integers(0, min(n, 4) + 1))
            paulis[t, rng.choice(n, w, replace=False)] = 3
            paulis[t, rng.choice(min(n, 11), min(w, 2), replace=False)] = rng.integers(1, 4, min(w, 2))
        elif kind == "z":
            paulis[t] = 3 * rng.integers(0, 2, n)
        else:
            paulis[t, n - 1] = 1
    return rng.normal(size=terms), paulis


def _run(fsa, name, call):
    fsa.profile_enable(True)
    out = call()
    ran = [k for k in fsa.profile_read() if k.startswith("pauli_")]
    fsa.profile_enable(False)
    assert ran == [name], ran
    return out


@pytest.mark.parametrize("n,terms,kind,expec,apply64,apply32", [
    (4, 1000, "z", "terms", "terms", "terms"),
    (13, 100, "near", "terms", "terms", "terms"),
    (18, 40, "near", "terms", "terms", "terms"),
    (19, 3, "far", "terms", "terms", "terms"),
    (19, 4, "near", "groups", "terms", "terms"),
    (20, 1, "z", "terms", "terms", "terms"),
    (20, 1, "one", "groups", "terms", "terms"),
    (20, 2, "far", "groups", "terms", "terms"),
    (20, 4, "z", "groups", "groups", "groups"),
    (20, 99, "far", "groups", "terms", "terms"),
    (20, 100, "far", "groups", "groups", "terms"),
    (21, 1, "one", "groups", "terms", "terms"),
    (21, 3, "near", "groups", "terms", "groups"),
    (21, 64, "far", "groups", "groups", "groups"),
    (22, 1, "one", "groups", "terms", "groups"),
    (22, 23, "far", "groups", "terms", "groups"),
    (22, 24, "far", "groups", "groups", "groups"),
    (24, 5, "near", "groups", "groups", "groups"),
])
def test_form_of_a_pauli_sum(fsa, orc, n, terms, kind, expec, apply64, apply32):
    rng = np.random.default_rng(100 * n + terms)
    coeffs, paulis = _sum(rng, n, terms, kind)
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
