"""Register-tile passes of the adjoint (wave_sweep.hpp): on the
CPU stand-in under AddressSanitizer and on the GPU, against the oracle's adjoint.

The circuit holds every op the passes take, on every kind of bit (lane,
register, outside the tile): X and Y gadgets, Y and X with Z factors, Z strings
and phase gadgets, one-target matrices with controls, Pauli tensors, and the ops
they leave to other kernels (swap, dense gate, gadgets with two X/Y qubits).
Sizes: the first with passes (10 qubits FP64, 12 FP32), the next ones, and enough
tiles for several workgroups.
"""
import numpy as np
import pytest

from test_emu_kernels import _run, _unitary, _write_op, drive  # noqa: F401


def circuit(rng, n, layers, forms=False):
    """forms: only ops with a register-tile form (the forward sweep takes them too)"""
    ang = lambda: float(rng.uniform(0, 6.3))
    ops = []
    for layer in range(layers):
        for q in range(n - 1):
            ops.append(("pauliGadget", ([q, q + 1], [3, 3], ang())))
        for q in range(n):
            ops.append(("pauliGadget", ([q], [1 + (q + layer) % 2], ang())))
        q = [int(x) for x in rng.permutation(n)]
        ops.append(("pauliGadget", (q[:3], [1, 3, 3], ang())))
        ops.append(("pauliGadget", (q[3:6], [3, 2, 3], ang())))
        if not forms:
            ops.append(("pauliGadget", (q[:3], [1, 2, 3], ang())))
        ops.append(("oneTargGate", (q[0], _unitary(rng, 2))))
        for c in (1, 2):
            for s in range(0, n - c, 3):
                ops.append(("manyCtrlOneTargGate", (q[s + 1:s + 1 + c], q[s], _unitary(rng, 2))))
        ops.append(("pauliGadget", (q[:4], [3, 3, 3, 3], ang())))
        if layer and not forms:
            ops.append(("manyTargGate", (q[2:5], _unitary(rng, 8))))
    return ops


def observable(rng, n, terms=6):
    paulis = np.zeros((terms, n), np.uint32)
    for t in range(terms):
        w = int(rng.integers(1, 4))
        paulis[t, rng.choice(n, w, replace=False)] = rng.integers(1, 4, w)
    return rng.normal(size=terms), paulis


def oracle_adjoint(orc, psi, ops, coeffs, paulis):
    psi = psi.copy()
    for name, a in ops:
        getattr(orc, "sv_" + name)(psi, *a)
    lam = orc.sv_applyPauliSum(psi, coeffs, paulis)
    expec, phi, grads = np.vdot(psi, lam).real, psi, []
    for name, a in reversed(ops):
        if name in ("pauliGadget", "phaseGadget"):
            codes = a[1] if name == "pauliGadget" else [3] * len(a[0])
            p = phi.copy()
            orc.sv_pauliTensor(p, a[0], codes)
            grads.append(-2 * np.vdot(lam, p).imag)
            inv = a[:-1] + (-a[-1],)
        elif name in ("swapGate", "pauliTensor"):
            inv = a
        else:
            inv = a[:-1] + (a[-1].conj().T,)
        for v in (phi, lam):
            getattr(orc, "sv_" + name)(v, *inv)
    return expec, np.array(grads[::-1])


# rounding of L ops on unit vectors: L * a few eps on <H> and on the gradient's norm
@pytest.mark.parametrize("n,prec,forms,tol", [(10, 0, False, 1e-12), (12, 0, True, 1e-12), (12, 1, True, 2e-5)])
def test_sweep_passes_on_cpu(drive, orc, tmp_path, n, prec, forms, tol):  # noqa: F811
    rng = np.random.default_rng(900 + n + prec)
    ops = circuit(rng, n, 2, forms)
    coeffs, paulis = observable(rng, n)
    psi = np.zeros(1 << n, complex)
    psi[0] = 1
    expec, grads = oracle_adjoint(orc, psi, ops, coeffs, paulis)
    path = tmp_path / "sweep.bin"
    with open(path, "wb") as f:
        np.array([n, len(ops), len(coeffs)], np.uint32).tofile(f)
        for name, args in ops:
            _write_op(f, name, args)
        np.asarray(coeffs, np.float64).tofile(f)
        np.asarray(paulis, np.uint32).tofile(f)
        np.concatenate([[expec], grads]).astype(np.float64).tofile(f)
    out = _run(drive, ["adjoint", path, prec])
    assert out["expec_abs_err"] <= tol and out["grad_rel_err"] <= tol, out
    assert out["adjoint_sweep"] >= 2, out
    assert ("forward_sweep" in out) == forms, out


@pytest.mark.gpu
@pytest.mark.parametrize("forms", [False, True])
@pytest.mark.parametrize("n", [10, 11, 12, 13, 18])
def test_sweep_passes_on_gpu(orc, n, forms):
    import __graft_entry__ as ge

    fsa = ge.load_package()
    rng = np.random.default_rng(950 + n)
    ops = circuit(rng, n, 3, forms)
    if not forms:
        ops.insert(20, ("swapGate", (0, n - 1)))
    ops.insert(50, ("pauliTensor", ([1, 3, n - 1], [2, 3, 3])))
    ops.insert(70, ("pauliTensor", ([2, n - 2], [3, 3])))
    ops.insert(30, ("phaseGadget", ([0, 5, n - 2], 0.7)))
    coeffs, paulis = observable(rng, n, 12)
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    v /= np.linalg.norm(v)
    expec, grads = oracle_adjoint(orc, v, ops, coeffs, paulis)
    c = fsa.Circuit(ops)
    for prec, tol in (("fp64", 1e-12), ("fp32", 3e-6)):
        psi0 = fsa.StateVector(n, precision=prec)
        psi0.upload(v)
        fsa.profile_enable(True)
        e, g = fsa.adjoint_gradient(c, psi0, coeffs, paulis)
        launches = fsa.profile_read()
        fsa.profile_enable(False)
        if n >= (10 if prec == "fp64" else 12):
            assert launches["adjoint_sweep"][0] >= 2, launches
            assert ("forward_sweep" in launches) == forms, launches
        assert abs(e - expec) <= tol * np.abs(coeffs).sum()
        assert np.linalg.norm(g - grads) <= tol * np.linalg.norm(grads), (prec, np.linalg.norm(g - grads))
        # new angles, same passes; then the first ones again, bit for bit
        th = np.array([a[-1] for name, a in ops if name in ("pauliGadget", "phaseGadget")])
        c.set_params(th + 0.1)
        fsa.adjoint_gradient(c, psi0, coeffs, paulis)
        c.set_params(th)
        e2, g2 = fsa.adjoint_gradient(c, psi0, coeffs, paulis)
        assert e2 == e and np.array_equal(g2, g)
