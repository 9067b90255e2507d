"""Batched circuits with more gradient terms in a stage than it holds (96): the
stage is run as two, three or four parts, in LDS and streamed, against the
oracle's adjoint.

Tolerances: L ops on unit vectors round to L times a few eps; an FP32 <H> and
gradient keep 3e-6 of their scale (as in test_wave_sweep.py).
"""
import numpy as np
import pytest

from test_wave_sweep import observable, oracle_adjoint

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fsa():
    import __graft_entry__ as ge

    return ge.load_package()


def _ang(rng):
    return float(rng.uniform(0, 6.3))


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 3e-6)])
@pytest.mark.parametrize("gadgets", [96, 97, 193, 300])
def test_batch_stages_of_many_gradients(fsa, orc, gadgets, prec, tol):
    rng = np.random.default_rng(gadgets)
    jobs = []
    # tiles of 2^10 amplitudes: 9 qubits stay in LDS, 13 are streamed (eight tiles)
    for n in (9, 13):
        ops = [("pauliGadget", ([q], [1], _ang(rng))) for q in range(n)]
        # Z strings: one stage whatever their qubits
        for _ in range(gadgets):
            q = [int(x) for x in rng.permutation(n)[:2]]
            ops.append(("pauliGadget", (q, [3, 3], _ang(rng))))
        coeffs, paulis = observable(rng, n, 5)
        jobs.append((n, ops, coeffs, paulis))
    b = fsa.Batch(prec)
    b.set_config(512, 10, 4)
    for n, ops, coeffs, paulis in jobs:
        b.add(fsa.Circuit(ops), n, coeffs, paulis)
    e, g = b.run()
    for j, (n, ops, coeffs, paulis) in enumerate(jobs):
        v = np.zeros(1 << n, complex)
        v[0] = 1
        expec, grads = oracle_adjoint(orc, v, ops, coeffs, paulis)
        assert abs(e[j] - expec) <= tol * np.abs(coeffs).sum()
        assert np.linalg.norm(g[j] - grads) <= tol * np.linalg.norm(grads), (n, np.linalg.norm(g[j] - grads))
    for _ in range(2):
        e2, g2 = b.run()
        assert np.array_equal(e2, e) and all(np.array_equal(x, y) for x, y in zip(g2, g))
