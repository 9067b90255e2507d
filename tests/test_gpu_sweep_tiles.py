"""Register-tile passes (wave_sweep.hpp) and H psi in which a wave or workgroup
takes more than one piece of work, against the oracle's adjoint.

24 qubits: 2^14 (FP64) and 2^13 (FP32) forward tiles for at most 4096 waves, 2^15
and 2^14 reverse tiles for at most 3072.  A wave adds its tiles' gradient terms
up, the last term of a pass of an odd number of gadgets without a partner.
Tolerances as in test_wave_sweep.py.
"""
import numpy as np
import pytest

from test_emu_kernels import _unitary
from test_wave_sweep import observable, oracle_adjoint

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gadgets", [1, 8, 13])
def test_waves_of_several_tiles(orc, gadgets):
    import __graft_entry__ as ge

    fsa = ge.load_package()
    n = 24
    rng = np.random.default_rng(gadgets)
    ops = []
    for g in range(gadgets):
        # qubits that one tile can hold, and Z factors anywhere
        q = [int(x) for x in rng.permutation(n)[:2]]
        if g % 3 == 0:
            ops.append(("pauliGadget", (q, [3, 3], float(rng.uniform(0, 6.3)))))
        else:
            low = (3 * g) % 8
            ops.append(("pauliGadget", ([low, 12 + q[0] % 12], [g % 3, 3], float(rng.uniform(0, 6.3)))))
    ops.insert(len(ops) // 2, ("manyCtrlOneTargGate", ([n - 1], 4, _unitary(rng, 2))))
    ops.append(("oneTargGate", (5, _unitary(rng, 2))))
    coeffs, paulis = observable(rng, n, 3)
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
        assert launches["adjoint_sweep"][0] >= 1 and launches["forward_sweep"][0] >= 1, launches
        assert abs(e - expec) <= tol * np.abs(coeffs).sum()
        # an FP32 gradient is as far off as its state: relative to sum |c|, which bounds each term
        assert np.linalg.norm(g - grads) <= tol * max(np.linalg.norm(grads), np.abs(coeffs).sum()), prec
        e2, g2 = fsa.adjoint_gradient(c, psi0, coeffs, paulis)
        assert e2 == e and np.array_equal(g2, g)
        psi0.close()
