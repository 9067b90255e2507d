"""Dense gates of 3-5 targets in full tiles (tile_matk_mfma), with the items that
share their passes: batched gadgets, and diagonals and dephasing applied as the
tile leaves LDS.

Sizes: one tile of either precision (12 qubits in FP64, 13 in FP32), two and
four.  Targets at the bottom, at the top and spread, so that a column block's
groups are contiguous, strided and mixed.  Tolerance, relative to the norm: an
output is a sum of 2D rounded products (D = 2^k), at most three such sums in
the three-product form, so the rounding of an op stays below 4 sqrt(2D) eps
(independent roundings), and those of the ops add up.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fsa():
    import __graft_entry__ as ge

    return ge.load_package()


def _unitary(rng, d):
    m = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    return np.linalg.qr(m)[0]


def _targets(rng, n, k, where):
    if where == "low":
        return list(range(k))
    if where == "high":
        return list(range(n - 1, n - 1 - k, -1))
    return [int(q) for q in rng.permutation(n)[:k]]


def _state(rng, n):
    v = rng.normal(size=1 << n) + 1j * rng.normal(size=1 << n)
    return v / np.linalg.norm(v)


def _eps(precision):
    return float(np.finfo(np.float64 if precision == "fp64" else np.float32).eps)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("k", [3, 4, 5])
@pytest.mark.parametrize("n", [12, 13, 14])
def test_dense_gates_in_full_tiles(fsa, orc, n, k, precision):
    rng = np.random.default_rng(100 * n + k)
    psi = fsa.StateVector(n, precision=precision, mode=1)
    psi.upload(_state(rng, n))
    ref = psi.download()
    ops = 0
    for where in ("low", "high", "spread", "spread"):
        q = _targets(rng, n, k, where)
        seq = [("manyTargGate", (q, _unitary(rng, 1 << k))),
               ("pauliGadget", ([0, 3, n - 1], [1, 3, 2], 0.7)),
               ("phaseGadget", ([1, n - 2], 0.4))]
        for name, args in seq:
            getattr(fsa, "distributed_statevector_" + name)(psi, *args)
            getattr(orc, "sv_" + name)(ref, *args)
            ops += 1
    err = np.linalg.norm(psi.download() - ref) / np.linalg.norm(ref)
    assert err <= ops * 4 * np.sqrt(2 << k) * _eps(precision), err


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_dense_gates_with_channels(fsa, orc, precision):
    """A density matrix of 2^14 elements: dense gates act on rows and columns."""
    N = 7
    rng = np.random.default_rng(7)
    rho = fsa.DensityMatrix(N, precision=precision, mode=1)
    rho.upload(_state(rng, 2 * N))
    ref = rho.download()
    ops = 0
    for t in range(4):
        q = [int(x) for x in rng.permutation(N)[:3]]
        seq = [("manyTargGate", (q, _unitary(rng, 8))), ("damping", (q[0], 0.2)),
               ("oneQubitDepolarising", (q[1], 0.1)), ("oneQubitDephasing", (q[2], 0.15))]
        for name, args in seq:
            getattr(fsa, "distributed_densitymatrix_" + name)(rho, *args)
            getattr(orc, "dm_" + name)(ref, *args)
            ops += 2
    err = np.linalg.norm(rho.download() - ref) / np.linalg.norm(ref)
    assert err <= ops * 4 * np.sqrt(16) * _eps(precision), err
