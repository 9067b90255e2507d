"""The pass scheduler against a plain form of its search (no GPU needed).

The plain form scans whole lists for every seed; the library's scans stop early
and skip equal seeds, and must find the same stages: same tiles, same ops in the
same order.  Compared through the schedule dump, on mixed circuits (controls,
swaps, gadgets without targets, gates too large for a tile) at several tile sizes
and search depths.
"""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parent.parent

DRIVER = """
import sys, pickle
sys.path.insert(0, sys.argv[1])
import __graft_entry__ as ge
fsa = ge.load_package()
n, ops = pickle.load(open(sys.argv[2], 'rb'))
fsa.Circuit(ops).num_passes(n, 'fp64')
"""


def masks(name, a):
    """(mixed qubits, touched qubits, kind/size/mixed text of the dump) of an op without swaps"""
    bit = lambda qs: sum(1 << q for q in qs)
    if name == "oneTargGate":
        return 1 << a[0], 1 << a[0], "1/1"
    if name == "manyCtrlOneTargGate":
        return 1 << a[1], bit(a[0]) | 1 << a[1], "1/1"
    if name == "manyTargGate":
        return bit(a[0]), bit(a[0]), f"2/{len(a[0])}"
    if name == "phaseGadget":
        return 0, bit(a[0]), "5/0"
    xy = bit(q for q, p in zip(a[0], a[1]) if p in (1, 2))
    return xy, xy | bit(q for q, p in zip(a[0], a[1]) if p in (2, 3)), "4/0"


def plain_schedule(recs, n, m, low, seeds=16, look=16, window=256):
    lowmask, free = (1 << low) - 1, m - low
    fits = lambda r: r[3] <= 5 and bin(r[0] & ~lowmask).count("1") <= free
    def scan(lst, limit, tile):
        tk, df, bnd, ball = [], [], 0, 0
        for r in lst[:limit]:
            if fits(r) and not r[0] & ball and not r[1] & bnd and bin(tile | r[0]).count("1") <= m:
                tile |= r[0]
                tk.append(r)
            else:
                df.append(r)
                bnd |= r[0] if fits(r) else r[1]
                ball |= r[1]
        return tile, tk, df
    def seeds_of(lst, k):
        return [lowmask] + [lowmask | r[0] for r in lst if fits(r) and r[0] & ~lowmask][:k]
    out, rest = [], list(recs)
    while rest:
        if not fits(rest[0]):
            out.append("S : " + rest.pop(0)[2])
            continue
        best, seed = -1, lowmask
        s1 = seeds_of(rest, seeds)
        for s in s1 if len(s1) > 1 else []:
            _, tk, df = scan(rest, window, s)
            score = len(tk) + (max(len(scan(df, window, t)[1]) for t in seeds_of(df, look)) if look and df else 0)
            if score > best:
                best, seed = score, s
        tile, tk, rest = scan(rest, len(rest), seed)
        q = 0
        while bin(tile).count("1") < m and q < n:
            tile |= 1 << q
            q += 1
        tq = " ".join(str(q) for q in range(n) if tile >> q & 1)
        out.append(("T " if len(tk) > 1 else "S ") + tq + " : " + " ".join(r[2] for r in tk))
    return out


def unitary(rng, d):
    return np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))[0]


@pytest.mark.parametrize("seed", range(6))
@pytest.mark.parametrize("env", [{}, {"FSA_SCHED_WINDOW": "12"}, {"FSA_SCHED_LOOK": "0"}, {"FSA_SCHED_SEEDS": "0"}])
def test_stages_are_those_of_the_plain_search(tmp_path, seed, env):
    import pickle

    rng = np.random.default_rng(seed)
    n, low, m = 9 + seed, 2 + seed % 2, 6 + seed % 3
    ops = []
    for i in range(70):
        q = [int(x) for x in rng.permutation(n)]
        k = int(rng.integers(6))
        if k == 0:
            ops.append(("oneTargGate", (q[0], unitary(rng, 2))))
        elif k == 1:
            ops.append(("manyCtrlOneTargGate", (q[1:3], q[0], unitary(rng, 2))))
        elif k == 2:
            t = int(rng.integers(2, 5)) if i % 20 else 6
            ops.append(("manyTargGate", (q[:t], unitary(rng, 1 << t))))
        elif k == 3:
            ops.append(("phaseGadget", (q[:int(rng.integers(0 if seed == 5 else 1, 4))], 0.3)))
        elif k == 4:
            w = int(rng.integers(1, 4))
            ops.append(("pauliGadget", (q[:w], [int(x) for x in rng.integers(1, 4, w)], 0.2)))
        else:
            ops.append(("pauliTensor", (q[:2], [3, 3])))
    recs = []
    for name, a in ops:
        nd, touch, text = masks(name, a)
        size = len(a[0]) if name == "manyTargGate" else 1
        recs.append((nd, touch, f"{text}/{bin(nd).count('1')}", size))
    path, dump = tmp_path / "ops.pkl", tmp_path / "dump.txt"
    path.write_bytes(pickle.dumps((n, ops)))
    e = dict(os.environ, FSA_SCHEDULE_DUMP=str(dump), FSA_TILE_BITS=str(m), FSA_TILE_LOW=str(low), **env)
    subprocess.run([sys.executable, "-c", DRIVER, str(ROOT), str(path)], check=True, env=e, timeout=300)
    got = [" ".join(line.split()) for line in dump.read_text().splitlines()]
    par = {k.split("_")[-1].lower(): int(v) for k, v in env.items()}
    want = plain_schedule(recs, n, m, low, **par)
    assert got == [" ".join(w.split()) for w in want]
