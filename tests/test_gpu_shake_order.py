"""SHAKE of three-atom molecules whose constraints come in every order and
orientation (48 ways), and of molecules with two constraints only: positions
and velocities after one step against the leapfrog and the Gauss-Seidel sweeps
in plain numpy, from the engine's own gradient.

Tolerance: both sides do the same double-precision operations up to fused
products, on coordinates below 20; 1e-10 is a thousand times their rounding."""
import itertools

import numpy as np
import pytest

from q_amd import synth

pytestmark = pytest.mark.gpu

DT = float(np.float32(0.020462))   # of a 1 fs step
WAYS = [(o, f) for o in itertools.permutations(range(3)) for f in itertools.product((0, 1), repeat=3)]


def shake(xx, x, bonds, d2, winv):
    ready = [False] * len(bonds)
    while not all(ready):
        for c, (i, j) in enumerate(bonds):
            if ready[c]:
                continue
            xij, oij = x[i] - x[j], xx[i] - xx[j]
            diff = d2[c] - xij @ xij
            ready[c] = abs(diff) < float(np.float32(1e-4)) * d2[c]
            corr = diff / (2.0 * (xij @ oij) * float(np.float32(winv[i] + winv[j])))
            x[i] = x[i] + oij * corr * float(winv[i])
            x[j] = x[j] - oij * corr * float(winv[j])


@pytest.mark.parametrize("radius", [6.0, 15.0])
def test_constraint_orders(tmp_path, radius):
    from q_amd.engine import Engine
    s = synth.water_droplet(radius, seed=1)
    n = len(s.bonds) // 3
    bonds = []
    for m in range(n):
        order, flip = WAYS[m % 48]
        b = [s.bonds[3 * m + k] for k in order]
        b = [(j, i, c) if f else (i, j, c) for (i, j, c), f in zip(b, flip)]
        bonds += b[:2] if m % 7 == 6 else b
    s.bonds = bonds
    inp = synth.make_window("water", str(tmp_path), seed=0, system=s, bath_coupling=1e15, steps=100, energy=1000,
                            output=1000)
    e = Engine(0)
    w = e.add_window(inp)
    e.set_log(w, None)
    e.prepare()
    x0, v0 = e.coords(w).reshape(-1, 3).copy(), e.velocities(w).reshape(-1, 3).copy()
    e.run(1, finalize=False)
    g = e.forces(w).reshape(-1, 3)
    mass = np.array([round(synth.LJ_TYPES[k - 1][3], 4) for k in s.iac])
    winv = np.float32(1.0 / mass)
    x = x0 + (v0 - g * winv[:, None].astype(float) * DT) * DT
    by = [[] for _ in range(n)]
    for i, j, c in s.bonds:
        by[(i - 1) // 3].append((i - 1, j - 1, round(s.bond_lib[c - 1][1], 5) ** 2))
    for b in by:
        shake(x0, x, [p[:2] for p in b], [p[2] for p in b], winv)
    assert np.abs(e.coords(w).reshape(-1, 3) - x).max() <= 1e-10
    assert np.abs(e.velocities(w).reshape(-1, 3) - (x - x0) / DT).max() <= 1e-10 / DT
    e.close()
