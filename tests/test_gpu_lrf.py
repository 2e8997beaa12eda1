"""LRF expansions of small droplets, whose group counts lie around the build's
64 targets per block and 32 shares of the sources (fewer groups than shares
included): energy and forces of the third-order Taylor expansion against the
same sums in plain numpy.  The forces are the difference of two evaluations,
with LRF on and off (exact: the gradient is a sum of integers).

Tolerance: the engine's 1/r is good to 1e-12 and every term takes it to at
most the seventh power; 1e-9 of the largest value leaves two digits."""
import numpy as np
import pytest

from q_amd import synth

pytestmark = pytest.mark.gpu

RC = 4.5


def reference(x, q):
    """(energy, gradient): for every molecule the derivatives up to the third
    of the potential of the molecules beyond the cut-off, about its centre"""
    x = x.reshape(-1, 3, 3)
    c = x.mean(1)
    f = np.zeros_like(x)
    e = 0.0
    eye = np.eye(3)
    for g in range(len(x)):
        far = ((x[:, 0] - x[g, 0]) ** 2).sum(1) > RC * RC
        d = (x[far] - c[g]).reshape(-1, 3)
        w = np.tile(q, int(far.sum()))
        r = np.sqrt((d * d).sum(1))
        p0 = (w / r).sum()
        p1 = -(w / r ** 3) @ d
        dd = np.einsum("ni,nj->nij", d, d)
        p2 = np.einsum("n,nij->ij", 3 * w / r ** 5, dd) - (w / r ** 3).sum() * eye
        t = (np.einsum("ni,jk->nijk", d, eye) + np.einsum("nj,ik->nijk", d, eye) + np.einsum("nk,ij->nijk", d, eye))
        p3 = np.einsum("n,nijk->ijk", -3 * w / r ** 7, 5 * np.einsum("nij,nk->nijk", dd, d) - (r * r)[:, None, None, None] * t)
        for a in range(3):
            u = c[g] - x[g, a]
            v = p0 + p1 @ u + 0.5 * u @ p2 @ u
            e += 0.5 * q[a] * v
            f[g, a] = -q[a] * (p1 + p2 @ u + 0.5 * np.einsum("ijk,j,k->i", p3, u, u))
    return e, f.reshape(-1)


@pytest.mark.parametrize("radius", [6.3, 8.2, 9.3, 10.0, 12.7])
def test_lrf_of_droplets(tmp_path, radius):
    from q_amd.engine import Engine
    system = synth.water_droplet(radius, seed=int(10 * radius))
    got = []
    for lrf in (True, False):
        inp = synth.make_window("water", str(tmp_path), seed=0, system=system, tag=f"l{lrf}", lrf=lrf,
                                rc_solute=RC, rc_solvent=RC)
        e = Engine(0)
        e.set_autotune(False)
        w = e.add_window(inp)
        e.prepare()
        x = e.coords(w)
        e.evaluate(rebuild_lists=True)
        got.append((e.energies(w)["LRF"], e.forces(w)))
        e.close()
    sq = np.sqrt(332.0716)
    q = np.array([np.float32(synth.SPC_QO), np.float32(-synth.SPC_QO / 2), np.float32(-synth.SPC_QO / 2)])
    energy, grad = reference(x, (q.astype(np.float64) * sq).astype(np.float32).astype(np.float64))
    print("molecules", len(x) // 9, "LRF energy", got[0][0], energy)
    assert abs(got[0][0] - energy) <= 1e-9 * np.abs(grad).max() * len(x) / 9 + 1e-9 * abs(energy)
    assert np.abs(got[0][1] - got[1][1] - grad).max() <= 1e-9 * np.abs(grad).max() + 2e-9
