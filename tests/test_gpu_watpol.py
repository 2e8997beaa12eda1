"""Water polarisation with shells of different populations (a member's place
is counted by several threads, by one, or over the window's waters in memory):
energy and forces against the reference's formulas in plain numpy.  The
systems are hollow droplets, so the shells alone are populated; the forces are
the difference of two evaluations with the restraint on and off (exact: the
gradient is a sum of integers).

Tolerances: both sides evaluate the same expressions in 64 bits; 1/sin(theta)
amplifies rounding by at most 1e3 in 1e4 waters (theta > 1e-3), so 1e-6 of the
largest force and of the energy leaves three digits over that and the
fixed-point quantum."""
import math

import numpy as np
import pytest

from q_amd import synth

pytestmark = pytest.mark.gpu


def hollow_droplet(radius, thickness, seed):
    rng = np.random.default_rng(seed)
    n = int(math.ceil(radius / 3.1)) + 1
    g = np.arange(-n, n + 1) * 3.1
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    r = np.sqrt((p * p).sum(1))
    p = p[(r <= radius) & (r >= radius - thickness)]
    s = synth.System(name="hollow", radius=radius)
    half = math.radians(synth.SPC_HOH / 2)
    for q in p:
        rot = synth._rand_rot(rng)
        h = [rot @ np.array([sx * math.sin(half), math.cos(half), 0.0]) * synth.SPC_ROH for sx in (1, -1)]
        base = s.natom + 1
        s.x += [q, q + h[0], q + h[1]]
        s.iac += [synth.T_OW, synth.T_HW, synth.T_HW]
        s.crg += [synth.SPC_QO, -synth.SPC_QO / 2, -synth.SPC_QO / 2]
        s.bonds += [(base, base + 1, synth.B_OW_H), (base, base + 2, synth.B_OW_H),
                    (base + 1, base + 2, synth.B_HW_HW)]
        s.angles += [(base + 1, base, base + 2, synth.A_WAT)]
        s.cgps.append((base, [base, base + 1, base + 2]))
        s.residues.append((base, "HOH"))
        s.molecules.append(base)
    return s


def reference(x, radius):
    """(energy, gradient, members per shell); theta_corr and cstb are 0 for a
    neutral droplet before the first step"""
    x = x.reshape(-1, 3, 3)
    mu = x[:, 1] + x[:, 2] - 2 * x[:, 0]
    rm = np.sqrt((mu * mu).sum(1))
    mu = mu / rm[:, None]
    rc = np.sqrt((x[:, 0] ** 2).sum(1))
    u = x[:, 0] / rc[:, None]
    scp = np.clip((mu * u).sum(1), -1, 1)
    theta = np.arccos(scp)
    edges = [radius, radius - 0.5, radius - 1.5, radius - 3.0]
    e, grad, counts = 0.0, np.zeros_like(x), []
    for s in range(3):
        m = np.nonzero((rc > edges[s + 1]) & ((rc <= edges[s]) | (s == 0)))[0]
        counts.append(len(m))
        m = m[np.lexsort((m, theta[m]))]
        n = np.float32(len(m))
        arg = np.float32(1) + (np.float32(1) - np.float32(2) * np.arange(1, len(m) + 1, dtype=np.float32)) / n
        dth = theta[m] - np.clip(np.arccos(arg.astype(np.float64)), 0.0, math.pi)
        e += 0.5 * 20.0 * (dth * dth).sum()
        f0 = -20.0 * dth / np.maximum(np.sin(np.arccos(scp[m])), 1e-12)
        f1 = (u[m] - mu[m] * scp[m, None]) / rm[m, None]
        f2 = (mu[m] - u[m] * scp[m, None]) / rc[m, None]
        grad[m, 0] += f0[:, None] * (-2 * f1 + f2)
        grad[m, 1] += f0[:, None] * f1
        grad[m, 2] += f0[:, None] * f1
    return e, grad.reshape(-1), counts


@pytest.mark.parametrize("radius,thickness,most", [(6.0, 6.0, 64), (21.0, 4.0, 300), (30.0, 4.0, 1024),
                                                   (46.0, 4.0, 4096), (90.0, 4.0, 10000)])
def test_shell_populations(tmp_path, radius, thickness, most):
    from q_amd.engine import Engine
    system = hollow_droplet(radius, thickness, seed=int(radius))
    got = []
    for pol in (True, False):
        inp = synth.make_window("water", str(tmp_path), seed=0, system=system, tag=f"p{pol}", polarization=pol)
        e = Engine(0)
        e.set_autotune(False)
        w = e.add_window(inp)
        e.prepare()
        x = e.coords(w)
        e.evaluate(rebuild_lists=True)
        got.append((e.energies(w)["restraint.water_pol"], e.forces(w)))
        e.close()
    energy, grad, counts = reference(x, radius)
    print("members per shell", counts)
    assert 0 < max(counts) <= most and (most <= 64 or max(counts) > most // 4)
    assert got[1][0] == 0.0
    assert abs(got[0][0] - energy) <= 1e-6 * energy + 1e-6
    assert np.abs(got[0][1] - got[1][1] - grad).max() <= 1e-6 * np.abs(grad).max()
    # many windows in one engine take narrower blocks: the same bits
    inp = synth.make_window("water", str(tmp_path), seed=0, tag="many")
    e = Engine(0)
    e.set_autotune(False)
    for _ in range(25):
        e.add_window(inp)
        e.set_log(len(e.windows) - 1, None)
    e.prepare()
    e.evaluate(rebuild_lists=True)
    assert e.energies(24)["restraint.water_pol"] == got[0][0]
    assert np.array_equal(e.forces(24), got[0][1])
    e.close()
