"""The q kernels at the edges of their work split: numbers of q-atoms around a
chunk's 16 and a round's 64, a solute whose other atoms are not q-atoms (1-4
pairs between the two), few and many waters per block of 64.  Energies and
gradient of the whole window against the numpy restatement of the reference.

Tolerances: those of the step-0 parity gates (energies 1e-6 relative, gradient
1e-3 of its RMS: FP32 pair terms)."""
import dataclasses
import os
import re

import numpy as np
import pytest

from q_amd import synth

pytestmark = pytest.mark.gpu


def partly_q(radius, n_heavy, n_h, nq, seed):
    """a ligand of n_heavy + n_h atoms in water whose first nq atoms are
    q-atoms (no q-bonded terms)"""
    for k in range(20):
        try:
            s = synth.ligand_in_water(radius=radius, seed=seed + 1000 * k, n_heavy=n_heavy, n_h=n_h, n_pert=2)
            break
        except RuntimeError:
            continue
    empty = {f: [] for f in ("qbonds", "qangles", "qtorsions", "qimpropers", "qbond_lib", "qangle_lib")}
    return dataclasses.replace(s, qatoms=s.qatoms[:nq], qcharges=s.qcharges[:nq], qtypes=s.qtypes[:nq],
                               qalpha=s.qalpha[:nq], **empty)


@pytest.mark.parametrize("radius,n_heavy,n_h,nq", [(10.0, 6, 4, 1), (10.0, 6, 4, 5), (12.0, 30, 20, 1), (12.0, 30, 20, 3),
                                                   (9.0, 12, 8, 16), (11.0, 12, 8, 17),
                                                   (12.0, 30, 20, 33), (12.0, 30, 20, 50)])
def test_q_atom_counts(tmp_path, radius, n_heavy, n_h, nq):
    from oracle import qdyn_np as O
    from q_amd.engine import Engine
    system = partly_q(radius, n_heavy, n_h, nq, seed=0)
    inp = synth.make_window("ligwat", str(tmp_path), seed=0, system=system, lam=0.3)
    e = Engine(0)
    w = e.add_window(inp)
    e.prepare()
    x = e.coords(w)
    e.evaluate(rebuild_lists=True)
    q, f = e.q_energies(w), e.forces(w)
    e.close()
    # the radial restraint takes the free temperature, which the log has
    tfree = float(re.search(r"Tfree =\s*([0-9.]+)", open(os.path.splitext(inp)[0] + ".log").read()).group(1))
    _, EQ, d, _ = O.evaluate(inp, x, tfree)
    names = ["qx.el", "qx.vdw", "qq.el", "qq.vdw", "qp.el", "qp.vdw", "qw.el", "qw.vdw"]
    print("q-atoms", nq, "q-solute energy", [float(EQ[s][10]) for s in range(2)])
    for s in range(2):
        for k, name in enumerate(names):
            ref = EQ[s][6 + k]
            assert abs(q[s, 6 + k] - ref) <= 1e-6 * abs(ref) + 1e-6, (s, name, q[s, 6 + k], ref)
    assert np.abs(f - d).max() <= 1e-3 * np.sqrt((d ** 2).mean())
