"""Energies and gradient of windows with one, three and four FEP states against
the numpy restatement of the reference.

Tolerances: energies those of the step-0 parity gates (1e-6 relative).  Gradient:
the kernels' FP32 coordinates are good to 2e-6 A, which the stiffest listed pairs
(contacts, some 500 kcal/mol/A^2) turn into 1e-3 kcal/mol/A, 1e-4 of the
gradient's RMS of 9."""
import os
import re

import numpy as np
import pytest

from tests.golden import trajectory_bits as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config,n", [("ligwat", 1), ("ligwat", 3), ("ligwat", 4), ("ligtip3", 3), ("ligarithlibq", 4)])
def test_number_of_states(systems, config, n):
    from oracle import qdyn_np as O
    from q_amd.engine import Engine
    inp = T.with_states(systems(config), n)
    e = Engine(0)
    w = e.add_window(inp)
    e.prepare()
    x = e.coords(w)
    e.evaluate(rebuild_lists=True)
    q, f = e.q_energies(w), e.forces(w)
    assert e.info(w)["nstates"] == n
    e.close()
    # the radial restraint takes the free temperature, which the log has
    tfree = float(re.search(r"Tfree =\s*([0-9.]+)", open(os.path.splitext(inp)[0] + ".log").read()).group(1))
    _, EQ, d, _ = O.evaluate(inp, x, tfree)
    for s in range(n):
        for k in range(6, 14):
            ref = EQ[s][k]
            assert abs(q[s, k] - ref) <= 1e-6 * abs(ref) + 1e-6, (s, k, q[s, k], ref)
    rms = np.sqrt((d ** 2).mean())
    print("states", n, "gradient error / RMS", np.abs(f - d).max() / rms, "RMS", rms)
    assert np.abs(f - d).max() <= 1e-4 * rms
