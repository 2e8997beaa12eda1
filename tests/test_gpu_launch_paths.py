"""Several kernels hold the same device code: the one force launch of a small
engine, the two of a large one and the kernels of the timing pass.  Energies,
term by term, and gradient of several frames, and a short run, must have the
same bits from each (a window alone; beside one of another solvent model; in the
timing pass)."""
import numpy as np
import pytest

from tests.golden import trajectory_bits as T

pytestmark = pytest.mark.gpu

FRAMES = 12


def record(inputs, timing):
    from q_amd.engine import Engine
    e = Engine(0)
    for p in inputs:
        e.set_log(e.add_window(p), None)
    e.prepare()
    large = e.tuning()["us"]["rows"] > 0
    x = e.coords(0)
    out = []

    def keep():
        out.append(np.concatenate([list(e.energies(0).values()), e.q_energies(0).ravel(), e.forces(0), e.coords(0)]))

    for k in range(FRAMES):
        e.set_state(0, x=x + np.random.default_rng(k).normal(0.0, 0.02, x.shape) * (k > 0))
        e.evaluate(rebuild_lists=True)
        keep()
    e.set_state(0, x=x)
    e.set_timing(timing)
    for n in (11, 30):   # both end on an energy step
        e.run(n, finalize=False)
        keep()
    e.close()
    return out, large


@pytest.mark.parametrize("name", ["protein_lrf", "ligand_lrf", "dual_lrf", "tip3", "three", "water_lrf"])
def test_same_bits(systems, name):
    window = T.window(systems, name)
    other = T.window(systems, "ligand_lrf" if name == "tip3" else "tip3")
    alone, alone_large = record([window], False)
    beside, beside_large = record([window, other], False)
    timed, _ = record([window], True)
    assert not alone_large and beside_large
    for k, (a, b, c) in enumerate(zip(alone, beside, timed)):
        assert np.array_equal(a, b), (k, np.nonzero(a != b)[0][:8], np.abs(a - b).max())
        assert np.array_equal(a, c), (k, np.nonzero(a != c)[0][:8], np.abs(a - c).max())
