"""A window that has done its [MD] steps keeps its last gradient, positions and
velocities while the engine's other windows run on, list updates among their
steps: equal bits to the window alone.  With one solvent model the forces of a
step are one launch, with two they are those of a large engine; the timing pass
launches the kernels one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHORT, LONG = 10, 60


def run(inputs, steps, timing=False):
    from q_amd.engine import Engine
    e = Engine(0)
    for p in inputs:
        e.set_log(e.add_window(p), None)
    e.prepare()
    e.set_timing(timing)
    e.run(steps, finalize=False)
    out = [e.forces(0), e.coords(0), e.velocities(0)]
    moving = e.forces(len(inputs) - 1)
    e.close()
    return out, moving


@pytest.mark.parametrize("other,timing", [("ligwat", False), ("ligtip3", False), ("ligwat", True)])
def test_gradient_of_a_stopped_window(systems, other, timing):
    short = systems("ligwat", steps=SHORT, md_seed=3)
    alone, _ = run([short], LONG)
    got, moving = run([short, systems(other, steps=LONG, md_seed=4)], 30, timing)
    assert np.abs(alone[0]).max() > 1.0 and np.abs(moving).max() > 1.0
    for a, b in zip(alone, got):
        assert np.array_equal(a, b)
