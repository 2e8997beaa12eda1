"""Engines of many windows, or of windows with different solvent models, run
their forces as the launches of a large engine, one window alone as a single
launch.  A window's trajectory and energies must be the same bits either way:
its sums do not depend on how the work is launched.  30 steps with one list
update and energy steps between; the window counts lie on both sides of the
change of the polarisation's block size, and the arithmetic combining rule and
1-4 pairs are among the windows."""
import numpy as np
import pytest

from q_amd import synth

pytestmark = pytest.mark.gpu

STEPS = 30


def run(tmp_path, windows):
    from q_amd.engine import Engine
    e = Engine(0)
    for cfg, k in windows:
        w = e.add_window(synth.make_window(cfg, str(tmp_path / cfg), seed=0, md_seed=1 + k, lam=0.25 * k, steps=1000,
                                           energy=10, output=10, nb_cycle=25, tag=f"w{k}"))
        e.set_log(w, None)
    e.prepare()
    e.run(STEPS, finalize=False)
    out = [(e.coords(w), e.velocities(w), e.forces(w), e.energies(w)) for w in range(len(windows))]
    e.evaluate(rebuild_lists=True)
    out = [o + (e.forces(w), e.energies(w)) for w, o in enumerate(out)]
    large = e.tuning()["us"]["rows"] > 0
    e.close()
    return out, large


@pytest.mark.parametrize("windows", [[("ligwat", 0), ("ligtip3", 1)],
                                     [("ligwat", 0), ("ligtip3", 1)] + [("ligarithlibq", 2)] * 11,
                                     [("ligwat", k % 4) for k in range(40)]],
                         ids=["two-solvents", "thirteen-windows", "forty-windows"])
def test_windows_alone_and_together(tmp_path, windows):
    got, large = run(tmp_path, windows)
    assert large
    for spec in sorted(set(windows)):
        (alone,), alone_large = run(tmp_path, [spec])
        assert not alone_large
        for w, s in enumerate(windows):
            if s != spec:
                continue
            for a, b in zip(alone, got[w]):
                if isinstance(a, dict):
                    assert a == b
                else:
                    assert np.array_equal(a, b)
