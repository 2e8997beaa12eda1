"""A prepared engine has its pair lists and LRF expansions: queries and
evaluations that keep the lists work before any step, with the bits of an
evaluation that rebuilds them (the coordinates are the same)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("windows", [["ligwat"], ["ligwat", "ligtip3"], ["protein"], ["ligqcut"]], ids="+".join)
def test_lists_after_prepare(systems, windows):
    from q_amd.engine import Engine
    e = Engine(0)
    for c in windows:
        e.set_log(e.add_window(systems(c, seed=2 if c == "protein" else 0)), None)
    e.prepare()

    def lists():
        return [e.pairlist(w, kind) for w in range(len(windows)) for kind in range(5)]

    def values():
        e.evaluate(rebuild_lists=False)
        return [np.concatenate([e.forces(w), list(e.energies(w).values()), e.q_energies(w).ravel()])
                for w in range(len(windows))]

    prepared, first = lists(), values()
    e.evaluate(rebuild_lists=True)
    rebuilt, second = lists(), values()
    e.close()
    assert all(sum(len(p[0]) for p in prepared[5 * w:5 * w + 5]) > 0 for w in range(len(windows)))
    for a, b in zip(prepared, rebuilt):
        assert all(np.array_equal(u, v) for u, v in zip(a, b))
    for a, b in zip(first, second):
        assert np.abs(a).max() > 0 and np.array_equal(a, b)
