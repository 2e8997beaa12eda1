"""The water polarisation's blocks of each launch: 512 threads in the one launch
of a small engine, 256 in those of a large one (a second solvent model makes it
large), 1024 where a shell has more waters than a block holds.  The same bits
from the first two; the third takes large engines' launches by itself, and its
values against the formulas are in test_gpu_watpol.py."""
import numpy as np
import pytest

from q_amd import synth
from tests.test_gpu_watpol import hollow_droplet

pytestmark = pytest.mark.gpu


def evaluate(inputs):
    from q_amd.engine import Engine
    e = Engine(0)
    for p in inputs:
        e.set_log(e.add_window(p), None)
    e.prepare()
    e.evaluate(rebuild_lists=True)
    out = e.energies(0)["restraint.water_pol"], e.forces(0)
    large = e.tuning()["us"]["rows"] > 0   # only a large engine's launches are timed
    e.close()
    return out, large


@pytest.mark.parametrize("radius,thickness", [(6.0, 6.0), (21.0, 4.0), (30.0, 4.0), (46.0, 4.0)])
def test_block_sizes(systems, tmp_path, radius, thickness):
    inp = synth.make_window("water", str(tmp_path), seed=0, system=hollow_droplet(radius, thickness, seed=int(radius)))
    alone, alone_large = evaluate([inp])
    other, other_large = evaluate([inp, systems("ligtip3")])
    assert not alone_large and other_large
    assert alone[0] > 0 and alone[0] == other[0]
    assert np.array_equal(alone[1], other[1])


def test_shells_in_memory(tmp_path):
    inp = synth.make_window("water", str(tmp_path), seed=0, system=hollow_droplet(90.0, 4.0, seed=90))
    (energy, _), large = evaluate([inp])
    assert energy > 0 and large
