"""Gradient and trajectory to the last bit against committed values: the
gradient is a sum of integers whose terms do not depend on how the work is
split, so a change of the kernels' tiling or launches keeps it.  Last-bit
differences are not harmless in a trajectory: a SHAKE sweep that ends one sweep
earlier turns a quantum of 2^-32 into 1e-4 A, which grows.

No tolerance: equal bits."""
import os

import numpy as np
import pytest

from tests.golden import trajectory_bits as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def golden():
    return np.load(os.path.join(os.path.dirname(T.__file__), "trajectory_bits.npz"))


def compare(golden, name, got):
    for key, (digest, values) in got.items():
        ref = golden[f"{name}.{key}"]
        off = int((values != ref).sum())
        assert off == 0, f"{name} {key}: {off} of {len(ref)} values differ, by up to {np.abs(values - ref).max()}"
        assert digest == str(golden[f"{name}.{key}.digest"]), f"{name} {key}"


@pytest.mark.parametrize("name", [n for n, c in T.CASES.items() if c[0] == T.Q])
def test_q_sums(systems, golden, name):
    from q_amd.engine import Engine
    (got,) = T.record(Engine, [T.window(systems, name)])
    compare(golden, name, got)


@pytest.mark.parametrize("name", [n for n, c in T.CASES.items() if c[0] == T.LRF])
def test_lrf_sums(systems, golden, name):
    from q_amd.engine import Engine
    (got,) = T.record(Engine, [T.window(systems, name)])
    compare(golden, name, got)


def test_many_windows(systems, golden):
    """the launches of a large engine: two solvent models, enough groups for the
    LRF build's other form"""
    from q_amd.engine import Engine
    names = ["ligand_lrf", "tip3", "protein_lrf", "dual_lrf", "arith", "qcut"] + ["ligand_lrf"] * 8
    inputs = {n: T.window(systems, n) for n in set(names)}
    for name, got in zip(names, T.record(Engine, [inputs[n] for n in names])):
        compare(golden, name, got)


@pytest.mark.parametrize("name", [n for n, c in T.CASES.items() if c[0] == T.STATES])
def test_states(systems, golden, name):
    from q_amd.engine import Engine
    (got,) = T.record(Engine, [T.window(systems, name)])
    compare(golden, name, got)


def test_states_together(systems, golden):
    """windows of one to four states in one launch, with one solvent model and
    with two"""
    from q_amd.engine import Engine
    for names in (["one", "ligand_lrf", "three", "four"], ["four_tip3", "one", "three_protein", "ligand_lrf", "four"]):
        for name, got in zip(names, T.record(Engine, [T.window(systems, n) for n in names])):
            compare(golden, name, got)
