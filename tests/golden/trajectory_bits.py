"""What tests/test_gpu_trajectory_bits.py compares: the gradient at the start
and, after short runs, positions, velocities and gradient, of windows that
between them reach every kernel of a step.

    python tests/golden/trajectory_bits.py [TREE]

writes trajectory_bits.npz with the engine of TREE (default: this one).  The
committed file holds the values of commit 71aaec4, whose gradient is a sum of
integers formed per pair tile; every later form of the kernels keeps them.  A
window alone and among others has one set of values.
"""
import hashlib
import os
import sys

import numpy as np

STEPS = (25, 120)   # one list update; four, and the polarisation's update at step 100
EVERY = 37          # components kept as values beside the digest of all
Q, LRF = "q-atoms, no LRF", "LRF"
STATES = "numbers of states"
# name: (what it covers, configuration, input options; states other than 2)
CASES = {
    "ligand": (Q, "ligwat", dict(lrf=False)),
    "tip3": (Q, "ligtip3", dict(lrf=False)),
    "dual": (Q, "ligdual", dict(lrf=False)),          # 100 q-atoms: more than one round of chunks
    "protein": (Q, "protein", dict(lrf=False)),       # 1-4 pairs and LJ with solute atoms
    "qcut": (Q, "ligqcut", dict(lrf=False)),          # dynamic Q lists
    "arith": (Q, "ligarithlibq", dict(lrf=False)),
    "water_lrf": (LRF, "water", dict(lrf=True)),
    "ligand_lrf": (LRF, "ligwat", {}),
    "dual_lrf": (LRF, "ligdual", {}),
    "protein_lrf": (LRF, "protein", {}),
    "one": (STATES, "ligwat", dict(states=1)),
    "three": (STATES, "ligwat", dict(states=3)),
    "four": (STATES, "ligqcut", dict(states=4)),
    "four_tip3": (STATES, "ligtip3", dict(states=4)),
    "three_protein": (STATES, "protein", dict(states=3)),
}
LAMBDAS = {1: (1.0,), 3: (0.5, 0.2, 0.3), 4: (0.4, 0.3, 0.2, 0.1)}


def with_states(inp, n):
    """The window of `inp` (two states) with n: state 3 has the types and terms of
    the first and state 4 those of the second, with charges of their own"""
    folder = os.path.dirname(inp)
    text = open(inp).read().split("\n")
    k = next(i for i, l in enumerate(text) if l.startswith("fep "))
    fep = text[k].split()[1]
    text[k] = f"fep {n}_{fep}"
    k = text.index("[lambdas]") + 1
    text[k] = " ".join(f"{v:.6f}" for v in LAMBDAS[n])
    out, section = [], ""
    for line in open(os.path.join(folder, fep)):
        t = line.split()
        if line.startswith("["):
            section = t[0]
        elif t and t[0] == "states":
            line = f"states {n}\n"
        elif t and (section.startswith("[change_") or section == "[softcore]"):
            two = t[-2:]
            if section == "[change_charges]":
                mean = 0.5 * (float(two[0]) + float(two[1]))
                two += [f"{mean:.4f}", f"{0.9 * mean:.4f}"]
            else:
                two += two
            line = " ".join(t[:-2] + two[:n]) + "\n"
        out.append(line)
    with open(os.path.join(folder, f"{n}_{fep}"), "w") as f:
        f.writelines(out)
    path = os.path.join(folder, f"states{n}_{os.path.basename(inp)}")
    with open(path, "w") as f:
        f.write("\n".join(text))
    return path


def window(make, name):
    """input file of a case; make(config, seed=, **options)"""
    _, config, options = CASES[name]
    options = dict(options)
    states = options.pop("states", 2)
    inp = make(config, seed=2 if config == "protein" else 0, md_seed=7, lam=0.3, steps=100000, energy=10,
               output=100000, **options)
    return inp if states == 2 else with_states(inp, states)


def record(Engine, inputs):
    """per window: {quantity: (digest of all bytes, every EVERY-th value)}"""
    e = Engine(0)
    for p in inputs:
        e.set_log(e.add_window(p), None)
    e.prepare()
    out = [{} for _ in inputs]

    def keep(key, arrays):
        for o, a in zip(out, arrays):
            a = np.ascontiguousarray(a, np.float64) + 0.0
            o[key] = (hashlib.sha256(a.tobytes()).hexdigest(), a[::EVERY].copy())

    def all_of(get):
        return [get(w) for w in range(len(inputs))]

    e.evaluate(rebuild_lists=True)
    keep("gradient", all_of(e.forces))
    done = 0
    for n in STEPS:
        e.run(n - done, finalize=False)
        done = n
        keep(f"x{n}", all_of(e.coords))
        keep(f"v{n}", all_of(e.velocities))
        keep(f"gradient{n}", all_of(e.forces))
    e.close()
    return out


def main():
    tree = os.path.abspath(sys.argv[1]) if len(sys.argv) > 1 else os.path.dirname(os.path.dirname(os.path.dirname(
        os.path.abspath(__file__))))
    sys.path.insert(0, tree)
    import tempfile

    from q_amd import synth
    from q_amd.engine import Engine
    out = {}
    with tempfile.TemporaryDirectory() as d:
        def make(config, seed, **kw):
            builder, bkw, _ = synth.CONFIGS[config]
            return synth.make_window(config, os.path.join(d, name), seed=seed, system=builder(seed=seed, **bkw), **kw)
        for name in CASES:
            (r,) = record(Engine, [window(make, name)])
            for k, (digest, values) in r.items():
                out[f"{name}.{k}.digest"] = np.array(digest)
                out[f"{name}.{k}"] = values
            print(name, flush=True)
    np.savez_compressed(os.path.join(os.path.dirname(os.path.abspath(__file__)), "trajectory_bits.npz"), **out)


if __name__ == "__main__":
    main()
