"""Resident steps around the sizes where the step's units of 64 items change:
chains whose term counts fill a unit exactly, miss it or pass it by one, and
systems with bonded terms only, pairs only or neither.  The standard path is
the reference; both sum the same fixed-point words, so the states are equal
bit for bit (no tolerance)."""
import sys

import numpy as np
import pytest

from opencafemol_amd import abi, configs
from opencafemol_amd.context import Batch, Context
from opencafemol_amd.model import SystemSpec

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-case] {request.node.nodeid}\n")
    sys.__stderr__.flush()
    yield


def _both(s, it, x, steps):
    v = np.random.default_rng(1).normal(scale=0.1, size=x.shape)
    got = []
    for resident in (-1, 0):
        with Context(s, it, resident=resident) as c:
            assert (c.resident_threads() > 0) == (resident != 0)
            c.set_positions(x)
            c.set_velocities(v)
            for n in steps if isinstance(steps, tuple) else (steps,):
                assert c.step(n) == 0
            st = c.get_state(abi.STATE_POSITIONS | abi.STATE_VELOCITIES | abi.STATE_FORCES)
            got.append((st["positions"], st["velocities"], st["forces"], st["step"]))
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [5, 64, 65, 66, 67, 68, 129, 130, 131, 450, 1024])
def test_go_chain_unit_edges(n):
    s, it, x = configs.go_chain(n, seed=n)
    _both(s, it, x, 60)


def _only(s, keep):
    out = SystemSpec(masses=s.masses, box=s.box)
    for f in s.forces:
        if keep(f):
            out.add(f)
    return out


@pytest.mark.parametrize("n", [70, 300])
@pytest.mark.parametrize("what", ["bonded", "pairs", "none", "one pair group"])
def test_partial_sequences(what, n):
    """300 beads: the size that keeps two-level lists where it has pair groups."""
    s, it, x = configs.go_chain(n, seed=4)
    keep = {"bonded": lambda f: f.kind < abi.EXCLUDED_VOLUME, "pairs": lambda f: f.kind >= abi.EXCLUDED_VOLUME,
            "none": lambda f: False, "one pair group": lambda f: f.kind == abi.DEBYE_HUCKEL}[what]
    _both(_only(s, keep), it, x, 40)


def test_bonded_only_beside_pairs():
    """Without pair groups beside a system that has them: beads move past the
    batch's prune margin, and there is no list to prune."""
    made = [configs.go_chain(300, seed=6), configs.go_chain(300, seed=7)]
    made[0] = (_only(made[0][0], lambda f: f.kind < abi.EXCLUDED_VOLUME),) + made[0][1:]
    got = []
    for resident in (-1, 0):
        with Batch([m[0] for m in made], [m[1] for m in made], resident=resident) as b:
            assert (b.resident_threads() > 0) == (resident != 0)
            for k, (s, it, x) in enumerate(made):
                b.set_positions(k, x)
                b.set_velocities(k, np.random.default_rng(k).normal(scale=0.3, size=x.shape))
            for steps in (1, 60, 7):
                assert b.step(steps) == 0
            got.append([b.state(k, abi.STATE_POSITIONS | abi.STATE_VELOCITIES | abi.STATE_FORCES) for k in (0, 1)])
    for a, b in zip(*got):
        for key in ("positions", "velocities", "forces"):
            assert np.array_equal(a[key], b[key])


def test_open_hps_chain():
    """Open Ashbaugh-Hatch and Debye-Hueckel groups (their own row loops)."""
    s, it, x = configs.hps_open_cluster(6, 100, extent=(5.0, 5.0), seed=2)
    x = x + np.random.default_rng(0).normal(scale=0.005, size=x.shape)
    _both(s, it, x, 5)


@pytest.mark.parametrize("what", ["cluster", "slab", "lipids"])
def test_pruned_lists_past_the_lds(what):
    """Dense systems whose pruned lists pass the LDS list (16,384 entries at
    most): open Ashbaugh-Hatch and Debye-Hueckel groups, the periodic ones, and
    four groups of the membrane kinds; calls of several lengths."""
    s, it, x = {"cluster": lambda: configs.hps_open_cluster(7, 140, extent=(5.0, 5.0), seed=1),
                "slab": lambda: configs.hps_slab(n_chains=10, chain_len=100, box=(8.0, 8.0, 60.0), slab_z=15.0, seed=1),
                "lipids": lambda: configs.lipid_patch(216, box=(6.0, 6.0, 9.0), spacing=1.0, seed=1)}[what]()
    with Context(s, it) as c:
        c.set_positions(x + np.random.default_rng(0).normal(scale=0.005, size=x.shape))
        c.minimize(50.0, 200)
        x = c.get_state(abi.STATE_POSITIONS)["positions"]
    for steps in ((80,), (1, 30, 49)):
        _both(s, it, x, steps)


@pytest.mark.parametrize("n", [640, 704, 1000])
def test_more_systems_than_cus_with_a_large_one(n):
    """Beyond one workgroup per CU half the LDS is the limit, and a system that
    needs more than half takes a CU for itself: it stays resident."""
    made = [configs.go_chain(n, seed=2)] + [configs.go_chain(5, seed=3)] * 256
    got = []
    for resident in (-1, 0):
        with Batch([m[0] for m in made], [m[1] for m in made], resident=resident) as b:
            assert (b.resident_threads() > 0) == (resident != 0)
            for k, (s, it, x) in enumerate(made):
                b.set_positions(k, x)
                b.set_velocities(k, np.random.default_rng(k).normal(scale=0.1, size=x.shape))
            assert b.step(40) == 0
            got.append([b.state(k, abi.STATE_POSITIONS | abi.STATE_VELOCITIES | abi.STATE_FORCES) for k in (0, 1, 256)])
    for a, b in zip(*got):
        for key in ("positions", "velocities", "forces"):
            assert np.array_equal(a[key], b[key])


@pytest.mark.parametrize("count", [23, 24])
def test_exclusion_tables_that_do_not_fit(count):
    """1,000 beads with six exclusions beyond the mask bits for each bead and
    nonbonded force: the tables do not fit the LDS, and batches of 24 systems
    and more read them from memory (fewer step on the standard path)."""
    s, it, x = configs.go_chain(1000, seed=3)
    i = np.arange(960)
    far = np.concatenate([np.stack([i, i + 34 + k], 1) for k in range(6)]).astype(np.int32)
    for f in s.forces:
        if f.kind >= abi.EXCLUDED_VOLUME:
            f.category, f.n_categories = np.zeros(s.n, np.int32), 1   # every bead takes part
            f.exclusions = np.concatenate([np.asarray(f.exclusions, np.int32).reshape(-1, 2), far])
    got = []
    for resident in (-1, 0):
        with Batch([s] * count, [it] * count, resident=resident) as b:
            assert (b.resident_threads() > 0) == (resident != 0 and count >= 24)
            for k in range(count):
                b.set_positions(k, x)
                b.set_velocities(k, np.random.default_rng(k).normal(scale=0.1, size=x.shape))
            assert b.step(60) == 0
            got.append([b.state(k, abi.STATE_POSITIONS | abi.STATE_VELOCITIES | abi.STATE_FORCES) for k in (0, count - 1)])
    for a, b in zip(*got):
        for key in ("positions", "velocities", "forces"):
            assert np.array_equal(a[key], b[key])
