"""State reads that need the standard path's lists after steps that made the
rows outgrow their slots: 600 beads without bonds start 3 nm apart, where a row
has a few partners and the slots of the estimate (264 for an open group of 256
beads or more), and fall into a cube of 1.6 nm, where every row has 599.
Resident steps do not widen the standard path's rows, so the read does.  Also
the reads that keep a list between them.  The oracle is the reference."""
import ctypes as C
import sys

import numpy as np
import pytest

from opencafemol_amd import abi, configs
from opencafemol_amd.context import Context
from opencafemol_amd.model import ForceSpec, IntegratorSpec, SystemSpec
from tests.tolerances import assert_energies_close, assert_forces_close

pytestmark = pytest.mark.gpu

STEPS, DT = 200, 0.01
PAIRS, CHARGES, ALL = 1, 2, 0xFFFFFFFF   # group masks


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-case] {request.node.nodeid}\n")
    sys.__stderr__.flush()
    yield


def _falling():
    g = np.stack(np.meshgrid(np.arange(10), np.arange(10), np.arange(6), indexing="ij"), -1).reshape(-1, 3)
    x = 3.0 * g + np.random.default_rng(3).uniform(-0.3, 0.3, size=(600, 3))
    n = len(x)
    s = SystemSpec(masses=np.full(n, 1000.0))
    s.add(ForceSpec(abi.EXCLUDED_VOLUME, "ExcludedVolume", particle_params=np.full((n, 1), 0.04),
                    globals=np.array([0.5]), cutoff=0.3))
    q = np.where(np.arange(n) % 2 == 0, 0.1, -0.1).reshape(n, 1)
    s.add(ForceSpec(abi.DEBYE_HUCKEL, "DebyeHuckel", particle_params=q, globals=np.array([1.8, 0.8, 0.05]), cutoff=2.5))
    # no friction and no noise: straight lines to 6% of the start's extent
    v = -(x - x.mean(axis=0)) * (0.94 / (STEPS * DT))
    return s, IntegratorSpec(0.0, 0.0, DT, 1), x, v


def _fallen():
    s, it, x, v = _falling()
    c = Context(s, it)
    assert c.resident_threads() == 1024
    c.set_positions(x)
    c.set_velocities(v)
    assert c.step(STEPS) == abi.OCM_OK
    return s, c


def _check(oracle, s, c, st, groups):
    # the positions do not move between reads
    x = c.get_state(abi.STATE_POSITIONS)["positions"]
    assert np.ptp(x, axis=0).max() < 2.0   # every pair within the cutoff and skin
    F, E = oracle.evaluate(s, x, groups)
    if "forces" in st:
        assert_forces_close(st["forces"], F)
    if "potential" in st:
        assert_energies_close(st["energy_by_group"], E)


@pytest.mark.parametrize("groups", [PAIRS, CHARGES, PAIRS | CHARGES])
def test_forces_and_energies_when_rows_overflow(oracle, groups):
    s, c = _fallen()
    with c:
        _check(oracle, s, c, c.get_state(abi.STATE_FORCES | abi.STATE_ENERGY, groups), groups)
        _check(oracle, s, c, c.get_state(abi.STATE_FORCES, CHARGES), CHARGES)


@pytest.mark.parametrize("groups", [PAIRS, CHARGES])
def test_forces_alone_when_rows_overflow(oracle, groups):
    s, c = _fallen()
    with c:
        for _ in range(2):   # the second read reuses the list of the first
            _check(oracle, s, c, c.get_state(abi.STATE_FORCES, groups), groups)


@pytest.mark.parametrize("groups", [PAIRS, CHARGES])
def test_forces_after_a_refused_noalloc_dump(oracle, groups):
    """The dump that does not widen rows refuses and leaves a truncated list."""
    s, c = _fallen()
    with c:
        count = C.c_int64(-1)
        for k in (0, 1):
            assert c.lib.ocm_get_neighbor_pairs_noalloc(c.h, k, None, 0, C.byref(count)) == abi.OCM_ERR_OOM
        _check(oracle, s, c, c.get_state(abi.STATE_FORCES, groups), groups)
        assert c.lib.ocm_get_neighbor_pairs_noalloc(c.h, 0, None, 0, C.byref(count)) == abi.OCM_OK


@pytest.mark.parametrize("resident", [-1, 0])
def test_reads_that_keep_a_list_between_them(oracle, resident):
    """Energies build a list after steps, a subset's forces and energies after
    them keep it, and new positions or further steps end it."""
    s, it, x = configs.go_chain(120, seed=9)
    rng = np.random.default_rng(2)
    with Context(s, it, resident=resident) as c:
        c.set_positions(x)
        c.set_velocities(rng.normal(scale=0.3, size=x.shape))
        sub = 1 << s.forces[-1].group
        for new in (None, x + rng.normal(scale=0.02, size=x.shape), None, 3.0 * x):
            if new is None:
                assert c.step(150) == abi.OCM_OK
            else:
                c.set_positions(new)
            for what, groups in ((abi.STATE_ENERGY, ALL), (abi.STATE_FORCES, sub), (abi.STATE_ENERGY, sub),
                                 (abi.STATE_FORCES | abi.STATE_ENERGY, ALL)):
                st = c.get_state(what | abi.STATE_POSITIONS, groups)
                F, E = oracle.evaluate(s, st["positions"], groups)
                if what & abi.STATE_FORCES:
                    assert_forces_close(st["forces"], F)
                if what & abi.STATE_ENERGY:
                    assert_energies_close(st["energy_by_group"], E)
