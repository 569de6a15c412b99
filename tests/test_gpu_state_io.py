"""Positions and velocities set and read back, bit for bit, around the size
where a state stops going through the pinned staging (131,072 values over the
arrays of one read: 21,845 beads with positions and velocities, 43,690 with
one array), from a batch's second system, and between steps."""
import sys

import numpy as np
import pytest

from opencafemol_amd import abi
from opencafemol_amd.context import Batch
from opencafemol_amd.model import ForceSpec, IntegratorSpec, SystemSpec

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-case] {request.node.nodeid}\n")
    sys.__stderr__.flush()
    yield


def _bonded(n):
    """n fixed beads, neighbours joined by bonds of 0.4 nm."""
    s = SystemSpec(masses=np.zeros(n))
    if n > 1:
        idx = np.stack([np.arange(n - 1), np.arange(1, n)], 1).astype(np.int32)
        s.add(ForceSpec(abi.HARMONIC_BOND, "HarmonicBond", indices=idx, params=np.tile([0.4, 1000.0], (n - 1, 1))))
    return s


@pytest.mark.parametrize("n", [1, 85, 86, 14563, 14564, 21845, 21846, 43690, 43691])
def test_state_round_trip(n):
    rng = np.random.default_rng(n)
    it = IntegratorSpec(300.0, 0.5, 0.01, seed=n)
    with Batch([_bonded(7), _bonded(n)], [it, it]) as b:
        x = np.cumsum(np.tile([[0.3, 0.2, 0.1]], (n, 1)), axis=0) + rng.normal(scale=0.01, size=(n, 3))
        v = rng.normal(size=(n, 3))
        b.set_positions(0, np.arange(21.0).reshape(7, 3))
        b.set_positions(1, x)
        b.set_velocities(1, v)
        st = b.state(1, abi.STATE_POSITIONS | abi.STATE_VELOCITIES)
        assert np.array_equal(st["positions"], x) and np.array_equal(st["velocities"], v)
        b.step(3)   # fixed beads keep their state
        st = b.state(1, abi.STATE_POSITIONS | abi.STATE_VELOCITIES | abi.STATE_FORCES | abi.STATE_ENERGY)
        assert np.array_equal(st["positions"], x) and np.array_equal(st["velocities"], v)
        assert st["step"] == 3 and st["kinetic"] == 0.0
        one = b.state(1, abi.STATE_FORCES)["forces"]
        assert np.array_equal(one, st["forces"])
        if n > 1:   # the bonds' forces and energy in FP64
            d = x[1:] - x[:-1]
            r = np.linalg.norm(d, axis=1)
            g = (1000.0 * (r - 0.4) / r)[:, None] * d
            f = np.zeros((n, 3))
            f[:-1] += g
            f[1:] -= g
            # FP32 term arithmetic: ~1e-6 of the largest bond force, 2^-32 fixed point
            assert np.abs(one - f).max() <= 4e-6 * np.abs(g).max() + 1e-9
            assert abs(st["potential"] - 500.0 * np.sum((r - 0.4) ** 2)) <= 1e-9 * st["potential"] + n * 2.0 ** -32
        assert np.array_equal(b.state(0, abi.STATE_POSITIONS)["positions"], np.arange(21.0).reshape(7, 3))
