"""Energy sums of the FP64 pass against the oracle, at the sizes where the
number of copies of the energy words changes (one per 256 member rows of a
system), for batches, for partial wavefronts and for a subset of groups.

Tolerances: the parity bars of tests/tolerances.py; kinetic energies are FP64
per bead, rounded once to 2^-32 kJ/mol (n * 2^-32 absolute)."""
import sys

import numpy as np
import pytest

from opencafemol_amd import abi, configs
from opencafemol_amd.context import Batch
from tests.tolerances import assert_energies_close

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-case] {request.node.nodeid}\n")
    sys.__stderr__.flush()
    yield


# (chains of 65 beads, systems): 65, 455, 585, 1,170 and 2,340 beads, 30% of
# them in the charged group too
@pytest.mark.parametrize("chains,systems", [(1, 1), (7, 1), (9, 3), (18, 1), (36, 2)])
def test_energy_sums_over_copies(oracle, chains, systems):
    sys_, integ, pos, vel = [], [], [], []
    for k in range(systems):
        s, it, x = configs.hps_slab(n_chains=chains, chain_len=65, box=(9.0, 9.0, 40.0), slab_z=12.0, seed=k)
        rng = np.random.default_rng(k)
        sys_.append(s)
        integ.append(it)
        pos.append(x + rng.normal(scale=0.01, size=x.shape))
        vel.append(rng.normal(scale=0.15, size=x.shape))
    with Batch(sys_, integ) as b:
        for k in range(systems):
            b.set_positions(k, pos[k])
            b.set_velocities(k, vel[k])
        for k in range(systems):
            for groups in (0xFFFFFFFF, 0b101):
                st = b.state(k, abi.STATE_ENERGY, groups)
                _, eo = oracle.evaluate(sys_[k], pos[k], groups)
                assert_energies_close(st["energy_by_group"], eo)
                ke = 0.5 * np.sum(np.asarray(sys_[k].masses)[:, None] * vel[k] ** 2)
                assert abs(st["kinetic"] - ke) <= sys_[k].n * 2.0 ** -32 + 1e-14 * ke
