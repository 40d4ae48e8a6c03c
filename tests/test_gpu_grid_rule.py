"""The grid and list build chosen for short cutoffs (half cells with fewer
than 8 atoms give way to full cells and the direct build) at the edges of the
rule: 27 and 64 full cells, fewer than 8 atoms in a full cell, unequal axes,
the largest direct system and the one behind it, two densities.  Forces
against the lanes build on its half-cell grid (summation order: 1e-12) and
the oracle (1e-10), and a trajectory with rebuilds."""
import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import LennardJones, MolecularDynamics, PairInteraction, Simulation, System, UnitCell, VelocityVerlet

pytestmark = pytest.mark.gpu


def fluid(n, box, rc, seed=2):
    rng = np.random.default_rng([seed, n])
    box = np.array(box, float)
    m = np.ceil(box / (box.prod() / n) ** (1.0 / 3.0) - 1e-9).astype(int)
    sites = np.array([(i, j, k) for i in range(m[0]) for j in range(m[1]) for k in range(m[2])], float)
    sites = sites[np.sort(rng.permutation(len(sites))[:n])] + 0.5
    pos = sites * (box / m) + rng.uniform(-0.1, 0.1, size=(n, 3))
    s = System.from_arrays(["Ar"] * n, pos, UnitCell.ortho(*box), masses=np.full(n, 39.948),
                           velocities=rng.normal(0, 4e-3, size=(n, 3)))
    s.set_pair_potential(("Ar", "Ar"), PairInteraction(LennardJones(3.4, 1e-4), rc))
    return s


# atoms, box, cutoff, build of the rule (None: not asserted)
CASES = {
    "27-cells": (1000, (30.0, 30.0, 30.0), 9.0, 3),
    "64-cells": (1700, (42.0, 42.0, 42.0), 9.0, 3),
    "125-cells": (2500, (50.0, 50.0, 50.0), 9.0, 3),
    "sparse": (1000, (60.0, 60.0, 60.0), 9.0, None),
    "slab": (3000, (30.0, 45.0, 60.0), 9.0, 3),
    "argon-7919": (7919, (72.0, 72.0, 72.0), 8.5, 3),
    "largest": (32768, (115.6, 115.6, 115.6), 8.5, 3),
    "too-large": (32769, (115.6, 115.6, 115.6), 8.5, None),
}


@pytest.mark.parametrize("case", list(CASES))
def test_forces(case):
    n, box, rc, build = CASES[case]
    s, t = fluid(n, box, rc), fluid(n, box, rc)
    t.set_tuning(nlist_build=1)
    f, g = s.forces(), t.forces()
    if build is not None:
        assert s.tuning()["nlist_build"] == build
    scale = np.abs(g).max()
    assert np.abs(f - g).max() <= 1e-12 * scale
    assert abs(s.potential_energy() - t.potential_energy()) <= 1e-12 * abs(t.potential_energy())
    assert np.abs(f - lo.OracleSystem(s, nthreads=8).forces()).max() <= 1e-10 * scale


@pytest.mark.parametrize("case", ["64-cells", "argon-7919"])
def test_trajectory(case):
    n, box, rc, _ = CASES[case]
    out = []
    for build in (0, 1):
        s = fluid(n, box, rc)
        s.set_tuning(nlist_build=build)
        Simulation(MolecularDynamics(VelocityVerlet(2.0))).run(s, 60)
        out.append(s.positions.copy())
    assert np.abs(out[0] - out[1]).max() < 1e-8


# atoms of argon's density, cutoff, lanes per atom: by the entries of a list
# (24, 68, 193, 548 at 6, 8.5, 12, 17 A) and the lanes that fill the card
@pytest.mark.parametrize("n,rc,lanes", [(1600, 8.5, 64), (1600, 17.0, 64), (4000, 8.5, 32), (4000, 12.0, 64),
                                        (4000, 17.0, 64), (8000, 8.5, 16), (8192, 6.0, 16), (8193, 6.0, 8),
                                        (8000, 12.0, 32), (8000, 17.0, 64), (32000, 8.5, 8), (32000, 17.0, 16),
                                        (50000, 8.5, 8)])
def test_lanes_without_coulomb(n, rc, lanes):
    s = fluid(n, [(n / 0.02115) ** (1.0 / 3.0)] * 3, rc)
    assert s.tuning()["pair_lanes"] == lanes
    if n <= 8193:
        f, fo = s.forces(), lo.OracleSystem(s, nthreads=8).forces()
        assert np.abs(f - fo).max() <= 1e-10 * np.abs(fo).max()


def test_few_large_cells():
    # 36 cells: workgroups per cell up to the direct build's largest system,
    # lanes per atom above it, where a cell has one workgroup
    for n, build in ((3000, 3), (33000, 1)):
        s = fluid(n, (30.0, 30.0, 24.0), 9.0)
        assert s.tuning()["nlist_build"] == build
