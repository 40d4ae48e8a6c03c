"""Which form of the Ewald k-space a system runs, at the line between them:
octants up to kmax 32 and, up to kmax 64, for systems of enough atoms (fewer in
FP64); rows elsewhere.  Told apart by the launches of an MD segment without a
thermostat: the octant form carries the half-steps between two force
evaluations in its k-space launch, the row form has them in launches of their
own.  Forces of either side against the oracle."""
import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import Ewald, LennardJones, MolecularDynamics, PairInteraction, Simulation, System, UnitCell, VelocityVerlet
from lumol_amd._native import LG_PRECISION_FP64, LG_PRECISION_MIXED

pytestmark = pytest.mark.gpu


def ions(n, kmax, seed=1):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    L = max(20.0, 2.8 * m)
    grid = np.array([(i, j, k) for i in range(m) for j in range(m) for k in range(m)], float)[:n]
    pos = (grid + 0.5 + rng.uniform(-0.2, 0.2, size=(n, 3))) * L / m
    q = np.where(np.arange(n) % 2 == 0, 1.0, -1.0) * rng.uniform(0.5, 1.0, size=n)
    s = System.from_arrays(["Ar"] * n, pos, UnitCell.cubic(L), charges=q, masses=np.full(n, 39.948),
                           velocities=rng.normal(0, 5e-3, size=(n, 3)))
    rc = min(9.0, 0.4 * L)
    s.set_pair_potential(("Ar", "Ar"), PairInteraction(LennardJones(0.5 * L / m, 1e-4), rc))
    s.set_coulomb_potential(Ewald(rc, kmax))
    return s


CASES = [(64, 16, True, True), (64, 17, True, True), (64, 24, True, True), (64, 25, True, True), (64, 32, True, True),
         (64, 33, False, False), (511, 44, False, False), (512, 44, False, True), (1279, 43, False, False),
         (1280, 43, False, True), (2047, 33, False, True),
         (2048, 33, True, True), (2048, 64, True, True), (2048, 65, False, False)]


@pytest.mark.parametrize("n,kmax,mixed,fp64", CASES)
def test_form(n, kmax, mixed, fp64):
    s = ions(n, kmax)
    fo = lo.OracleSystem(s, nthreads=16).forces()
    sim = Simulation(MolecularDynamics(VelocityVerlet(1.0)))
    start = s.positions.copy()
    for precision, octants, bar in ((LG_PRECISION_MIXED, mixed, 1e-4), (LG_PRECISION_FP64, fp64, 1e-10),
                                    (LG_PRECISION_MIXED, mixed, 1e-4)):
        s.positions = start
        s.set_precision(precision)
        assert np.abs(s.forces() - fo).max() <= bar * np.abs(fo).max()
        sim.run(s, 1)
        s.profile_begin(["integrate"])
        sim.run(s, 8)
        launches = s.profile_end()["integrate"][1]
        assert launches == (1 if octants else 9)
