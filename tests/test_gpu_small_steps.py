"""MD steps of small atomic systems in one launch, without a neighbour list
(k_small_step): against the CPU oracle's dynamics at the edges of its forms
(one block that takes the system through all steps, a wave per atom, the
largest size and the list path behind it), with both integrators, the
thermostat, Wolf charges, Harmonic pairs, a cutoff of half the box and an
infinite cell; in both precisions; and the same bits however the steps are
divided over calls."""
import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import (Harmonic, LeapFrog, LennardJones, MolecularDynamics, PairInteraction, Simulation, System, UnitCell,
                       VelocityVerlet, Wolf)
from lumol_amd._native import LG_PRECISION_MIXED
from lumol_amd.system import BerendsenThermostat

pytestmark = pytest.mark.gpu
STEPS, DT = 20, 2.0


def system(n, wolf=False, harmonic=False, half=False, infinite=False, seed=5):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    box = 4.0 * m * np.array([1.0, 1.0, 1.0] if m > 2 else [3.0, 3.1, 3.2])
    g = np.array([(i, j, k) for i in range(m) for j in range(m) for k in range(m)], float)[:n]
    pos = (g + 0.5 + rng.uniform(-0.1, 0.1, size=(n, 3))) * 4.0
    names = ["A" if i % 3 else "B" for i in range(n)]
    q = np.where(np.arange(n) % 2 == 0, 0.3, -0.3) if wolf else np.zeros(n)
    s = System.from_arrays(names, pos, UnitCell.infinite() if infinite else UnitCell.ortho(*box), charges=q,
                           masses=np.full(n, 39.948), velocities=rng.normal(0, 3e-3, size=(n, 3)))
    rc = 0.5 * box.min() if half else min(8.5, 0.45 * box.min())
    lj = LennardJones(3.4, 1e-4)
    s.set_pair_potential(("A", "A"), PairInteraction.shifted(lj, rc))
    s.set_pair_potential(("A", "B"), PairInteraction(Harmonic(1e-5, 4.0) if harmonic else lj, rc))
    s.set_pair_potential(("B", "B"), PairInteraction(lj, 0.9 * rc))
    if wolf:
        s.set_coulomb_potential(Wolf(rc))
    return s


def dynamics(leapfrog=False, T=None):
    md = MolecularDynamics((LeapFrog if leapfrog else VelocityVerlet)(DT))
    if T:
        md.set_thermostat(BerendsenThermostat(T, 50.0))
    return Simulation(md)


def check(s, mixed, leapfrog=False, T=None):
    o = lo.OracleSystem(s, nthreads=8)
    amax = np.abs(o.forces()).max() / 39.948
    o.md_reset()
    o.md_run(int(leapfrog), DT, STEPS, T if T else -1.0, 50.0)
    if mixed:
        s.set_precision(LG_PRECISION_MIXED)
    dynamics(leapfrog, T).run(s, STEPS)
    # a force error of 1e-10 (FP64) or 2e-5 (FP32 pairs) of the largest force,
    # the same way in every step, with a factor of 4 for the forces' growth
    err = 4.0 * (2e-5 if mixed else 1e-10) * amax
    t = DT * STEPS
    assert np.abs(s.positions - o.positions()).max() <= 0.5 * err * t * t + 1e-12
    assert np.abs(s.velocities - o.velocities()).max() <= err * t + 1e-14


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 95, 96, 97, 127, 255, 1023, 1024, 1025, 1535, 1536, 1537])
def test_sizes(n, mixed):
    check(system(n), mixed)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [64, 300, 1100])
@pytest.mark.parametrize("form", ["leapfrog", "thermostat", "both", "wolf", "harmonic", "half", "infinite", "wolf-infinite"])
def test_forms(form, n, mixed):
    s = system(n, wolf="wolf" in form, harmonic=form == "harmonic", half=form == "half", infinite="infinite" in form)
    check(s, mixed, form in ("leapfrog", "both"), 80.0 if form in ("thermostat", "both") else None)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("T", [None, 80.0])
@pytest.mark.parametrize("n", [50, 200, 1200])
def test_same_bits_however_divided(n, T, graph):
    out = []
    for parts in ([9], [1] * 9, [4, 5]):
        s = system(n)
        if graph:
            s.set_tuning(md_graph=2)
        sim = dynamics(T=T)
        for k in parts:
            sim.run(s, k)
        out.append((s.positions.copy(), s.velocities.copy()))
    for p, v in out[1:]:
        assert np.array_equal(p, out[0][0]) and np.array_equal(v, out[0][1])


def test_energy_after_steps():
    # the list of an evaluation before the steps is not the one after them
    s = system(500)
    s.potential_energy()
    dynamics().run(s, 199)
    o = lo.OracleSystem(s, nthreads=8)
    assert abs(s.potential_energy() - o.potential_energy()) <= 1e-10 * abs(o.potential_energy())
    assert np.abs(s.forces() - o.forces()).max() <= 1e-10 * np.abs(o.forces()).max()


@pytest.mark.parametrize("n,wolf,mixed,small", [(900, True, False, True), (901, True, False, False), (1200, True, True, True),
                                                (1201, True, True, False), (1024, False, False, True),
                                                (1536, False, True, True), (1537, False, True, False)])
def test_line_between_the_paths(n, wolf, mixed, small):
    s = system(n, wolf)
    if mixed:
        s.set_precision(LG_PRECISION_MIXED)
    sim = dynamics()
    sim.run(s, 1)
    s.profile_begin(["pairs"])
    sim.run(s, 5)
    assert (s.profile_end()["pairs"][1] == 0) == small
    if wolf:
        check(system(n, wolf), mixed)
