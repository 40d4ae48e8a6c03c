"""Neighbour lists whose entries name sorted places (large systems; the pair
kernels gather copies of the positions kept in that order): everything that
reads the lists, against the oracle, in both precisions and across what
changes the order or the copies: steps with rebuilds, new positions, a change
of precision, Monte Carlo moves."""
import ctypes

import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import MolecularDynamics, Simulation, VelocityVerlet
from lumol_amd import _native as nat
from lumol_amd._native import LG_PRECISION_FP64, LG_PRECISION_MIXED
from lumol_amd.workloads import lj_mc_chain, spce

pytestmark = pytest.mark.gpu
BARS = {LG_PRECISION_FP64: 1e-10, LG_PRECISION_MIXED: 1e-4}


def check(s, bar, full=True):
    o = lo.OracleSystem(s, nthreads=16)
    f, fo = s.forces(), o.forces()
    assert np.abs(f - fo).max() <= bar * np.abs(fo).max()
    if full:
        assert abs(s.potential_energy() - o.potential_energy()) <= bar * abs(o.potential_energy())
        assert np.abs(s.virial() - o.virial()).max() <= bar * np.abs(o.virial()).max()
    return o


@pytest.mark.parametrize("precision", [LG_PRECISION_FP64, LG_PRECISION_MIXED])
def test_fluid(precision):
    s, _, _ = lj_mc_chain(33000, seed=3)
    s.set_precision(precision)
    o = check(s, BARS[precision])
    if precision == LG_PRECISION_FP64:
        assert (s.pairs_within(5.0) == o.pairs_within(5.0)).all()
    # thermal steps that pass the skin, then what they left
    s.velocities = np.random.default_rng(1).normal(0, 8e-3, size=(33000, 3))
    Simulation(MolecularDynamics(VelocityVerlet(2.0))).run(s, 41)
    check(s, BARS[precision], full=False)
    # new positions in another order
    s.positions = s.positions[np.random.default_rng(2).permutation(33000)]
    check(s, BARS[precision], full=False)


def test_water_molecules():
    s = spce(nmol=11000, L=69.1, cutoff=8.0, kmax=3)
    o = check(s, 1e-10)
    w, wo = s.molecular_virial(), o.molecular_virial()
    assert np.abs(w - wo).max() <= 1e-9 * np.abs(wo).max()


def test_precision_and_moves():
    s, beta, delta = lj_mc_chain(33000, seed=4)
    for p in (LG_PRECISION_FP64, LG_PRECISION_MIXED, LG_PRECISION_FP64):
        s.set_precision(p)
        check(s, BARS[p], full=False)
        s.cache_init()
        s.mc_run(7, 0, 40, beta, delta)
        check(s, BARS[p], full=False)


@pytest.mark.parametrize("rho", [0.01, 0.2])
def test_many_cells(rho):
    # 210 000 and 11 000 cells: several passes of the cell scan, and one
    s, _, _ = lj_mc_chain(33000, seed=6, rho_star=rho)
    check(s, 1e-10, full=False)


def test_precision_change_without_allocation():
    # the evaluation that may not allocate, in each precision after the other
    # alone was evaluated
    L = nat.lib()
    for first, then in ((LG_PRECISION_MIXED, LG_PRECISION_FP64), (LG_PRECISION_FP64, LG_PRECISION_MIXED)):
        s, _, _ = lj_mc_chain(33000, seed=8)
        s.set_precision(first)
        s.potential_energy()
        h = s._sync()
        nat.check(L.lg_system_set_precision(h, then))
        t, u = nat.EnergyTerms(), nat.EnergyTerms()
        assert L.lg_potential_energy_noalloc(h, ctypes.byref(t)) == nat.LG_OK
        nat.check(L.lg_potential_energy(h, ctypes.byref(u)))
        assert [getattr(t, f) for f, _ in t._fields_] == [getattr(u, f) for f, _ in u._fields_]
        eo = lo.OracleSystem(s, nthreads=16).potential_energy()
        assert abs(t.total - eo) <= BARS[then] * abs(eo)
