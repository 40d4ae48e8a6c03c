"""The octant form of the Ewald k-space (lumol_amd/csrc/lg_kspace.hpp) at the
edges of its tables, against the oracle at the FP64 parity bar: kmax around
the sizes where a row tile gains a step or a column tile (2, 4, 7, 8, 9, 16,
17, 31), the smallest kmax of the row form that takes over (65), boxes whose
k set is not symmetric (-kmax without +kmax on the long axes), atom counts
around the 16 of a matrix tile, and MD steps with every number of atom groups
per block."""
import ctypes

import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import Ewald, LennardJones, MolecularDynamics, PairInteraction, Simulation, System, UnitCell, VelocityVerlet
from lumol_amd._native import LG_PRECISION_FP64, LG_PRECISION_MIXED
from lumol_amd.system import BerendsenThermostat

pytestmark = pytest.mark.gpu


def ions(n, box, kmax, seed=1):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    grid = np.array([(i, j, k) for i in range(m) for j in range(m) for k in range(m)], float)[:n]
    pos = (grid + 0.5 + rng.uniform(-0.2, 0.2, size=(n, 3))) * np.array(box) / m
    q = np.where(np.arange(n) % 2 == 0, 1.0, -1.0) * rng.uniform(0.5, 1.0, size=n)
    s = System.from_arrays(["Ar"] * n, pos, UnitCell.ortho(*box), charges=q, masses=np.full(n, 39.948),
                           velocities=rng.normal(0, 5e-3, size=(n, 3)))
    rc = 0.4 * min(box)
    s.set_pair_potential(("Ar", "Ar"), PairInteraction(LennardJones(0.5 * min(box) / m, 1e-4), rc))
    s.set_coulomb_potential(Ewald(rc, kmax))
    return s


def check(s):
    o = lo.OracleSystem(s, nthreads=8)
    f, fo = s.forces(), o.forces()
    assert np.abs(f - fo).max() < 1e-10 * np.abs(fo).max()
    e, eo = s.energy_terms(), o.energy_terms()
    assert abs(e.total - eo["total"]) <= 1e-10 * abs(eo["total"])
    w, wo = s.virial(), o.virial()
    assert np.abs(w - wo).max() <= 1e-10 * np.abs(wo).max()


@pytest.mark.parametrize("kmax", [2, 4, 7, 8, 9, 16, 17, 31, 65])
def test_kmax_edges(kmax):
    check(ions(48, (20.0, 20.0, 20.0), kmax))


@pytest.mark.parametrize("box", [(20.0, 31.0, 44.0), (44.0, 20.0, 20.5), (20.0, 20.1, 60.0)])
@pytest.mark.parametrize("kmax", [3, 8, 16])
def test_unequal_axes(box, kmax):
    check(ions(100, box, kmax))


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 255])
def test_atom_counts(n):
    s = ions(n, (20.0, 20.0, 20.0), 7)
    if n == 1:  # no pair: only the k-space and self terms
        e, eo = s.energy_terms(), lo.OracleSystem(s, nthreads=1).energy_terms()
        assert abs(e.total - eo["total"]) <= 1e-10 * abs(eo["total"])
    else:
        check(s)


@pytest.mark.parametrize("width", [0, 64, 128, 192, 512])
@pytest.mark.parametrize("thermostat", [False, True])
@pytest.mark.parametrize("kmax", [4, 10, 16])
def test_md_groups(width, thermostat, kmax):
    # rho_width / 64 groups of 16 atoms per block; the reference steps against
    # the oracle, the mixed form against FP64 within its force error
    def run(precision=0):
        s = ions(300, (24.0, 24.0, 24.0), kmax)
        s.set_precision(precision)
        s.set_tuning(rho_width=width)
        md = MolecularDynamics(VelocityVerlet(1.0))
        if thermostat:
            md.set_thermostat(BerendsenThermostat(300.0, 50.0))
        Simulation(md).run(s, 6)
        return s
    s = run()
    o = lo.OracleSystem(ions(300, (24.0, 24.0, 24.0), kmax), nthreads=8)
    o.md_reset()
    o.md_run(0, 1.0, 6, *((300.0, 50.0) if thermostat else ()))
    assert np.abs(s.positions - o.positions()).max() < 1e-10
    assert np.abs(run(LG_PRECISION_MIXED).positions - s.positions).max() < 1e-6


def test_partial_sums_stay_small():
    # steps of 4096 ions at 40 k-vectors an axis: one set of partial sums of
    # rho(k) per 16 atoms would be 700 MB
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    s = ions(4096, (45.0, 45.0, 45.0), 40)
    # what does not depend on the k-vectors is allocated first
    s.set_coulomb_potential(Ewald(18.0, 2))
    md = Simulation(MolecularDynamics(VelocityVerlet(1.0)))
    md.run(s, 2)
    before = free()
    s.set_coulomb_potential(Ewald(18.0, 40))
    md.run(s, 2)
    assert before - free() < 300 << 20
    o = lo.OracleSystem(s, nthreads=16)
    f, fo = s.forces(), o.forces()
    assert np.abs(f - fo).max() < 1e-10 * np.abs(fo).max()


@pytest.mark.parametrize("width", [0, 64, 320, 512])
@pytest.mark.parametrize("kmax", [9, 16, 24, 26, 28, 32])
def test_mixed_sums_hold_32_atoms(kmax, width):
    # a lattice whose structure factors are n q at every eighth k-vector and
    # nothing between, with charges of 19 bits: sums of up to 32 of them are
    # exact in FP32 and longer ones are not.  The rest is the phases' own
    # FP32 rounding, off by a thousandth of 1e-7 of n q, squared
    g = np.array([(i, j, k) for i in range(8) for j in range(8) for k in range(8)], float) * 4.0
    e = []
    for precision in (LG_PRECISION_FP64, LG_PRECISION_MIXED):
        s = System.from_arrays(["Ar"] * 512, g, UnitCell.cubic(32.0), charges=np.full(512, 2.0 ** 19 - 1.0),
                               masses=np.ones(512))
        s.set_coulomb_potential(Ewald(9.0, kmax, 2.0))
        s.set_precision(precision)
        s.set_tuning(rho_width=width)
        e.append(s.energy_terms().coulomb_kspace)
    assert abs(e[1] - e[0]) <= 1e-11 * e[0]


def test_tables_follow_the_k_set():
    # the octant tables are kept while the k set stays: cells that scale, cells
    # that change its members, another kmax, launch shape and precision
    s = ions(300, (20.0, 24.0, 31.0), 9)

    def same(bar=1e-10):
        o = lo.OracleSystem(s, nthreads=8)
        f, fo = s.forces(), o.forces()
        assert np.abs(f - fo).max() < bar * np.abs(fo).max()
        w, wo = s.virial(), o.virial()
        assert np.abs(w - wo).max() <= bar * np.abs(wo).max()

    same()
    for box in ((20.2, 24.24, 31.31), (20.0, 24.0, 36.0), (28.0, 20.0, 20.0), (20.0, 24.0, 31.0)):
        s.cell = UnitCell.ortho(*box)
        s.cell_changed()
        same()
    for kmax in (8, 17, 9):
        s.set_coulomb_potential(Ewald(8.0, kmax))
        same()
    s.set_tuning(rho_width=64)
    same()
    s.set_precision(LG_PRECISION_MIXED)
    s.cell = UnitCell.ortho(20.2, 24.24, 31.31)
    s.cell_changed()
    same(1e-4)
