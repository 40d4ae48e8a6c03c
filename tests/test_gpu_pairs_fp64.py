"""The FP64 pair kernel where its shortcuts could differ from the reference's
order: pairs at exactly the cutoff (`r < rc` for pairs, `r <= rc` for Coulomb,
tested on r^2), components at exactly half the box when the cutoff reaches it
(the checked minimum image), an alpha whose tables miss their bound (library
erfc), and Harmonic pair terms beside Lennard-Jones.  Oracle at the FP64
parity bar, relative to the largest force."""
import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import Ewald, Harmonic, LennardJones, PairInteraction, System, UnitCell, Wolf

pytestmark = pytest.mark.gpu


def system(box, rc, coulomb, pos, harmonic=False):
    n = len(pos)
    names = ["A" if i % 3 else "B" for i in range(n)]
    q = np.where(np.arange(n) % 2 == 0, 0.8, -0.8)
    s = System.from_arrays(names, pos, UnitCell.ortho(*box), charges=q, masses=np.full(n, 20.0))
    lj = LennardJones(2.0, 1e-4)
    s.set_pair_potential(("A", "A"), PairInteraction.shifted(lj, rc))
    s.set_pair_potential(("A", "B"), PairInteraction(Harmonic(1e-4, 4.0) if harmonic else lj, rc))
    s.set_pair_potential(("B", "B"), PairInteraction(lj, 0.8 * rc))
    if coulomb is not None:
        s.set_coulomb_potential(coulomb)
    return s


def check(s):
    o = lo.OracleSystem(s, nthreads=4)
    f, fo = s.forces(), o.forces()
    assert np.abs(f - fo).max() < 1e-10 * np.abs(fo).max()
    e, eo = s.energy_terms(), o.energy_terms()
    scale = max(abs(eo[k]) for k in ("pairs", "coulomb", "total"))
    assert abs(e.pairs - eo["pairs"]) <= 1e-10 * scale
    assert abs(e.coulomb - eo["coulomb"]) <= 1e-10 * scale
    w, wo = s.virial(), o.virial()
    assert np.abs(w - wo).max() <= 1e-10 * np.abs(wo).max()


def lattice(box, m, seed=0, jitter=0.0):
    g = np.array([(i, j, k) for i in range(m) for j in range(m) for k in range(m)], float)
    return g * np.array(box) / m + np.random.default_rng(seed).uniform(-jitter, jitter, size=(m ** 3, 3))


COULOMB = {"none": lambda rc: None, "ewald": lambda rc: Ewald(rc, 5), "wolf": Wolf}


@pytest.mark.parametrize("kind", list(COULOMB))
def test_pairs_at_the_cutoff(kind):
    # 3-4-5 triangles: distances of exactly 5 between many pairs
    pos = np.array([(x, y, z) for x in (0, 3, 6) for y in (0, 4, 8) for z in (0, 6, 12)], float)
    check(system((20.0, 20.0, 20.0), 5.0, COULOMB[kind](5.0), pos))


@pytest.mark.parametrize("kind", list(COULOMB))
@pytest.mark.parametrize("jitter", [0.0, 1e-12, 0.05])
def test_cutoff_of_half_the_box(kind, jitter):
    # sites at exactly (or within rounding of) half the box from each other
    box = (12.0, 12.0, 14.0)
    check(system(box, 6.0, COULOMB[kind](6.0), lattice(box, 4, jitter=jitter) + 0.1))


@pytest.mark.parametrize("alpha", [0.4, 1.5, 4.0])
def test_alpha_beyond_the_tables(alpha):
    box = (20.0, 20.0, 20.0)
    check(system(box, 9.0, Ewald(9.0, 6, alpha), lattice(box, 6, jitter=0.4)))


@pytest.mark.parametrize("kind", list(COULOMB))
@pytest.mark.parametrize("box", [(20.0, 20.0, 20.0), (18.5, 24.0, 31.0)])
def test_harmonic_beside_lennard_jones(kind, box):
    check(system(box, 8.0, COULOMB[kind](8.0), lattice(box, 6, jitter=0.4), harmonic=True))
