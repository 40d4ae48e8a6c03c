"""Monte Carlo chains of single Lennard-Jones sites with the chain's state in
LDS (k_mc_atoms), against the oracle: decisions, accepted counts and final
positions identical, the running energy to 1e-10.  At the edges of the
kernel's forms: fewer atoms than a wave, around one and two passes of the
block and of its unrolled test, the last size that fits the LDS and the other
kernel behind it, unequal axes, two kinds with a Null pair, an infinite cell,
a cutoff of half the box (the other kernel), launches that end within a batch
of draws, and moves as long as the box."""
import numpy as np
import pytest

import lumol_oracle as lo
from lumol_amd import K_BOLTZMANN, LennardJones, NullPotential, PairInteraction, System, UnitCell

pytestmark = pytest.mark.gpu
SIGMA, EPS = 3.405, 9.96e-5


def chain(n, box=None, kinds=1, infinite=False, rc=2.5 * SIGMA, seed=0):
    rng = np.random.default_rng([seed, n])
    box = np.array(box if box else [(n / 0.8) ** (1.0 / 3.0) * SIGMA] * 3)
    m = np.ceil(box / (box.prod() / n) ** (1.0 / 3.0)).astype(int)
    sites = np.array([(i, j, k) for i in range(m[0]) for j in range(m[1]) for k in range(m[2])], float)
    sites = sites[np.sort(rng.permutation(len(sites))[:n])] + 0.5
    pos = sites * (box / m) + rng.uniform(-0.05, 0.05, size=(n, 3)) * SIGMA
    names = ["A" if kinds == 1 or i % 3 else "B" for i in range(n)]
    s = System.from_arrays(names, pos, UnitCell.infinite() if infinite else UnitCell.ortho(*box),
                           masses=np.full(n, 39.948))
    rc = min(rc, 0.5 * box.min() * (1.0 if rc > 2.5 * SIGMA else 0.99))
    lj = LennardJones(SIGMA, EPS)
    s.set_pair_potential(("A", "A"), PairInteraction(lj, rc))
    if kinds == 2:
        s.set_pair_potential(("A", "B"), PairInteraction.shifted(LennardJones(0.9 * SIGMA, EPS), 0.8 * rc))
        s.set_pair_potential(("B", "B"), PairInteraction(NullPotential(), rc))
    return s


def check(s, attempts=(700,), delta=0.3 * SIGMA, seed=99):
    o = lo.OracleSystem(s, nthreads=8)
    o.cache_init()
    s.cache_init()
    beta, t = 1.0 / (1.2 * EPS), 0
    for k in attempts:
        assert s.mc_run(seed, t, k, beta, delta) == o.mc_run(seed, t, k, beta, delta)
        t += k
    assert np.array_equal(s.positions, o.positions())
    assert abs(s.cache_energy() - o.cache_energy()) <= 1e-10 * abs(o.cache_energy())
    assert abs(s.cache_energy() - s.potential_energy()) <= 1e-9 * abs(s.cache_energy())


@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 255, 256, 257, 511, 512, 513, 801, 1024, 1025, 2049, 3999, 4608, 4609, 5500])
def test_sizes(n):
    check(chain(n))


@pytest.mark.parametrize("box", [(36.0, 36.0, 36.0), (34.5, 45.0, 60.0), (90.0, 35.0, 40.0), (34.5, 34.5, 200.0)])
@pytest.mark.parametrize("kinds", [1, 2])
def test_boxes_and_kinds(box, kinds):
    check(chain(1000, box, kinds))


@pytest.mark.parametrize("n", [100, 1000])
def test_infinite_cell(n):
    check(chain(n, infinite=True))


def test_cutoff_of_half_the_box():
    check(chain(500, rc=100.0))


@pytest.mark.parametrize("attempts", [(1, 62, 1, 1, 63, 64, 65, 300), (63, 129, 500), (128, 128)])
@pytest.mark.parametrize("n", [500, 1500])
def test_launches(n, attempts):
    check(chain(n), attempts)


@pytest.mark.parametrize("delta", [0.01, 2.4 * SIGMA, 6.0 * SIGMA])
def test_amplitudes(delta):
    check(chain(1500), (300, 300), delta)


def test_switching_amplitude():
    # moves past a cell and past half the box in between
    s = chain(1200)
    o = lo.OracleSystem(s, nthreads=8)
    o.cache_init()
    s.cache_init()
    beta, t = 1.0 / (1.2 * EPS), 0
    for delta in (1.0, 25.0, 1.0, 0.5):
        assert s.mc_run(3, t, 200, beta, delta) == o.mc_run(3, t, 200, beta, delta)
        t += 200
    assert np.array_equal(s.positions, o.positions())


def test_every_move_decides_the_next():
    # a few sites, most moves accepted: an attempt tests sites whose fractions
    # the attempt before has just written
    for n in (2, 4, 7):
        s = chain(n, box=(4.0 * SIGMA,) * 3, rc=1.9 * SIGMA, seed=5)
        o = lo.OracleSystem(s, nthreads=1)
        o.cache_init()
        s.cache_init()
        beta, t = 0.05 / EPS, 0
        for k in (1, 2, 61, 400, 1500):
            a = s.mc_run(31, t, k, beta, 1.2 * SIGMA)
            assert a == o.mc_run(31, t, k, beta, 1.2 * SIGMA)
            t += k
            assert np.array_equal(s.positions, o.positions())
        assert a > 1000


def test_same_bits_however_divided():
    out = []
    for parts in ([900], [100] * 9, [450, 450]):
        s = chain(1500)
        s.cache_init()
        t = 0
        for k in parts:
            s.mc_run(4, t, k, 1.0 / (1.2 * EPS), 1.0)
            t += k
        out.append((s.cache_energy(), s.positions.copy()))
    for e, p in out[1:]:
        assert e == out[0][0] and np.array_equal(p, out[0][1])
