"""GPU parity of EquilibriumInit (nrq_equilibrium.hip) against
oracle/equilibrium_oracle.py: the same number of projection sweeps, links
and E within 1e-10 after the projections and the leapfrog steps, energies
and Gauss deviations within 1e-10 relative."""
import numpy as np
import pytest

from oracle import equilibrium_oracle as eo
from oracle import gaugefix_oracle as gf

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


@pytest.mark.parametrize("ext,sp,beta,nef,neq,tol,charge", [
    ((4, 4, 4), (0.05, 1.0, 1.0, 1.0), 16.0, 2, 5, None, False),
    # an even and an odd number of leapfrog steps leave the links in either
    # of the gauge field's two buffers before the second pass
    ((4, 4, 4), (0.05, 1.0, 1.0, 1.0), 16.0, 2, 4, None, False),
    ((3, 4, 5), (0.1, 1.0, 0.8, 1.2), 8.0, 1, 3, 5e-3, True),
    # less than one block of 64 sites; a last block with 7 sites
    ((2, 3, 2), (0.05, 1.0, 1.0, 1.0), 16.0, 2, 1, 1e-2, True),
    ((5, 3, 9), (0.1, 1.0, 0.8, 1.2), 8.0, 1, 2, 2e-2, False),
])
def test_equilibrium_init_matches_oracle(nrq, oracle, lattice, ext, sp, beta, nef, neq, tol, charge):
    _say(f"EquilibriumInit {ext} beta {beta} x{nef}, {neq} steps, tol {tol}, charge {charge}")
    lattice(ext, sp)
    oracle.lattice_init(ext, sp)
    lat = gf.Lattice(ext, sp, oracle.generators())
    rho = None
    if charge:
        rho = np.random.default_rng(3).normal(size=(3, lat.vol)) * 0.2
        rho -= rho.mean(axis=1, keepdims=True)
    nrq.random_init(5)
    oracle.ranlxd_init(2, 5)
    g = nrq.GaugeConfiguration()
    en, dev, nproj = g.EquilibriumInit(beta, nef, neq, tol, rho)
    U, E, rec = eo.equilibrium_init(oracle, lat, beta, nef, neq, tol, rho)
    assert list(nproj) == [r[0] for r in rec] and min(nproj) > 0
    Ug, Eg = g.download()
    assert np.max(np.abs(Ug - U)) < 1e-10
    assert np.max(np.abs(Eg - E)) < 1e-10 * max(1.0, np.max(np.abs(E)))
    assert np.allclose(en, [r[1] for r in rec], rtol=1e-10)
    assert np.allclose(dev, [r[2] for r in rec], rtol=1e-8)
    # the same random stream position afterwards
    assert np.array_equal(nrq.random_uniform(5), oracle.ranlxd(5))


def test_equilibrium_init_rejects_bad_arguments(nrq, lattice):
    lattice((4, 4, 4), (0.05, 1.0, 1.0, 1.0))
    nrq.random_init(1)
    g = nrq.GaugeConfiguration()
    with pytest.raises(nrq.NRQError):
        g.EquilibriumInit(-1.0, 1, 1)
    with pytest.raises(nrq.NRQError):
        g.EquilibriumInit(16.0, -1, 1)


def test_equilibrium_init_without_a_sweep(nrq, lattice):
    """A tolerance above the starting deviation: no projection, the field as drawn."""
    lattice((5, 3, 9), (0.05, 1.0, 1.0, 1.0))
    nrq.random_init(4)
    g = nrq.GaugeConfiguration()
    _, dev, nproj = g.EquilibriumInit(16.0, 1, 0, 1e6)
    assert nproj[0] == 0 and 0 < dev[0] < 1e6
    assert np.isclose(dev[0], g.GetGaussMax(), rtol=1e-12)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_equilibrium_init_refuses_charges_that_are_not_numbers(nrq, lattice, bad):
    """A charge density with one entry that is not finite has no Gauss law to project
    on: an error, where the deviation's maximum once dropped the NaN and the call returned
    a field without a number in it.  The next call is not affected."""
    ext = (4, 3, 6)
    _say(f"EquilibriumInit with a charge of {bad}")
    lattice(ext, (0.05, 1.0, 1.0, 1.0))
    rho = np.zeros((3, 72))
    rho[0, 40] = bad
    nrq.random_init(5)
    g = nrq.GaugeConfiguration()
    with pytest.raises(nrq.NRQError):
        g.EquilibriumInit(16.0, 1, 2, 1e-2, rho)
    _, dev, nproj = g.EquilibriumInit(16.0, 1, 2, 1e-2)
    assert nproj[0] > 0 and np.all(np.isfinite(dev)) and np.all(np.isfinite(g.download()[1]))


def test_equilibrium_init_that_diverges_is_an_error(nrq, lattice):
    """At a tenth of the usual spatial spacing the projection's step (kappa = 0.01) is unstable,
    0.01 * 12 / 0.1^2 > 2: E grows until it is not finite, which is no small deviation."""
    _say("EquilibriumInit that diverges")
    lattice((4, 4, 4), (0.05, 0.1, 0.1, 0.1))
    nrq.random_init(5)
    g = nrq.GaugeConfiguration()
    with pytest.raises(nrq.NRQError):
        g.EquilibriumInit(16.0, 1, 0)
