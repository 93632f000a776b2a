"""What a call leaves and answers whichever kernels it takes: state after a
minimisation, launch choices, host copies, network inputs, pair-kernel forms."""
import numpy as np
import pytest

from origami_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    from origami_amd import engine
    return engine


def _jittered(systems, seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([s.pos + rng.normal(scale=0.02, size=s.pos.shape) for s in systems])


# systems that converge at once (any change is within the tolerances) and, in
# the last two, at steps of their own
@pytest.mark.parametrize("sasa", [False, True])
@pytest.mark.parametrize("mode_a", [False, True])
@pytest.mark.parametrize("chains, tol, profiled", [([(3, 3)], 1e9, False), ([(2, 40), (3, 3)], 1e9, False),
                                                   ([(2, 40), (3, 3)], 1e9, True), ([(5, 300)], 1e9, False),
                                                   ([(1, 20), (3, 10)], 20.0, False),
                                                   ([(1, 20), (3, 10)], 20.0, True)])
def test_integrals_after_a_converged_minimisation(E, chains, tol, profiled, mode_a, sasa):
    """The radii and descreening integrals after og_minimize are those at the
    coordinates it leaves, also for a system that converged while others went
    on; a force call there gives the same integers."""
    from origami_amd.minimize import minimize_device
    systems = [S.seeded_chain(*c) for c in chains]
    eng = E.Engine(systems)
    eng.set_positions(_jittered(systems, 3))
    eng.profile(profiled)
    res = minimize_device(eng, max_steps=500, gradient_tol=tol, energy_tol=tol / 20.0, mode_a=mode_a,
                          include_sasa=sasa)
    assert all(r.converged for r in res)
    radii, integral = eng.born_radii()
    clamped = eng.status()["clamped"]
    fresh = E.Engine(systems)
    fresh.total_force(eng.positions(), mode_a=mode_a)
    r, h = fresh.born_radii()
    assert np.any(h != 0.0)
    assert np.array_equal(integral, h)
    assert np.array_equal(radii, r)
    assert np.array_equal(clamped, fresh.status()["clamped"])


@pytest.mark.parametrize("apart", [1e7, 1e8, 1e12])
@pytest.mark.parametrize("chains", [[(16, 4)], [(9, 15), (16, 4)]])
def test_descriptors_of_tiles_that_reach_far(E, chains, apart):
    """Neighbour counts of tiles whose atoms lie in two groups so far apart
    that single-precision positions about the tile's centre would be off by
    more than the range: the counts are exact."""
    from oracle import surrogate as SO
    systems = [S.seeded_chain(*c) for c in chains]
    rng = np.random.default_rng(11)
    x = rng.uniform(-5.0, 5.0, size=(sum(s.n_atoms for s in systems), 3))
    x[::3, 0] += apart
    eng = E.Engine(systems)
    eng.surrogate_setup(0, seed=1)
    got = eng.surrogate_descriptors(x)
    mass = np.concatenate([s.mass for s in systems])
    rho = np.concatenate([s.gb_rho for s in systems])
    assert np.array_equal(got.astype(np.float64), SO.descriptors(x, mass, rho, eng.offsets))
