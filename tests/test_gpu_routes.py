"""What a call leaves and answers whichever kernels it takes: state after a
minimisation, launch choices, host copies, network inputs, pair-kernel forms."""
import time

import numpy as np
import pytest

from oracle import oracle as O
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


def test_autotune_without_sasa_leaves_the_sasa_width(E):
    """A width that was not timed is not chosen: choice 0, which og_set_launch keeps."""
    systems = [S.seeded_chain(3, 10)] * 4
    eng = E.Engine(systems)
    ch = eng.autotune()
    assert ch["sasa_blocks"] == 0 and ch["pair_blocks"] > 0
    eng.set_launch(pair_blocks=ch["pair_blocks"], sasa_blocks=ch["sasa_blocks"])
    x = _jittered(systems, 4)
    assert np.array_equal(eng.total_force(x, include_sasa=True), E.Engine(systems).total_force(x, include_sasa=True))
    assert eng.autotune(include_sasa=True)["sasa_blocks"] > 0


def test_autotune_times_the_force_pass_that_runs(E):
    """The strip length it keeps is the fastest of the three, within a few per
    cent, in the steps that follow (64 chains of 20 residues, whose force pass
    takes a block per item: 8 j tiles are a tenth faster than 2 or 4)."""
    systems = [S.seeded_chain(4, 20)] * 64
    eng = E.Engine(systems)
    eng.set_positions(_jittered(systems, 2))
    eng.set_velocities(np.zeros((eng.n_atoms, 3)))
    kept = eng.autotune()["strip_tiles"]
    eng.dynamics_setup([300.0] * 64, dt_fs=1e-3, seed=1)
    best = {n: np.inf for n in (2, 4, 8)}
    for _ in range(8):
        for n in best:
            eng.strip_tiles(n)
            eng.run(5)
            t = time.perf_counter()
            eng.run(40)
            best[n] = min(best[n], time.perf_counter() - t)
    assert best[kept] <= 1.05 * min(best.values()), (kept, best)


@pytest.mark.parametrize("residues", [1, 42, 43, 44, 300, 520])
def test_state_copies_of_every_size(E, residues):
    """Positions and velocities come back as they were set and forces as the
    call returned them, on both sides of the sizes where copies change route
    (16 KB: 682 atoms; 8 192 atoms)."""
    s = S.seeded_chain(5, residues)
    eng = E.Engine([s])
    rng = np.random.default_rng(residues)
    x, v = s.pos + rng.normal(scale=0.02, size=s.pos.shape), rng.normal(size=s.pos.shape)
    eng.set_velocities(v)
    eng.set_positions(x)
    assert np.array_equal(eng.positions(), x) and np.array_equal(eng.velocities(), v)
    f = eng.total_force()
    assert np.array_equal(eng.forces(), f)
    assert np.array_equal(E.Engine([s]).total_force(x), f)
    x[-1, 2] = np.nan
    with pytest.raises(E.EngineError, match="non-finite input at %d" % (x.size - 1)):
        eng.set_positions(x)


@pytest.mark.parametrize("steps", [3, 1024, 1025])
def test_kinetic_energies_of_every_length(E, steps):
    """Recorded kinetic energies on both sides of the copy's route, against those of the call without allocation."""
    s = S.seeded_chain(3, 2)
    out = []
    for noalloc in (False, True):
        eng = E.Engine([s, s])
        eng.set_velocities(np.random.default_rng(1).normal(scale=0.002, size=(eng.n_atoms, 3)))
        eng.dynamics_setup([300.0, 310.0], dt_fs=0.1, friction_ps_inv=1.0, seed=3)
        out.append(eng.run(steps, record_ke=True, noalloc=noalloc))
    assert np.all(out[0] > 0.0) and np.array_equal(*out)
    ref = O.Oracle(s).kinetic_energy(eng.split(eng.velocities())[1])
    assert abs(out[0][-1][1] - ref) <= s.n_atoms * 2.0 ** -33 + 1e-14 * s.n_atoms * ref


# (systems, strip length): one chain of 4 915 atoms, whose strips are too many
# to be split over their i and j sides (two coefficient buffers, one barrier a
# j tile; with 5 and 8 j tiles a second group of them), and lists of more work
# items than the block-per-item descreening takes with a force pass of that
# form (systems of 3 to 5, 8 or 9, and 20 to 22 tiles)
@pytest.mark.parametrize("mode_a", [False, True])
@pytest.mark.parametrize("chains, strip", [([(5, 300)], 1), ([(5, 300)], 4), ([(5, 300)], 5), ([(5, 300)], 8),
                                           ([(40 + k, 14) for k in range(70)], 4),
                                           ([(40 + k, 30) for k in range(16)], 8),
                                           ([(40 + k, 80) for k in range(9)], 8)])
def test_pair_forms_of_long_lists_agree(E, chains, strip, mode_a):
    """Block-per-item and one-wave pair kernels (the profiled path runs the
    latter) leave the same bits where strips are evaluated whole and where only
    the force pass has the block form."""
    systems = [S.seeded_chain(*c) for c in chains]
    x = _jittered(systems, 6)
    out = []
    for profiled in (False, True):
        eng = E.Engine(systems)
        assert eng.info()["tile_pairs"] <= 4864
        eng.strip_tiles(strip)
        eng.profile(profiled)
        f = eng.total_force(x, mode_a=mode_a)
        r, h = eng.born_radii()
        eng.set_velocities(np.zeros_like(x))
        eng.dynamics_setup([300.0] * len(systems), dt_fs=0.01, seed=9, mode_a=mode_a)
        eng.run(3)
        out.append((f, r, h, eng.positions(), eng.velocities(), eng.status()["clamped"]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
