"""The step kernels at the edges of their tiles and launches."""
import numpy as np
import pytest

from oracle import oracle as O
from origami_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    from origami_amd import engine
    return engine


@pytest.mark.parametrize("lengths", [(1,), (3, 1, 4), (20,), (2, 30, 2, 5)])
def test_recorded_kinetic_energy_of_systems_sharing_waves(E, lengths):
    """Per-system kinetic energies of a recorded step are those of the
    velocities it leaves, for systems that share a wave or span several.
    Each atom's energy is rounded to 2^-32 kJ/mol (half a unit per atom) and
    formed in FP64 (a few 1e-16 of the sum)."""
    systems = [S.seeded_chain(40 + k, n) for k, n in enumerate(lengths)]
    eng = E.Engine(systems)
    rng = np.random.default_rng(1)
    eng.set_velocities(rng.normal(scale=0.002, size=(eng.n_atoms, 3)))
    eng.dynamics_setup([300.0] * len(systems), dt_fs=0.01, friction_ps_inv=1.0, seed=3)
    ke = eng.run(3, record_ke=True)
    for s, v, got in zip(systems, eng.split(eng.velocities()), ke[-1]):
        ref = O.Oracle(s).kinetic_energy(v)
        assert abs(got - ref) <= s.n_atoms * 2.0 ** -33 + 1e-14 * s.n_atoms * ref
    again = E.Engine(systems)
    again.set_velocities(np.random.default_rng(1).normal(scale=0.002, size=(eng.n_atoms, 3)))
    again.dynamics_setup([300.0] * len(systems), dt_fs=0.01, friction_ps_inv=1.0, seed=3)
    again.run(3)
    assert np.array_equal(again.velocities(), eng.velocities())


# (seed, residues) of chains whose atom counts end a tile: 63, 64, 65 (one
# tile and a bit), 256 / 257 (the last split system, the first with strips),
# 319, 320, 321, 512, 577 and, with strips of more than one group of j tiles,
# 1 201 atoms
EDGE_CHAINS = [(16, 4), (21, 4), (3, 3), (9, 15), (13, 16), (14, 19), (22, 18), (28, 19), (14, 30), (26, 33), (2, 70)]


@pytest.mark.parametrize("mode_a", [False, True])
@pytest.mark.parametrize("chains, strip", [([c], 4) for c in EDGE_CHAINS] + [(EDGE_CHAINS, 4), ([(2, 70)], 8),
                                                                             ([(2, 70)], 5), ([(2, 70)], 1)])
def test_block_per_item_equals_wave_per_item(E, chains, strip, mode_a):
    """The block-per-item pair kernels add the same pair terms in the same
    order as the one-wave kernels (which the profiled path runs): forces,
    radii and integrals agree bit for bit, and so does a trajectory."""
    systems = [S.seeded_chain(*c) for c in chains]
    rng = np.random.default_rng(5)
    x = np.concatenate([s.pos + rng.normal(scale=0.02, size=s.pos.shape) for s in systems])
    out = []
    for profiled in (False, True):
        eng = E.Engine(systems)
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


@pytest.mark.parametrize("stretch", [1.0, 1.7, 1.0e4])
@pytest.mark.parametrize("profiled", [False, True])
@pytest.mark.parametrize("mode_a", [False, True])
def test_pair_forces_against_oracle(E, mode_a, profiled, stretch):
    """Both pair-kernel forms against the FP64 oracle within the engine's force
    bar (1e-5): under the cutoffs, tile pairs on either side of them (stretched
    coordinates move more of them past it, up to all) are left out only where
    every pair is beyond."""
    s = S.seeded_chain(2, 70)
    x = stretch * (s.pos + np.random.default_rng(6).normal(scale=0.02, size=s.pos.shape))
    cut = (10.0, 10.0, 20.0) if mode_a else ()
    orc = O.Oracle(s)
    ref = orc.total_force(x, *cut)
    eng = E.Engine([s])
    eng.profile(profiled)
    got = eng.total_force(x, mode_a=mode_a)
    assert np.sqrt(((got - ref) ** 2).sum() / (ref ** 2).sum()) < 1e-5


@pytest.mark.parametrize("chains", [[(3, 3)], [(21, 4), (16, 4)], [(2, 70)]])
def test_sasa_terms_forms_agree(E, chains):
    """The SASA terms with a direction per lane (short lists) equal those with
    a thread per arc (batches above 4 096 SASA atoms) bit for bit: a system's
    SASA forces alone and inside a large batch."""
    systems = [S.seeded_chain(*c) for c in chains]
    rng = np.random.default_rng(8)
    x = [s.pos + rng.normal(scale=0.02, size=s.pos.shape) for s in systems]
    filler = S.seeded_chain(5, 300)
    fx = filler.pos + rng.normal(scale=0.02, size=filler.pos.shape)
    alone = E.Engine(systems)
    batch = E.Engine(systems + [filler] * 4)
    assert alone.info()["sasa_work_atoms"] <= 4096 < batch.info()["sasa_work_atoms"]
    n = alone.n_atoms

    def sasa(eng, pos):
        # the pair and bonded parts are the same integers in both calls
        return eng.total_force(pos, include_sasa=True) - eng.total_force(pos)

    xs = np.concatenate(x)
    a, b = sasa(alone, xs), sasa(batch, np.concatenate([xs] + [fx] * 4))[:n]
    assert np.array_equal(a, b)
    ref = np.concatenate([O.Oracle(s).sasa_forces(p)[0] for s, p in zip(systems, x)])
    assert np.abs(a - ref).max() < 1e-8


@pytest.mark.parametrize("chains", [[(3, 3)], [(2, 40)], [(2, 70)], [(2, 70), (3, 3)]])
def test_minimiser_direction_forms_agree(E, chains):
    """The L-BFGS direction with its vectors in registers (a form per system
    size) equals the strided form: a system's iterates do not depend on the
    largest system beside it (5 462 atoms and more select the strided form)."""
    from origami_amd.minimize import minimize_device
    systems = [S.seeded_chain(*c) for c in chains]
    big = S.seeded_chain(5, 340)
    assert big.n_atoms > 64 * 256 // 3
    n = sum(s.n_atoms for s in systems)
    alone, beside = E.Engine(systems), E.Engine(systems + [big])
    for eng in (alone, beside):
        minimize_device(eng, max_steps=14, mode_a=True)
    assert np.array_equal(alone.positions(), beside.positions()[:n])


@pytest.mark.parametrize("stretch", [1.0, 1.7, 40.0])
@pytest.mark.parametrize("profiled", [False, True])
@pytest.mark.parametrize("mode_a", [False, True])
@pytest.mark.parametrize("chains", [[(16, 4)], [(3, 3), (9, 15), (13, 16)], [(2, 70)]])
def test_energies_of_both_forms_against_oracle(E, chains, mode_a, profiled, stretch):
    """Pair energies by both forms (the profiled path runs the one-wave
    form), tile pairs on either side of the cutoff and of the distance where
    only q_i q_j / r is left: relative 1e-9 with a floor of 1e-6 kJ/mol, the
    engine's energy bar (one unit of 2^-32 kJ/mol per contribution)."""
    systems = [S.seeded_chain(*c) for c in chains]
    rng = np.random.default_rng(12)
    x = [stretch * (s.pos + rng.normal(scale=0.02, size=s.pos.shape)) for s in systems]
    eng = E.Engine(systems)
    eng.profile(profiled)
    for s, p, got in zip(systems, x, eng.total_energy(np.concatenate(x), mode_a=mode_a)):
        ref = O.Oracle(s).total_energy(p, *((10.0, 20.0) if mode_a else ()))
        for k in ("lj", "coulomb", "gb_self", "gb_pair"):
            assert abs(got[k] - ref[k]) <= 1e-9 * abs(ref[k]) + 1e-6, (k, got[k], ref[k])


@pytest.mark.parametrize("seed", [0, 1, 2])
@pytest.mark.parametrize("n_atoms", [1, 2, 7, 40])
def test_areas_of_clusters_against_oracle(E, n_atoms, seed):
    """Accessible areas (face walk, probe components) of isolated atoms, pairs
    and loose clusters with several boundary loops per atom, against the FP64
    oracle: 1e-9 relative, with a unit of the fixed-point sum per atom."""
    base = S.seeded_chain(2, 10)
    rng = np.random.default_rng(100 * n_atoms + seed)
    import copy
    s = copy.copy(base)
    m = base.n_atoms
    # spheres only: no bonded terms, no pair interactions
    for k in ("bonds", "bond_params", "angles", "angle_params", "dihedrals", "dihedral_params", "impropers",
              "improper_params", "constraints", "constraint_len"):
        setattr(s, k, getattr(base, k)[:0])
    s.charge, s.epsilon, s.epsilon_14 = np.zeros(m), np.zeros(m), np.zeros(m)
    # the first n_atoms atoms in a loose ball, the rest far from it and each other
    x = np.cumsum(np.full((m, 3), 40.0), axis=0) + 1000.0
    x[:n_atoms] = rng.uniform(-1.0, 1.0, size=(n_atoms, 3)) * 1.9 * n_atoms ** (1.0 / 3.0)
    got = E.Engine([s]).total_energy(x, include_sasa=True)[0]["sasa"]
    ref = float((O.Oracle(s).sasa_area(x)[1] * s.sasa_gamma).sum())
    assert abs(got - ref) <= 1e-9 * abs(ref) + m * 2.0 ** -32


@pytest.mark.parametrize("replicas", [2, 7, 66, 70])
def test_exchanges_of_a_round_at_once(E, replicas):
    """Pairs exchanged in one call leave the bits that one call each leaves, up to and past a launch's pairs."""
    s = S.seeded_chain(3, 2)
    pairs = [(k, k + 1) for k in range(0, replicas - 1, 2)]
    state = []
    for together in (True, False):
        eng = E.Engine([s] * replicas)
        rng = np.random.default_rng(1)
        eng.set_positions(np.concatenate([s.pos + rng.normal(scale=0.02, size=s.pos.shape) for _ in range(replicas)]))
        eng.set_velocities(rng.normal(scale=0.002, size=(eng.n_atoms, 3)))
        eng.dynamics_setup(list(300.0 + np.arange(replicas)), dt_fs=0.5, friction_ps_inv=1.0, seed=3)
        if together:
            eng.swap_pairs(pairs)
            with pytest.raises(E.EngineError):
                eng.swap_pairs([(0, 1), (1, 0)])
        else:
            for a, b in pairs:
                eng.swap(a, b)
        state.append((eng.positions(), eng.velocities()))
        eng.run(2)
        state[-1] += (eng.positions(), eng.velocities())
    assert all(np.array_equal(x, y) for x, y in zip(*state))


def _mix(x):
    m = (1 << 64) - 1
    x = (x + 0x9E3779B97F4A7C15) & m
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & m
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & m
    return x ^ (x >> 31)


@pytest.mark.parametrize("rows", [32, 96, 2080, 8192])
def test_network_batch_sizes(E, c2_system, rows):
    """Gradient of a batch and one training step at the ends of the batch range, against the oracle.

    The gradient's bounds are those of the network's own tests (bfloat16
    roundings on either side of a tie).  The step's batch is rebuilt on the
    host: its loss differs by the targets' rounding to float only (about 1e-6),
    and a first Adam step moves a parameter by lr against its gradient's sign,
    checked where the gradient is well clear of zero.
    """
    from oracle import surrogate as SO
    eng = E.Engine([c2_system])
    eng.surrogate_setup(eng.n_atoms, seed=7)
    p = SO.init_params(4).astype(np.float32)
    eng.surrogate_params(p)
    eng.set_positions(c2_system.pos)
    n = eng.surrogate_collect()
    x = eng.surrogate_descriptors(c2_system.pos)
    eng.total_force(c2_system.pos)
    r = eng.born_radii()[0]
    seed, lr = 3, 2e-3
    sd = seed * 0x9E3779B97F4A7C15 & ((1 << 64) - 1)
    pick = np.array([_mix(sd ^ _mix(b)) % n for b in range(rows)])
    g, loss = eng.surrogate_gradient(x[pick], r[pick])
    gref, lref = SO.gradient(p.astype(np.float64), x[pick].astype(np.float64), r[pick])
    assert abs(loss - lref) <= 1e-3 * lref
    for a, b in ((SO.OFF_W1, SO.OFF_B1), (SO.OFF_B1, SO.OFF_W2), (SO.OFF_W2, SO.OFF_B2), (SO.OFF_B2, SO.OFF_W3),
                 (SO.OFF_W3, SO.OFF_B3), (SO.OFF_B3, SO.P)):
        assert np.linalg.norm(g[a:b] - gref[a:b]) < 2e-2 * np.linalg.norm(gref[a:b])
    first = eng.surrogate_train(1, batch=rows, lr=lr, seed=seed)
    assert abs(first[0] - loss) <= 1e-4 * loss
    clear = np.abs(g) > 1e-3 * np.abs(g).max()
    moved = eng.surrogate_params().astype(np.float64) - p
    assert np.abs(moved + lr * np.sign(g))[clear].max() < 1e-3 * lr


def test_network_losses_of_long_runs(E, c1_system):
    """Every step's loss comes back, also past the number that is held on the device."""
    eng = E.Engine([c1_system])
    got = []
    for steps in (1030, 1024, 3):
        eng.surrogate_setup(eng.n_atoms, seed=1)
        eng.set_positions(c1_system.pos)
        eng.surrogate_collect()
        got.append(eng.surrogate_train(steps, batch=32, lr=1e-3, seed=9))
    assert np.all(got[0] > 0.0)
    assert np.array_equal(got[0][:1024], got[1]) and np.array_equal(got[0][:3], got[2])


@pytest.mark.parametrize("chains", [[(16, 4)], [(21, 4), (3, 3)], [(9, 15), (16, 4)], [(2, 70)]])
@pytest.mark.parametrize("places", ["lattice", "nudged", "far", "spread"])
def test_descriptors_at_bin_edges(E, chains, places):
    """Neighbour counts with distances on and next to the bin edges, coincident atoms, far origins and wide tiles.

    The counts are whole numbers and exact.  On a lattice of the bin width
    every distance along an axis is an edge; the nudged one is off by 1e-9 of
    itself either way; the spread one reaches beyond the range in which the
    kernel forms single-precision distances.  The radii that follow are those
    of the network's own test's bound.
    """
    from oracle import surrogate as SO
    systems = [S.seeded_chain(*c) for c in chains]
    rng = np.random.default_rng(5)
    pos = []
    for s in systems:
        x = 0.375 * rng.integers(-16, 17, size=(s.n_atoms, 3)).astype(np.float64)
        x[::5, 1:] = 0.0                        # a fifth on one axis
        if places == "nudged":
            x *= 1.0 + 1e-9 * rng.choice([-1.0, 1.0], size=x.shape)
        elif places == "far":
            x += 375.0 * 64
        elif places == "spread":
            x[1::3] *= 24.0
        pos.append(x)
    pos = np.concatenate(pos)
    eng = E.Engine(systems)
    eng.surrogate_setup(0, seed=1)
    x = eng.surrogate_descriptors(pos)
    mass = np.concatenate([s.mass for s in systems])
    rho = np.concatenate([s.gb_rho for s in systems])
    assert np.array_equal(x.astype(np.float64), SO.descriptors(pos, mass, rho, eng.offsets))
    p = SO.init_params(3)
    eng.surrogate_params(p.astype(np.float32))
    ref = SO.radius(SO.forward(p, x.astype(np.float64))[0])
    assert np.abs(eng.surrogate_radii(pos) / ref - 1.0).max() < 1e-3
