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
