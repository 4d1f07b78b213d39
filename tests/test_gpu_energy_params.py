"""GPU tests of the energies around a change of parameters: the state keeps
the energies of the parameters it was reached with until a step or an append,
whichever pass wrote (or left out) the blocks' records."""
import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_SPH
from liquidsimulation_amd.solver import solver_for

pytestmark = pytest.mark.gpu


def _solver(n, lanes):
    sc = scenes.small_block(20, 20, 20, seed=7, method=METHOD_SPH)
    sc.v[:] = np.array([0.3, -0.4, 0.2], np.float32)
    s = solver_for(sc.params)
    s.set_tuning(False, 1, 256, lanes)
    s.set_colliders(sc.colliders)
    s.set_particles(sc.x[:n], sc.v[:n])
    return s, sc


@pytest.mark.parametrize("n", [300, 5000])
def test_parameters_changed_after_steps(gpu, n):
    """Steps that integrate in the pressure pass (0 lanes: the automatic
    choice) and steps that write records report the same energies."""
    (a, sc), (b, _) = _solver(n, 0), _solver(n, 1)
    other = sc.params.replace(gravity=(1.0, -3.0, 0.5), mass_override=0.5 * a.getParticleMass())
    for s in (a, b):
        s.update(sc.dt, 3)
        s.set_params(other)
    np.testing.assert_array_equal(a.get_energy(), b.get_energy())
    for s in (a, b):
        s.update(sc.dt, 2)
    np.testing.assert_array_equal(a.get_energy(), b.get_energy())
    a.close()
    b.close()


@pytest.mark.parametrize("lanes", [0, 1])
@pytest.mark.parametrize("n,more", [(300, 20), (5000, 700)])
def test_append_after_a_change(gpu, lanes, n, more):
    """An append brings the energies to the present parameters: those of a new
    solver given the same state."""
    s, sc = _solver(n, lanes)
    s.update(sc.dt, 3)
    s.set_params(sc.params.replace(gravity=(1.0, -3.0, 0.5)))
    s.add_particles(sc.x[n:n + more], sc.v[n:n + more])
    got = s.get_energy()
    p = s.get_particles()
    t = solver_for(s.params)
    t.set_particles(p["x"], p["v"], p["vhalf"], p["first"])
    np.testing.assert_array_equal(got, t.get_energy())
    s.close()
    t.close()
