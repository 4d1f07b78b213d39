"""GPU tests of states with infinite or NaN components: a velocity that no
other particle sees (the leapfrog advances the half-step velocity, so the step
replaces it) leaves the step equal to the oracle's, whatever the lanes, and a
position fails the step and keeps the state."""
import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_PCISPH, METHOD_SPH
from liquidsimulation_amd._lib import LPSError
from liquidsimulation_amd.solver import solver_for
from tests.helpers import ulp_diff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", [METHOD_SPH, METHOD_PCISPH])
@pytest.mark.parametrize("lanes", [0, 1])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_nonfinite_velocity_of_a_lone_particle(gpu, oracle, method, lanes, value):
    """The viscosity and divergence terms leave the pair of a particle with
    itself out, so the lone particle feels gravity only."""
    sc = scenes.small_block(8, 8, 8, method=method)
    h = sc.params.particle_radius * sc.params.kernel_radius_factor
    lone = sc.x.max(0) + np.float32(3.0 * h)
    st = oracle.State.from_scene(np.concatenate([sc.x, lone[None]]).astype(np.float32))
    st.first[:] = 0
    st.v[-1] = (0.1, value, -0.2)
    st.vh[-1] = (0.1, 0.2, -0.2)
    s = solver_for(sc.params)
    s.set_tuning(True, 1, 256, lanes)
    s.set_colliders(sc.colliders)
    s.set_particles(st.x, st.v, st.vh, st.first)
    if method == METHOD_PCISPH:
        s.capture_features()
    s.update(sc.dt, 1)
    if method == METHOD_PCISPH:
        f = s.dump_pairs()[0]
        me = np.flatnonzero(s.get_particles()["id"] == st.n - 1)[0]
        np.testing.assert_array_equal(f[me, 1:3], 0.0)  # no neighbours, no divergence
    s.update(sc.dt, 3)
    p = s.get_particles()
    s.close()
    for _ in range(4):
        assert oracle.step_ocl(sc.params, sc.colliders, sc.dt, st).status == 0
    assert np.isfinite(p["x"]).all() and np.isfinite(p["v"]).all()
    for k, ref in (("x", st.x), ("v", st.v), ("vhalf", st.vh)):
        assert ulp_diff(p[k], ref) == 0, k


# one particle of the first, a middle and the last (partly filled) wave
@pytest.mark.parametrize("n,at", [(1, 0), (500, 0), (500, 123), (500, 499), (5000, 2600), (5000, 4999)])
@pytest.mark.parametrize("value", [0x7F800000, 0xFF800000, 0x7FC00000, 0xFFC00000, 0x7F800001, 0xFFFFFFFF])
def test_nonfinite_position_fails_the_step_and_keeps_the_state(gpu, n, at, value):
    """Infinities and NaN of either sign, found by the box from the positions
    (0 lanes: the automatic choice) or from the blocks' records: the status,
    and the state as it was, with the next state's steps unharmed."""
    sc = scenes.small_block(18, 18, 18, seed=3, method=METHOD_SPH)
    x = sc.x[:n].copy()
    x.view(np.uint32)[at, at % 3] = value
    v = np.full_like(x, 0.25)
    for lanes in (0, 1):
        s = solver_for(sc.params)
        s.set_tuning(True, 1, 256, lanes)
        s.set_colliders(sc.colliders)
        s.set_particles(x, v, v)
        with pytest.raises(LPSError) as e:
            s.update(sc.dt, 3)
        assert e.value.status == 4  # LPS_ERR_NONFINITE
        p = s.get_particles()
        np.testing.assert_array_equal(p["x"].view(np.uint32), x.view(np.uint32))
        for k, ref in (("v", v), ("vhalf", v), ("first", np.ones(n)), ("id", np.arange(n))):
            np.testing.assert_array_equal(p[k], ref, err_msg=k)
        s.set_particles(sc.x[:n], v)
        s.update(sc.dt, 3)
        assert np.isfinite(s.get_particles()["x"]).all()
        s.close()
