"""GPU tests of states with infinite or NaN components: a velocity that no
other particle sees (the leapfrog advances the half-step velocity, so the step
replaces it) leaves the step equal to the oracle's, whatever the lanes."""
import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_PCISPH, METHOD_SPH
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
