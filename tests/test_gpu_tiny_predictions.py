"""GPU test of predictions that reach a coordinate in (0, 2^-56) only within
the correction loop, so that a pressure pass itself finds the first of them
and the passes after it check their quotients' numerators."""
import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_PCISPH
from tests.helpers import gpu_run, ulp_diff

pytestmark = pytest.mark.gpu


# one lane, and by size a team of 16 lanes (625 particles) or a quad (62,500: 245 particle blocks)
@pytest.mark.parametrize("side,lanes", [(25, 1), (25, 4), (250, 1), (250, 4)])
def test_first_tiny_prediction_in_the_loop(gpu, oracle, side, lanes):
    """A compressed layer, one particle thick: all z lie in [2^-56, 1.8 * 2^-56],
    so the forces along z are as small, and without viscosity and tension the
    first prediction keeps every z.  The pressure then moves some below 2^-56."""
    sc = scenes.small_block(2, 2, 2, s=0.02, method=METHOD_PCISPH, dt=5e-4, viscosity=0.0, surface_tension=0.0,
                            min_iterations=6, max_iterations=6, stall_iterations=0)
    sc.colliders.boxes = []
    rng = np.random.default_rng(side)
    i = np.arange(side * side)
    x = np.stack([0.0155 * (i // side), 0.0155 * (i % side), np.zeros(i.size)], 1).astype(np.float32)
    x[:, :2] += rng.uniform(-1e-3, 1e-3, (i.size, 2)).astype(np.float32)
    x[:, 2] = (2.0 ** -56 * rng.uniform(1.0, 1.8, i.size)).astype(np.float32)
    x[:, 2] = np.maximum(x[:, 2], np.float32(2.0 ** -56))
    st = oracle.State.from_scene(x)
    st.first[:] = 0  # no velocity: the first prediction leaves z as it is
    s, stats = gpu_run(sc.params, sc.colliders, sc.dt, st, 1, lanes=lanes)
    p, f = s.get_particles(), s.get_fields()
    s.close()
    tr = oracle.step_ocl(sc.params, sc.colliders, sc.dt, st)
    z = np.abs(st.x[:, 2])
    assert tr.iterations == 6 and 0 < np.count_nonzero(z < 2.0 ** -56) < z.size
    assert stats[0].iterations == tr.iterations
    for k, ref in (("x", st.x), ("v", st.v), ("vhalf", st.vh)):
        assert ulp_diff(p[k], ref) == 0, k
    assert ulp_diff(f["rho_pred"], tr.rho_pred) == 0
    assert ulp_diff(f["pressure"], tr.pressure) == 0
