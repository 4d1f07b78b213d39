"""GPU tests of the stencil kernels with 16 lanes per particle against one
lane: bit-identical states where the team kernels' lists and ranges end."""
import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_PCISPH, METHOD_SPH
from liquidsimulation_amd.solver import solver_for
from tests.helpers import ulp_diff

pytestmark = pytest.mark.gpu


def _both(sc, steps):
    outs = []
    for lanes in (1, 4):
        s = solver_for(sc.params)
        s.set_colliders(sc.colliders)
        s.set_particles(sc.x, sc.v)
        s.set_tuning(False, 1, 256, lanes)
        its = [st.iterations for st in s.update(sc.dt, steps)]
        outs.append((s.get_particles(), its, s.get_fields()))
        s.close()
    (ref, its_ref, f_ref), (out, its, f) = outs
    assert its == its_ref
    for k in ("x", "v", "vhalf", "id"):
        np.testing.assert_array_equal(out[k], ref[k])
    for k in ("rho", "pressure", "force"):
        assert ulp_diff(f[k], f_ref[k]) == 0, k
    return its


@pytest.mark.parametrize("method", [METHOD_SPH, METHOD_PCISPH])
# about 1, 30, 120 to 140 and 250 neighbours: a recorded list holds 128, so
# the third has short and long lists in one wave
@pytest.mark.parametrize("radius_factor", [1.2, 3.2, 5.1, 6.3])
def test_list_lengths(gpu, method, radius_factor):
    sc = scenes.small_block(9, 11, 10, s=0.02, jitter_amp=4e-4, seed=21, method=method,
                            kernel_radius_factor=radius_factor)
    sc.v[:] = np.array([0.4, -0.6, 0.1], np.float32)
    _both(sc, 12)


@pytest.mark.parametrize("method", [METHOD_SPH, METHOD_PCISPH])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 257])
def test_ragged_counts(gpu, method, n):
    sc = scenes.small_block(7, 7, 7, seed=n, method=method)
    sc.x, sc.v = sc.x[:n], sc.v[:n]
    _both(sc, 5)


# 160 and 161 particle blocks
@pytest.mark.parametrize("dims", [(40, 32, 32), (41, 32, 32)])
def test_around_the_team_limit(gpu, dims):
    _both(scenes.small_block(*dims, s=0.016, jitter_amp=2e-4, seed=3, method=METHOD_PCISPH), 4)


@pytest.mark.parametrize("method", [METHOD_SPH, METHOD_PCISPH])
# a row's candidates are read 16, 32 or 64 at a time, then 32 by 32
@pytest.mark.parametrize("n", [16, 17, 32, 33, 64, 65, 96, 97, 129])
def test_row_lengths(gpu, method, n):
    sc = scenes.small_block(7, 7, 7, seed=n, method=method)
    # n particles of one cell, and a sparse row beside them
    rng = np.random.default_rng(n)
    h = sc.params.particle_radius * sc.params.kernel_radius_factor
    crowd = sc.x.mean(0) + rng.random((n, 3)) * 0.9 * h
    line = sc.x.mean(0) + np.array([0.0, 1.2, 0.0]) * h + np.linspace(-2.0, 2.0, 9)[:, None] * [h, 0.0, 0.0]
    sc.x = np.concatenate([crowd, line]).astype(np.float32)
    sc.v = np.zeros_like(sc.x)
    _both(sc, 2)


# 240 particle blocks (PCISPH: the last with a team) and 241 (a quad)
@pytest.mark.parametrize("dims", [(48, 40, 32), (47, 41, 32)])
def test_around_the_pcisph_limit(gpu, dims):
    _both(scenes.small_block(*dims, s=0.016, jitter_amp=2e-4, seed=3, method=METHOD_PCISPH), 4)
