"""GPU tests of the counting sort: keys, stable order and cell table against
the oracle where particles arrive in their cells out of order."""
import numpy as np
import pytest

from liquidsimulation_amd.abi import METHOD_SPH, Params
from liquidsimulation_amd.solver import SPHSolver

pytestmark = pytest.mark.gpu


# (particles, extent in cells): one particle; a block less one, a block, one
# more; every particle in one cell (runs that span waves and blocks); crowded
# cells; cell counts below, at and past one scan tile of 1024 and past 32 tiles
@pytest.mark.parametrize("n,extent", [(1, 1.0), (255, 3.2), (256, 3.2), (257, 3.2), (700, 0.9), (5000, 4.5),
                                      (2000, 9.95), (2000, 10.05), (3001, 33.0)])
def test_shuffled_particles_sort_stably(gpu, oracle, n, extent):
    p = Params(method=METHOD_SPH, particle_radius=0.01, kernel_radius_factor=3.2, gravity=(0.0, 0.0, 0.0))
    h = float(np.float32(0.01) * np.float32(3.2))
    rng = np.random.default_rng(n)
    x = (rng.random((n, 3), np.float32) * np.float32(extent * h)).astype(np.float32)
    s = SPHSolver(p)
    s.set_particles(x)
    for step in range(2):  # the second from the sorted order and the first's motion
        before = s.get_particles()["x"]
        s.update(1e-4, 1)
        g, ref = s.get_grid(), oracle.grid(p, before)
        np.testing.assert_array_equal(g["keys"], ref.keys)
        np.testing.assert_array_equal(g["perm"], ref.perm)
        np.testing.assert_array_equal(g["cell_start"], ref.cell_start)
        ids = s.get_particles()["id"]
        assert np.array_equal(np.sort(ids), np.arange(n))
        if step == 0:
            np.testing.assert_array_equal(ids, ref.perm)
    s.close()
