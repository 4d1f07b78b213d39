"""GPU tests of the upload, append and readback of particles: every row comes
back as it was given, through the pinned buffer (up to 1 MiB) and past it."""
import numpy as np
import pytest

from liquidsimulation_amd.abi import METHOD_SPH, Params
from liquidsimulation_amd.solver import Ensemble, SPHSolver

pytestmark = pytest.mark.gpu


def _rows(n, seed):
    rng = np.random.default_rng(seed)
    f = lambda: rng.normal(0, 1, (n, 3)).astype(np.float32)  # noqa: E731
    return f(), f(), f(), rng.integers(0, 3, n).astype(np.uint8)


def _same(p, x, v, vhalf, first, ids):
    np.testing.assert_array_equal(p["x"], x)
    np.testing.assert_array_equal(p["v"], np.zeros_like(x) if v is None else v)
    np.testing.assert_array_equal(p["vhalf"], np.zeros_like(x) if vhalf is None else vhalf)
    np.testing.assert_array_equal(p["first"], np.ones(len(x), np.uint8) if first is None else (first != 0))
    np.testing.assert_array_equal(p["id"], ids)


# a row of a full upload takes 37 bytes: 28339 of them fit 1 MiB, 28340 do not
@pytest.mark.parametrize("n", [1, 255, 256, 257, 28339, 28340, 70001])
@pytest.mark.parametrize("given", ["x", "xv", "all"])
def test_round_trip(gpu, n, given):
    x, v, vhalf, first = _rows(n, n)
    if given != "all":
        vhalf = first = None
    if given == "x":
        v = None
    s = SPHSolver(Params(method=METHOD_SPH))
    for _ in range(2):  # again into the arrays of the first upload
        s.set_particles(x, v, vhalf, first)
        _same(s.get_particles(), x, v, vhalf, first, np.arange(n))
    # fewer particles afterwards, in the same arrays
    m = max(n // 2, 1)
    s.set_particles(x[:m])
    _same(s.get_particles(), x[:m], None, None, None, np.arange(m))
    s.close()


# within the last block, exactly filling it, into new blocks, past the storage
@pytest.mark.parametrize("n,more", [(250, 3), (250, 6), (250, 7), (512, 1), (300, 40000)])
def test_append(gpu, n, more):
    x, v, vhalf, first = _rows(n + more, 7)
    s = SPHSolver(Params(method=METHOD_SPH))
    s.set_particles(x[:n], v[:n], vhalf[:n], first[:n])
    ke0 = 0.5 * s.getParticleMass() * np.sum(v.astype(np.float64) ** 2)
    s.add_particles(x[n:], v[n:], vhalf[n:], first[n:])
    _same(s.get_particles(), x, v, vhalf, first, np.arange(n + more))
    # the records of all blocks, old and new
    ke, _ = s.get_energy()
    assert abs(ke[0] - ke0) <= 1e-5 * ke0
    s.close()


def test_scenes_of_ragged_sizes(gpu):
    sizes = [1, 256, 300, 511]
    rows = [_rows(k, k) for k in sizes]
    e = Ensemble(Params(method=METHOD_SPH))
    e.set_scenes([r[0] for r in rows], [r[1] for r in rows])
    p = e.get_particles()
    _same(p, np.concatenate([r[0] for r in rows]), np.concatenate([r[1] for r in rows]), None, None,
          np.arange(sum(sizes)))
    e.close()
