"""GPU tests of the gradient kernel's sample tiles and block sums, and of the
training statistics, at the sizes where they end."""
import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_PCISPH, Params
from liquidsimulation_amd.solver import PCISPHSolver
from oracle import mlp as M

pytestmark = pytest.mark.gpu


# 16 and 32 samples to a tile pair, 128 to a block's round, 256 blocks
@pytest.mark.parametrize("n", [1, 16, 31, 32, 33, 127, 128, 129, 32767, 32769, 100003])
def test_gradient_at_tile_edges(gpu, n):
    """Per parameter block within 2e-3 (relative L2) of the BF16-emulating
    oracle, the loss within 1e-4; a second call, whose sums add in the same
    order, gives the same bits."""
    rng = np.random.default_rng(n)
    p = M.he_init(5)
    p[M.IN * M.HID:M.IN * M.HID + M.HID] = rng.normal(0, 0.1, M.HID)
    p[-1] = -0.3
    p = p.astype(np.float32)
    fs = np.concatenate([rng.normal(0, 1, M.IN), rng.uniform(0.5, 2.0, M.IN)]).astype(np.float32)
    x = (rng.normal(0, 1.5, (n, M.IN)) / fs[M.IN:] + fs[:M.IN]).astype(np.float32)
    t = rng.normal(0, 3.0, n).astype(np.float32)
    s = PCISPHSolver(Params(method=METHOD_PCISPH))
    s.set_warm_start_weights(p, fs, 2.5)
    g, loss = s.mlp_grad(x, t, 1.5)
    again, loss2 = s.mlp_grad(x, t, 1.5)
    s.close()
    assert np.array_equal(g, again) and loss == loss2
    ref, lref = M.grad(p, fs, 2.5, x, t, over_weight=1.5)
    assert abs(loss - lref) <= 1e-4 * lref
    o = 0
    for name, size in (("W1", M.HID * M.IN), ("b1", M.HID), ("W2", M.HID * M.HID), ("b2", M.HID), ("W3", M.HID),
                       ("b3", 1)):
        a, b = g[o:o + size].astype(np.float64), ref[o:o + size]
        assert np.linalg.norm(a - b) <= 2e-3 * max(np.linalg.norm(b), 1e-30), name
        o += size


@pytest.mark.parametrize("dims,stride", [((5, 5, 5), 1), ((9, 11, 7), 2), ((16, 16, 17), 1)])
def test_training_statistics(gpu, dims, stride):
    """Means, inverse deviations and target scale of the collected rows against
    numpy in 64 bits: one rounding to float32, and the cancellation of
    E[x^2] - E[x]^2 where the deviation is small against the mean."""
    sc = scenes.small_block(*dims, dt=0.002)
    s = PCISPHSolver(sc.params)
    s.set_colliders(sc.colliders)
    s.set_particles(sc.x, sc.v)
    s.update(sc.dt, 3)
    s.collect(sc.n, stride)
    s.update(sc.dt, 1)
    x, t = s.dump_pairs()
    x, t = x[::stride].astype(np.float64), t[::stride].astype(np.float64)
    assert s.collected() == len(t)
    s.train_warm_start(1, batch=64, seed=2)
    w = s.get_warm_start_weights()
    scale = float(np.float32(s.delta(sc.dt)) * np.float32(sc.params.rest_density))
    s.close()
    mean, var = x.mean(0), x.var(0)
    np.testing.assert_allclose(w["feature_scale"][:M.IN], mean, rtol=2e-7, atol=1e-12)
    big = var > 1e-6 * np.maximum(1.0, mean * mean)
    np.testing.assert_allclose(w["feature_scale"][M.IN:][big], 1 / np.sqrt(var[big]), rtol=1e-6)
    rms = np.sqrt(np.mean(t * t)) / scale
    np.testing.assert_allclose(w["target_scale"], rms if rms > 0 else 1.0, rtol=1e-6)  # 1 when every target is 0
