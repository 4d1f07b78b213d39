"""Distance and reciprocal distance of the pressure passes (dist_rn in
lps_kernels.hip), and the flag that sends the force passes to their checked
quotients."""
import os
import subprocess

import numpy as np
import pytest

from liquidsimulation_amd import scenes
from liquidsimulation_amd.abi import METHOD_PCISPH, METHOD_SPH
from tests import build_checks
from tests.helpers import gpu_run, ulp_diff

pytestmark = pytest.mark.gpu


def test_root_and_reciprocal_match_ieee(gpu):
    exe = build_checks.path("rsq_rn_check")
    if not os.path.exists(exe):
        raise RuntimeError(f"{exe} is not built; run `python tests/build_checks.py`")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and "1476395008 floats, 0 wrong roots, 0 wrong reciprocals" in r.stdout
    # the refused: about one significand in 2^24 and the neighbours of its residual
    assert int(r.stdout.split(",")[3].split()[0]) < 1476395008 // 1000


@pytest.mark.parametrize("method", [METHOD_SPH, METHOD_PCISPH])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("what", ["plain", "tiny velocity", "tiny coordinate", "coincident", "wide kernel"])
def test_force_passes_match_the_oracle(gpu, oracle, method, lanes, what):
    """Steps whose state has components too small for the unchecked quotients,
    two particles at one point, and a kernel so wide (h = 3.2 m) that its
    table entries are below 1."""
    kw = {"s": 1.0, "dt": 0.01} if what == "wide kernel" else {}
    sc = scenes.small_block(6, 7, 6, seed=4, method=method, **kw)
    st = oracle.State.from_scene(sc.x)
    st.v[:] = np.random.default_rng(1).normal(0, 0.1, st.v.shape).astype(np.float32)
    if what == "tiny velocity":
        st.v[17] = (1e-20, 0.0, -3e-30)
        st.v[18] = (2e-20, -1e-25, 1e-38)
    elif what == "tiny coordinate":
        st.x -= st.x[100]
        st.x[100] = (1e-20, 3e-30, -1e-22)
    elif what == "coincident":
        st.x[30] = st.x[31]
    ref = st.copy()
    for _ in range(3):
        oracle.step_ocl(sc.params, sc.colliders, sc.dt, ref)
    s, _ = gpu_run(sc.params, sc.colliders, sc.dt, st, 3, lanes=lanes)
    p = s.get_particles()
    for k, a in (("x", ref.x), ("v", ref.v), ("vhalf", ref.vh)):
        assert ulp_diff(p[k], a) == 0, k
