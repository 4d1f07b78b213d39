"""CPU tests of the library's host code where an allocation fails: the library
runs over a stand-in for the HIP runtime (fake_hip.cpp) in a process of its
own.  What a failed call left behind must not reach the device: later calls
either report an error or find everything they launch with in place."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
F = C.CDLL({fake!r}, C.RTLD_GLOBAL)  # before the library, which then binds to it
F.fake_bytes.restype = C.c_size_t
sys.path.insert(0, {root!r})
sys.modules["torch"] = None  # it would bring the real runtime
import numpy as np
from liquidsimulation_amd._lib import LPSError
from liquidsimulation_amd.abi import Box, Colliders, METHOD_PCISPH, METHOD_SPH, Params, WARM_LEARNED
from liquidsimulation_amd.solver import Ensemble, PCISPHSolver, SPHSolver
OOM, STATE = 3, 7
def status(call, *a):
    try:
        call(*a)
    except LPSError as e:
        return e.status
    return 0
def rows(n):
    return np.zeros((n, 3), np.float32)
def box(half):
    return Colliders(boxes=[Box(center=(0.0, 0.0, 0.0), half=(half,) * 3, boundary=True)])
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    from liquidsimulation_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("liblps.so is not built")
    fake = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "liquidsimulation_amd", "csrc"),
                    "-o", fake, os.path.join(HERE, "fake_hip.cpp")], check=True, capture_output=True)

    def go(body):
        code = PRELUDE.format(fake=fake, root=ROOT) + textwrap.dedent(body)
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


# 12,000 particles are sorted by one workgroup, 17,000 in several launches
@pytest.mark.parametrize("n", [12000, 17000])
# the three allocations of the cell table
@pytest.mark.parametrize("which", [0, 1, 2])
def test_cell_table_growth_fails_in_an_upload(run, n, which):
    run(f"""
    s = SPHSolver(Params(method=METHOD_SPH))
    s.set_colliders(box(0.5)); s.set_particles(rows({n})); s.set_colliders(box(0.5)); s.set_particles(rows({n}))
    s.update(1e-3, 2)
    s.set_colliders(box(2.0))
    F.fake_fail_malloc({which})
    assert status(s.set_particles, rows({n})) == OOM
    F.fake_fail_malloc(-1)
    assert status(s.update, 1e-3, 1) == STATE  # the table no longer fits the scene
    s.set_particles(rows({n}))
    s.update(1e-3, 2)
    assert F.fake_null_launches() == 0
    """)


@pytest.mark.parametrize("n", [12000, 17000])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_cell_table_growth_fails_in_a_step(run, n, which):
    run(f"""
    s = SPHSolver(Params(method=METHOD_SPH))
    s.set_particles(rows({n}))
    s.update(1e-3, 2)
    F.fake_overflow(1 << 20)
    F.fake_fail_malloc({which})
    assert status(s.update, 1e-3, 1) == OOM
    F.fake_fail_malloc(-1)
    F.fake_overflow(1 << 20)  # it still needs them
    s.update(1e-3, 2)
    assert F.fake_null_launches() == 0
    """)


# every allocation of a larger upload, and past the last
@pytest.mark.parametrize("method", ["METHOD_SPH", "METHOD_PCISPH"])
def test_upload_fails_at_any_allocation(run, method):
    run(f"""
    failed = 0
    for which in range(60):
        s = Ensemble(Params(method={method}))
        s.set_tuning(False)
        s.set_scenes([rows(300)]); s.update(1e-3, 2)
        F.fake_fail_malloc(which)
        st = status(s.set_scenes, [rows(9000), rows(20000)])
        F.fake_fail_malloc(-1)
        assert st in (0, OOM)
        failed += st == OOM
        assert status(s.update, 1e-3, 1) == (STATE if st else 0)
        assert status(s.get_energy) == (STATE if st else 0)
        s.set_scenes([rows(400), rows(500)]); s.update(1e-3, 2)
        s.set_scenes([rows(9000), rows(20000)]); s.update(1e-3, 2)
        s.close()
    assert 35 < failed < 60
    assert F.fake_null_launches() == 0
    """)


def test_append_fails_at_any_allocation(run):
    run("""
    lost = kept = 0
    for which in range(60):
        s = SPHSolver(Params(method=METHOD_SPH))
        s.set_particles(rows(300)); s.update(1e-3, 2)
        F.fake_fail_malloc(which)
        st = status(s.add_particles, rows(20000))
        F.fake_fail_malloc(-1)
        if st == 0:
            s.update(1e-3, 1)
        else:
            assert st == OOM
            # the state survives where the copy of it could not be made
            st = status(s.update, 1e-3, 1)
            assert st in (0, STATE)
            lost += st == STATE
            kept += st == 0
            s.set_particles(rows(300)); s.update(1e-3, 2)
        s.close()
    assert lost > 30 and kept == 6
    assert F.fake_null_launches() == 0
    """)


def test_steps_in_flight_when_a_call_fails_are_not_the_next_ones(run):
    """A seeded probe step in the middle of a call cannot allocate the network's
    features.  The steps before it are still on their way (the stand-in reports
    them when the stream is waited for); the next call counts its own only."""
    run("""
    s = PCISPHSolver(Params(method=METHOD_PCISPH, warm_start=WARM_LEARNED))
    s.set_tuning(False)
    s.set_warm_start_weights(np.zeros(5313, np.float32), np.ones(32, np.float32), 1.0)
    s.set_particles(rows(300))
    F.fake_iterations(4, 5)
    s.set_params(s.params.replace(max_iterations=8))
    st = s.update(1e-3, 20)  # the probe (step 16) is the cheaper one: the seed goes off
    assert [x.warm_start_used for x in st] == [1] * 15 + [0] * 5
    s.set_particles(rows(3000))  # larger: the features are allocated at the next probe (step 32)
    F.fake_fail_malloc(0)
    assert status(s.update, 1e-3, 20) == OOM
    F.fake_fail_malloc(-1)
    s.update(1e-3, 3)
    """)


def test_neighbour_lists_only_where_a_team_may_run(run):
    """A state of 600 particle blocks takes less than 400 bytes a slot; the lists
    of 16 lanes per particle (512 bytes a slot) come with a state that these
    may run for."""
    run("""
    before = F.fake_bytes()
    s = SPHSolver(Params(method=METHOD_SPH))
    s.set_particles(rows(153600)); s.update(1e-3, 2)
    large = F.fake_bytes() - before
    assert large < 153600 * 400
    s.set_particles(rows(300)); s.update(1e-3, 2)
    assert 131072 * 512 < F.fake_bytes() - before - large < 131072 * 520
    s.add_particles(rows(120000)); s.update(1e-3, 2)
    s.add_particles(rows(60000)); s.update(1e-3, 2)
    t = SPHSolver(Params(method=METHOD_SPH))
    t.set_particles(rows(300)); t.update(1e-3, 2)
    t.add_particles(rows(300)); t.update(1e-3, 2)
    t.add_particles(rows(3000)); t.update(1e-3, 2)
    assert F.fake_null_launches() == 0
    """)


def test_an_error_left_by_another_call_is_not_this_ones(run):
    """The runtime keeps a thread's last error until it is asked for it; calls
    that ask after their launches must not take one that was there before."""
    run("""
    def each(*calls):
        for call in calls:
            F.fake_leave_error()  # as another library's failed call would
            call()
    s = PCISPHSolver(Params(method=METHOD_PCISPH))
    s.set_tuning(False)
    each(lambda: s.set_particles(rows(300)), lambda: s.update(1e-3, 2), lambda: s.add_particles(rows(20)),
         s.get_particles, s.get_energy, lambda: s.set_params(s.params), lambda: s.set_colliders(box(0.5)),
         lambda: s.set_warm_start_weights(np.zeros(5313, np.float32), np.ones(32, np.float32), 1.0),
         lambda: s.mlp_forward(np.zeros((9, 16))), lambda: s.mlp_grad(np.zeros((9, 16)), np.zeros(9)),
         lambda: s.update(1e-3, 2), s.get_fields)
    """)


def test_cell_arrays_of_a_step_whose_table_could_not_grow(run):
    run("""
    s = SPHSolver(Params(method=METHOD_SPH))
    s.set_particles(rows(300)); s.update(1e-3, 2); s.get_grid()
    F.fake_overflow(1 << 20)
    F.fake_fail_malloc(0)
    assert status(s.update, 1e-3, 1) == OOM
    F.fake_fail_malloc(-1)
    assert status(s.get_grid) == STATE  # there is no table of so many cells to read
    s.get_particles()
    """)
