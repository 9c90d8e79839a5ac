"""The native library's host code without a GPU: its HIP calls are answered by tests/cpp/host_hip.cpp, which
is loaded in front of the HIP runtime in a process of its own and runs no kernels.  What is looked at:
which calls are refused, what is allocated and what is launched."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C
import sys
sys.path.insert(0, %r)
fake = C.CDLL(%r, mode=C.RTLD_GLOBAL)
import numpy as np
from isaac_sim_ros2_humble_amd import native, workloads
from isaac_sim_ros2_humble_amd.model import load_robot
from isaac_sim_ros2_humble_amd.scene import Scene


class Counts(C.Structure):
    _fields_ = [(f, C.c_longlong) for f in ("device_allocs", "device_bytes", "host_allocs", "host_bytes", "host_peak",
                                            "launches")] + [("workgroups", C.c_ulonglong)]


fake.host_hip_counts.restype = C.POINTER(Counts)
fake.host_hip_arg.restype = C.POINTER(C.c_ubyte)
counts = fake.host_hip_counts().contents
native.init(0)
L = native.lib()
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    lib = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(rocm, "include"),
                           os.path.join(HERE, "cpp", "host_hip.cpp"), "-o", lib])

    def go(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE % (REPO, lib) + code], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


def test_a_refused_call_does_not_fail_the_next_roadmap(run):
    run("""
r = native.Robot(load_robot("fr3"))
ns = native.Scene(Scene(spheres=np.array([[1, 0, 1, 0.1]], np.float32)))
q = np.zeros((2, r.dof), np.float32)
p = C.c_void_p()
assert L.mp_device_alloc(C.byref(p), 1 << 50) == native.MP_E_NOMEM
rm = native.Roadmap(r, ns, q[:1], q[1:], samples_per_iteration=8)
assert L.mp_device_alloc(C.byref(p), 1 << 50) == native.MP_E_NOMEM
got = rm.read()
assert got["nv"] == 2
# a launch that is refused itself is reported
fake.host_hip_fail(0, 719)
try:
    rm.read()
except native.MPError as e:
    assert "(-2)" in str(e)
else:
    raise AssertionError("the launch failed")
try:
    native.Roadmap(r, ns, q[:1], q[1:], samples_per_iteration=8)
except native.MPError as e:
    assert "(-2)" in str(e)
else:
    raise AssertionError("the launch failed")
""")


@pytest.mark.parametrize("nq", [1, 2, 3, (1 << 22) - 1, (1 << 22) + 1, 9000001, 67000000, (1 << 31) - 1])
def test_nearest_nodes_of_any_number_of_queries(nq, run):
    # a launch may hold fewer than 2^32 threads per dimension; two queries per workgroup
    run("""
for n in (1, 256, 257, 50000, (1 << 31) - 1):
    assert L.mp_nn_argmin(1 << 20, n, n, 7, 1 << 20, %d, 1 << 20, None) == 0, L.mp_last_error()
    assert counts.workgroups >= -(-%d // 2)
""" % (nq, nq))


def test_a_failed_update_leaves_the_scene_as_it_was(run):
    # the scene as the check kernel receives it: four counts, then the addresses of its sections
    run("""
m = load_robot("fr3")
r = native.Robot(m)
rng = np.random.default_rng(0)
big = workloads.c2_scene(seed=0)
assert all(c > 2 for c in big.counts)
small = Scene(spheres=big.spheres[:1], boxes=big.boxes[:2], cylinders=big.cylinders[:1], capsules=big.capsules[:2])
ns = native.Scene(big)
fake.host_hip_copy_arg(2, 80)


def seen():
    assert L.mp_check_states(r.h, ns.h, 1 << 20, 64, 1 << 20, None, None) == 0
    return bytes(fake.host_hip_arg()[:80])


before = seen()
fake.host_hip_fail(719, 0)
try:
    ns.update(small)
except native.MPError as e:
    assert "(-2)" in str(e)
else:
    raise AssertionError("the copy failed")
fake.host_hip_fail(0, 0)
assert seen() == before
ns.update(small)
assert seen() != before
ns.update(big)
assert seen() == before
""")


def test_pinned_memory_of_large_roadmaps(run):
    # the host memory that a roadmap pins does not grow with its states, nor with what is read of it
    run("""
fake.host_hip_limit.argtypes = [C.c_longlong]
r = native.Robot(load_robot("fr3"))
ns = native.Scene(Scene(spheres=np.array([[1, 0, 1, 0.1]], np.float32)))
n = 200000
q = np.zeros((n, r.dof), np.float32)
before = counts.host_bytes
MOST = 1 << 20
rm = native.Roadmap(r, ns, q, q, samples_per_iteration=8)
assert counts.host_bytes - before <= MOST
fake.host_hip_reset_peak()
weights = np.zeros(1, np.float32)
assert L.mp_roadmap_read(rm.h, None, None, None, native._p(weights), None, None) == 0
groups = np.zeros(2 * n, np.int32)
assert L.mp_roadmap_read(rm.h, None, native._p(groups), None, None, None, None) == 0
rm.read()
assert counts.host_peak - before <= 2 * MOST and counts.host_bytes - before <= MOST
small = native.Roadmap(r, ns, q[:3], q[:2], samples_per_iteration=8)
# without a byte more of it, reading goes on in smaller pieces
big = native.Roadmap(r, ns, q[:5000], q[:4000], samples_per_iteration=8)
fake.host_hip_limit(counts.host_bytes)
launched = counts.launches
big.read()
assert counts.launches > launched + 1
small.read()
""")


def test_kept_roadmap_storage_follows_the_roadmaps_in_use(run):
    # four roadmaps' storage is kept: the largest that were given back, the smallest that fits handed out
    run("""
r = native.Robot(load_robot("fr3"))
ns = native.Scene(Scene(spheres=np.array([[1, 0, 1, 0.1]], np.float32)))
q = np.zeros((70000, r.dof), np.float32)


def make(n):
    return native.Roadmap(r, ns, q[:n], q[:1], samples_per_iteration=8)


def allocates(f):
    before = counts.device_allocs
    f()
    return counts.device_allocs - before


for rm in [make(10) for _ in range(4)]:
    rm.close()
assert allocates(lambda: make(10).close()) == 0
# a larger one takes the place of a small one, also where four small ones are kept
assert allocates(lambda: make(6000).close()) == 1
assert allocates(lambda: make(6000).close()) == 0
for _ in range(3):  # small and large by turns, more than are kept
    assert allocates(lambda: make(10).close()) == 0
    assert allocates(lambda: make(6000).close()) == 0
# a small one leaves the large one alone
small = make(10)
assert allocates(lambda: make(6000).close()) == 0
small.close()
# what is too large to keep is freed
held = counts.device_bytes
assert allocates(lambda: make(70000).close()) == 1
assert counts.device_bytes == held
# four at once of the larger size: the small ones are gone, and a small roadmap takes a larger storage
for rm in [make(6000) for _ in range(4)]:
    rm.close()
assert allocates(lambda: make(10).close()) == 0
L.mp_shutdown()
""")


@pytest.mark.parametrize("kind,counts", [("check", (5, 2)), ("check", (20, 3)), ("check", (32, 4)), ("check", (200, 4)),
                                         ("cost", (5, 2)), ("cost", (200, 4))])
def test_waves_of_small_batches(kind, counts, run):
    # one wave a SIMD at most, fewer where there are few obstacles, until waves are full: four waves per
    # workgroup, 256 CUs
    run("""
obstacles, per_cu = %r
r = native.Robot(load_robot("fr3"))
ns = native.Scene(Scene(spheres=np.ones((obstacles, 4), np.float32)))
for n in (1, 2, 255, 511, 512, 513, 1025, 1537, 2049, 4099, 6001, 12001, 16385, 24001, 32767, 32768, 32769, 65537, 1 << 20):
    if %r == "check":
        assert L.mp_check_states(r.h, ns.h, 1 << 20, n, 1 << 20, None, None) == 0
    else:
        assert L.mp_state_costs(r.h, ns.h, 1 << 20, n, 1 << 20, 1 << 20, None) == 0
    waves = 256 * per_cu
    per_wave = min(64, -(-n // waves))
    assert counts.workgroups == -(-n // (4 * per_wave)), n
    assert per_wave == 64 or counts.workgroups * 4 < waves + 4
""" % (counts, kind))
