"""The device-resident roadmap planner (mp_roadmap_*, the RRG extend-connect loop of
RRG.cpp:241-424) against the oracle's restatement of the same loop: with the same sample stream
both build the same roadmap bit for bit -- vertices, groups, edges, weights, member order, loop
index and travel distances -- including a run that outgrows the initial buffers."""
import numpy as np
import pytest

import oracle
from helpers import point_robot
from isaac_sim_ros2_humble_amd import native, workloads
from isaac_sim_ros2_humble_amd.scene import Scene, box_record

pytestmark = pytest.mark.gpu

_R = {}


def robot(m):
    if m.name not in _R:
        native.init(0)
        _R[m.name] = native.Robot(m)
    return _R[m.name]


def run(model, scene, starts, goals, k, travel, seed, offset, max_passes):
    r, ns = robot(model), native.Scene(scene)
    rm = native.Roadmap(r, ns, starts, goals, samples_per_iteration=k, max_travel_distance=travel, resolution=0.02,
                        seed=seed, sample_offset=offset)
    n = 0
    while n < max_passes and not rm.iterate():
        n += 1
    got = rm.read()
    rm.close()
    want = oracle.rrg(oracle.OracleRobot(model), oracle.OracleScene(scene), starts, goals, k, travel, 0.02, seed, offset,
                      max_passes=got["passes"], vcap=1 << 15)
    return got, want


def assert_same(got, want):
    for f in ("solved", "passes", "loop_index", "nv", "ne", "start_group", "goal_group", "travel_start", "travel_goal"):
        assert got[f] == want[f], (f, got[f], want[f])
    for f in ("vertices", "groups", "edges", "weights", "start_members", "goal_members"):
        assert np.array_equal(got[f], want[f]), f


def _pair(model, scene, rng):
    r, ns = robot(model), native.Scene(scene)
    pair = workloads.sample_pair(model, scene, rng, lambda m, s, q: native.check_states(r, ns, q),
                                 lambda m, s, a, b: native.check_edges(r, ns, a, b, 0.02)[0], want_free_line=False)
    assert pair is not None
    return pair


@pytest.mark.parametrize("name,k,travel", [("fr3", 60, 6.0), ("fetch", 30, 0.5)])
def test_roadmap_equals_oracle(name, k, travel, request):
    """evaluate_cudampl.cpp's settings (60 samples per pass, travel 6.0) on FR3 with 20 sphere
    obstacles, and the RRG defaults (30, 0.5) on Fetch in mixed clutter."""
    model = request.getfixturevalue(name)
    rng = np.random.default_rng(7)
    if name == "fr3":
        c = rng.uniform([-0.8, -0.8, 0.0], [0.8, 0.8, 1.2], size=(40, 3))
        c = c[np.hypot(c[:, 0], c[:, 1]) > 0.3][:20]
        scene = Scene(spheres=np.concatenate([c, rng.uniform(0.03, 0.1, (len(c), 1))], axis=1).astype(np.float32))
    else:
        scene = workloads.random_scene(rng, 40, *workloads.workspace(model))
    s, g = _pair(model, scene, rng)
    got, want = run(model, scene, s[None], g[None], k, travel, seed=11, offset=1000, max_passes=300)
    assert got["nv"] > 2
    assert_same(got, want)


def test_roadmap_grows_and_halves(rng):
    """A goal sealed in a box shell: the goal side halves its travel distance down to the floor
    and the start group keeps growing past the first buffers (256 samples a pass)."""
    m = point_robot(0.02, lim=1.0)
    walls = [box_record([0.5 + dx, dy, dz], np.eye(3), h) for dx, dy, dz, h in [
        (-0.15, 0, 0, [0.01, 0.2, 0.2]), (0.15, 0, 0, [0.01, 0.2, 0.2]), (0, -0.15, 0, [0.2, 0.01, 0.2]),
        (0, 0.15, 0, [0.2, 0.01, 0.2]), (0, 0, -0.15, [0.2, 0.2, 0.01]), (0, 0, 0.15, [0.2, 0.2, 0.01])]]
    scene = Scene(boxes=np.array(walls))
    s = np.array([[-0.5, 0.0, 0.0], [-0.6, 0.3, 0.1]], np.float32)
    g = np.array([[0.5, 0.0, 0.0]], np.float32)
    got, want = run(m, scene, s, g, 256, 1.0, seed=5, offset=0, max_passes=48)
    assert got["solved"] == 0 and got["nv"] > 4096  # past the initial 4096-vertex buffers
    assert_same(got, want)
    # the oracle's run halved the goal side's travel distance on the way (the shell blocks it)
    part = oracle.rrg(oracle.OracleRobot(m), oracle.OracleScene(scene), s, g, 256, 1.0, 0.02, 5, 0, max_passes=2)
    assert part["travel_goal"] == np.float32(0.5) and part["loop_index"] == 3


def test_roadmaps_one_after_another_and_together(fr3, orc_fr3):
    """Roadmaps take over the storage of destroyed ones: several starts and goals, then fewer, then two at
    once, then one larger than the storage kept, each equal to the oracle's and read twice alike."""
    rng = np.random.default_rng(3)
    scene = workloads.random_scene(rng, 20, *workloads.workspace(fr3))
    r, ns = robot(fr3), native.Scene(scene)
    q = workloads.uniform_configs(fr3, 40000, rng)
    q = q[native.check_states(r, ns, q).astype(bool)]
    osc = oracle.OracleScene(scene)

    def make(a, b, seed):
        return native.Roadmap(r, ns, q[:a], q[a:a + b], samples_per_iteration=33, max_travel_distance=1.5, resolution=0.02, seed=seed)

    def finish(rm, a, b, seed):
        for _ in range(4):
            if rm.iterate():
                break
        got, again = rm.read(), rm.read()
        rm.close()
        want = oracle.rrg(orc_fr3, osc, q[:a], q[a:a + b], 33, 1.5, 0.02, seed, 0, max_passes=got["passes"], vcap=1 << 15)
        assert_same(got, want)
        assert_same(again, want)

    for a, b, seed in ((5, 3, 1), (1, 1, 2), (2, 64, 3), (5000, 4000, 4), (1, 2, 5)):
        finish(make(a, b, seed), a, b, seed)
    first, second = make(3, 1, 6), make(1, 4, 7)
    finish(second, 1, 4, 7)
    finish(first, 3, 1, 6)


def test_large_roadmap_in_pieces(fr3, orc_fr3):
    """States of some megabytes enter and leave through host memory of one megabyte; any array may be left
    out of a read."""
    rng = np.random.default_rng(8)
    scene = workloads.random_scene(rng, 12, *workloads.workspace(fr3))
    r, ns = robot(fr3), native.Scene(scene)
    q = workloads.uniform_configs(fr3, 300001, rng)
    a, b = 50003, 30011
    q = q[native.check_states(r, ns, q).astype(bool)][:a + b]
    assert len(q) == a + b
    rm = native.Roadmap(r, ns, q[:a], q[a:], samples_per_iteration=64, max_travel_distance=0.7, resolution=0.02, seed=9)
    rm.iterate()
    got = rm.read()
    assert_same(got, oracle.rrg(orc_fr3, oracle.OracleScene(scene), q[:a], q[a:], 64, 0.7, 0.02, 9, 0, max_passes=1, vcap=1 << 18))
    assert got["nv"] > a + b and got["ne"] > 0
    names = ("vertices", "groups", "edges", "weights", "start_members", "goal_members")
    for wanted in [{n} for n in names] + [set(names) - {n} for n in names] + [set()]:
        out = {n: np.full_like(got[n], -7) for n in wanted}
        native.check(native.lib().mp_roadmap_read(rm.h, *[native._p(out.get(n)) for n in names]), "mp_roadmap_read")
        for n in wanted:
            assert np.array_equal(out[n], got[n]), n
    rm.close()
