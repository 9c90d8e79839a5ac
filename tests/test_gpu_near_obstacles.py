"""The check kernels' choice of near obstacles: scenes whose obstacle count sits at the edges of the
64-obstacle chunks, batches at the edges of the states-per-wave split, a NaN state among free ones,
and a scene that shrinks.  Verdicts, costs and motions equal the oracle's bit for bit (the cull only
skips what cannot touch, so there is no tolerance)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import oracle
from isaac_sim_ros2_humble_amd import native, workloads
from isaac_sim_ros2_humble_amd.scene import Scene, box_record, capsule_record, cylinder_record, random_rotation

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def robots(fr3, fetch):
    native.init(0)
    return {"fr3": native.Robot(fr3), "fetch": native.Robot(fetch)}


def _scene(model, count, seed):
    """`count` obstacles of all four kinds, every fourth a capsule."""
    rng = np.random.default_rng(seed)
    lo, hi, keep = workloads.workspace(model)
    ncap = count // 4
    s = workloads.random_scene(rng, count - ncap, lo, hi, keep)
    caps = [capsule_record(rng.uniform([0.4, 0.4, 0.1], [1.0, 1.0, 1.4]), random_rotation(rng), rng.uniform(0.02, 0.08),
                           rng.uniform(0.1, 0.5)) for _ in range(ncap)]
    s.capsules = np.array(caps, np.float32).reshape(-1, 7)
    assert s.num_obstacles == count
    return s


@pytest.mark.parametrize("name,count,n", [
    ("fr3", 1, 1), ("fr3", 63, 65), ("fr3", 64, 2048), ("fr3", 65, 2049), ("fetch", 127, 300), ("fetch", 129, 4097),
    ("fr3", 200, 131073)])
def test_checks_at_chunk_edges(name, count, n, robots, request):
    m = request.getfixturevalue(name)
    orc = request.getfixturevalue("orc_" + name)
    scene = _scene(m, count, seed=count)
    q = workloads.uniform_configs(m, n, np.random.default_rng(n))
    ns, osc = native.Scene(scene), oracle.OracleScene(scene)
    v = native.check_states(robots[name], ns, q)
    vo, co, _, _ = oracle.check(orc, osc, q, want_cost=True, nthreads=8)
    assert np.array_equal(v, vo)
    cost, vc = native.state_costs(robots[name], ns, q)
    assert np.array_equal(cost, co) and np.array_equal(vc, vo)
    k = min(n // 2, 200)
    if k:
        ok, ln = native.check_edges(robots[name], ns, q[:k], q[k:2 * k], 0.02)
        oko, lno = oracle.edges(orc, osc, q[:k], q[k:2 * k], 0.02)
        assert np.array_equal(ok, oko) and np.array_equal(ln, lno)


def test_nan_state_does_not_hide_obstacles(fr3, orc_fr3, robots):
    # the lanes that the waves' balls are centred on (16, 48) hold NaN or infinite states
    scene = _scene(fr3, 64, seed=3)
    q = workloads.uniform_configs(fr3, 1 << 18, np.random.default_rng(4))
    q[16::64] = np.nan
    q[48::128, 3] = np.inf
    keep = np.isfinite(q).all(axis=1)
    v = native.check_states(robots["fr3"], native.Scene(scene), q)
    vo, _, _, _ = oracle.check(orc_fr3, oracle.OracleScene(scene), q[keep], nthreads=8)
    assert np.array_equal(v[keep], vo)


def test_scene_update_to_fewer_obstacles(fr3, orc_fr3, robots):
    big, small = _scene(fr3, 130, seed=5), _scene(fr3, 37, seed=6)
    ns = native.Scene(big)
    q = workloads.uniform_configs(fr3, 3000, np.random.default_rng(7))
    for s in (big, small, big):
        keep = Scene(spheres=s.spheres[:len(big.spheres)], boxes=s.boxes[:len(big.boxes)],
                     cylinders=s.cylinders[:len(big.cylinders)], capsules=s.capsules[:len(big.capsules)])
        ns.update(keep)
        vo, co, _, _ = oracle.check(orc_fr3, oracle.OracleScene(keep), q, want_cost=True, nthreads=8)
        cost, v = native.state_costs(robots["fr3"], ns, q)
        assert np.array_equal(v, vo) and np.array_equal(cost, co)
        assert np.array_equal(native.check_states(robots["fr3"], ns, q), vo)


@pytest.mark.parametrize("name,kind,count", [
    ("fr3", "boxes", 31), ("fr3", "boxes", 65), ("fetch", "cylinders", 33), ("fr3", "capsules", 32), ("fetch", "spheres", 64),
    ("fr3", "mixed", 97), ("fetch", "mixed", 64)])
def test_lanes_walk_their_own_obstacles(name, kind, count, robots, request):
    # states far from each other among obstacles within reach: nearly every link of a wave is near nearly
    # every obstacle, the waves whose lanes take their own; 70,001 states are the last wave's remainder too
    m = request.getfixturevalue(name)
    rng = np.random.default_rng(count)

    def pos():
        return rng.uniform([0.45, -0.8, 0.3], [1.0, 0.8, 1.2])
    make = {"boxes": lambda: box_record(pos(), random_rotation(rng), rng.uniform(0.01, 0.05, 3)),
            "cylinders": lambda: cylinder_record(pos(), random_rotation(rng), rng.uniform(0.01, 0.05), rng.uniform(0.05, 0.2)),
            "capsules": lambda: capsule_record(pos(), random_rotation(rng), rng.uniform(0.01, 0.05), rng.uniform(0.05, 0.2)),
            "spheres": lambda: np.append(pos(), rng.uniform(0.01, 0.06))}
    kinds = list(make) if kind == "mixed" else [kind]
    parts = {k: np.array([make[k]() for _ in range(len(range(i, count, len(kinds))))], np.float32) for i, k in enumerate(kinds)}
    scene = Scene(**parts)
    assert scene.num_obstacles == count
    q = workloads.uniform_configs(m, 70001, np.random.default_rng(count + 1))
    vo, _, _, _ = oracle.check(request.getfixturevalue("orc_" + name), oracle.OracleScene(scene), q, nthreads=8)
    assert 0 < vo.sum() < len(vo)
    assert np.array_equal(native.check_states(robots[name], native.Scene(scene), q), vo)


def _reachable(model, kind, count, seed):
    """`count` obstacles of a kind (or all four) among the arm's links."""
    rng = np.random.default_rng(seed)

    def pos():
        return rng.uniform([0.4, -0.8, 0.2], [1.0, 0.8, 1.3])
    make = {"boxes": lambda: box_record(pos(), random_rotation(rng), rng.uniform(0.01, 0.06, 3)),
            "cylinders": lambda: cylinder_record(pos(), random_rotation(rng), rng.uniform(0.01, 0.06), rng.uniform(0.05, 0.2)),
            "capsules": lambda: capsule_record(pos(), random_rotation(rng), rng.uniform(0.01, 0.06), rng.uniform(0.05, 0.2)),
            "spheres": lambda: np.append(pos(), rng.uniform(0.01, 0.07))}
    kinds = list(make) if kind == "mixed" else [kind]
    scene = Scene(**{k: np.array([make[k]() for _ in range(len(range(i, count, len(kinds))))], np.float32)
                     for i, k in enumerate(kinds)})
    assert scene.num_obstacles == count
    return scene


def _path(model, n, seed, step=0.005):
    """States along straight lines between random configurations, `step` rad apart."""
    knots = workloads.uniform_configs(model, 4 + int(n * step / 2.0) * 2, np.random.default_rng(seed)).astype(np.float64)
    at = np.concatenate([[0.0], np.cumsum(np.linalg.norm(np.diff(knots, axis=0), axis=1))])
    s = np.arange(n) * step
    assert s[-1] < at[-1]
    return np.stack([np.interp(s, at, knots[:, j]) for j in range(model.dof)], axis=1).astype(np.float32)


def _states(model, form, n, seed):
    """Unrelated states, states along a path, waves of the one beside waves of the other, or both in
    every wave.  The waves of these batches hold 16, 32 or 64 states."""
    spread, path = workloads.uniform_configs(model, n, np.random.default_rng(seed)), _path(model, n, seed)
    run = {"scattered": 1 << 30, "path": 0, "waves": 64, "within": 11}[form]
    return np.where((np.arange(n) // run % 2 == 0)[:, None], spread, path) if run else path


def _oracle_rows(orc, osc, q):
    with ThreadPoolExecutor(8) as ex:
        return np.concatenate(list(ex.map(lambda p: oracle.constraint_costs(orc, osc, p), np.array_split(q, 32))), axis=1)


@pytest.mark.parametrize("form,name,kind,count,n", [
    ("scattered", "fr3", "boxes", 31, 20001), ("scattered", "fetch", "boxes", 65, 17003), ("scattered", "fetch", "cylinders", 33, 20001),
    ("scattered", "fr3", "cylinders", 65, 33001), ("scattered", "fr3", "capsules", 32, 20001), ("scattered", "fetch", "capsules", 66, 17003),
    ("scattered", "fetch", "spheres", 64, 20001), ("scattered", "fr3", "spheres", 97, 66001), ("scattered", "fr3", "mixed", 130, 40003),
    ("scattered", "fetch", "mixed", 97, 40003), ("path", "fr3", "mixed", 97, 70003), ("path", "fetch", "mixed", 130, 17003),
    ("path", "fetch", "boxes", 65, 34001), ("path", "fr3", "spheres", 33, 17003), ("waves", "fr3", "mixed", 130, 70003),
    ("waves", "fetch", "mixed", 97, 34001), ("within", "fr3", "mixed", 65, 34001), ("within", "fetch", "mixed", 130, 17003),
    ("scattered", "fr3", "mixed", 0, 17003), ("path", "fetch", "mixed", 1, 17003)])
def test_large_batches_of_either_form(form, name, kind, count, n, robots, request):
    # verdicts, centres, total costs and every constraint's row of the launches whose waves choose between
    # taking their near obstacles one by one and letting each lane walk its own
    m = request.getfixturevalue(name)
    orc = request.getfixturevalue("orc_" + name)
    scene = _reachable(m, kind, count, seed=count + 2)
    q = _states(m, form, n, seed=n + count)
    ns, osc = native.Scene(scene), oracle.OracleScene(scene)
    vo, co, centres, _ = oracle.check(orc, osc, q, want_cost=True, want_centres=True, nthreads=8)
    rows = _oracle_rows(orc, osc, q)
    assert 0 < vo.sum() < n
    assert all((r > 0).any() for r, c in zip(rows, scene.counts) if c > 1)
    v, c = native.check_states(robots[name], ns, q, want_centres=True)
    assert np.array_equal(v, vo) and np.array_equal(c, centres)
    assert np.array_equal(native.check_states(robots[name], ns, q), vo)
    cost, vc = native.state_costs(robots[name], ns, q)
    assert np.array_equal(cost, co) and np.array_equal(vc, vo)
    parts, total, vp = native.constraint_costs(robots[name], ns, q)
    assert np.array_equal(parts, rows) and np.array_equal(total, co) and np.array_equal(vp, vo)


@pytest.mark.parametrize("form,name", [("scattered", "fr3"), ("path", "fr3"), ("scattered", "fetch"), ("path", "fetch")])
def test_costs_beside_nan_states(form, name, robots, request):
    # the lanes that the waves' balls are centred on, and others, hold NaN or infinite states
    m = request.getfixturevalue(name)
    orc = request.getfixturevalue("orc_" + name)
    scene = _reachable(m, "mixed", 70, seed=12)
    q = _states(m, form, 70001, seed=13)
    q[16::128] = np.nan
    q[48::192, 3] = np.inf
    q[5::100, 0] = -np.inf
    q[7::90, 5] = np.nan
    keep = np.isfinite(q).all(axis=1)
    ns, osc = native.Scene(scene), oracle.OracleScene(scene)
    vo, co, _, _ = oracle.check(orc, osc, q[keep], want_cost=True, nthreads=8)
    assert np.array_equal(native.check_states(robots[name], ns, q)[keep], vo)
    parts, total, v = native.constraint_costs(robots[name], ns, q)
    assert np.array_equal(parts[:, keep], _oracle_rows(orc, osc, q[keep]))
    assert np.array_equal(total[keep], co) and np.array_equal(v[keep], vo)


@pytest.mark.parametrize("name,count,n", [
    ("fr3", 5, 511), ("fr3", 5, 513), ("fetch", 5, 1025), ("fr3", 20, 2305), ("fetch", 20, 5377), ("fr3", 33, 7001), ("fetch", 33, 16385),
    ("fr3", 12, 16383), ("fr3", 130, 31749), ("fetch", 15, 32257), ("fr3", 15, 32768), ("fr3", 15, 32769)])
@pytest.mark.parametrize("form", ["scattered", "path"])
def test_any_number_of_states_per_wave(form, name, count, n, robots, request):
    # 1, 2, 3, 4, 7, 16, 17, 32, 63 and 64 states a wave, the last wave's run cut short: centres into a guarded
    # buffer, verdicts, every constraint's row
    m = request.getfixturevalue(name)
    orc = request.getfixturevalue("orc_" + name)
    scene = _reachable(m, "mixed", count, seed=count + 3)
    q = _states(m, form, n, seed=n)
    ns, osc = native.Scene(scene), oracle.OracleScene(scene)
    vo, co, centres, _ = oracle.check(orc, osc, q, want_cost=True, want_centres=True, nthreads=8)
    guard = np.float32(-77.25)
    dq = native.DeviceBuffer.from_array(q)
    dc = native.DeviceBuffer.from_array(np.full(n * m.S * 3 + 8, guard, np.float32))
    dv = native.DeviceBuffer.from_array(np.full(n + 8, 9, np.uint8))
    native.check(native.lib().mp_check_states(robots[name].h, ns.h, dq.ptr, n, dv.ptr + 3, dc.ptr + 4, None), "mp_check_states")
    v, c = dv.to_array(np.uint8, (n + 8,)), dc.to_array(np.float32, (n * m.S * 3 + 8,))
    assert np.array_equal(v[3:n + 3], vo) and (v[:3] == 9).all() and (v[n + 3:] == 9).all()
    assert np.array_equal(c[1:-7].reshape(n, m.S, 3), centres) and c[0] == guard and (c[-7:] == guard).all()
    parts, total, vp = native.constraint_costs(robots[name], ns, q)
    assert np.array_equal(total, co) and np.array_equal(vp, vo) and np.array_equal(parts, _oracle_rows(orc, osc, q))
