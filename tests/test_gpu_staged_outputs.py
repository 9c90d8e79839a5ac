"""Kernels that stage their rows through LDS or share a scan among waves, at the sizes where that can go
wrong: sphere centres and link poses of ragged batches into buffers aligned to one float only, with
guard values around them, and nearest nodes at the edges of the waves' shares.  Results equal the
oracle's (or numpy's argmin over the same float32 sums) exactly."""
import numpy as np
import pytest

import oracle
from isaac_sim_ros2_humble_amd import native, workloads

pytestmark = pytest.mark.gpu
GUARD = np.float32(-77.25)


@pytest.fixture(scope="module")
def robots(fr3, fetch):
    native.init(0)
    return {"fr3": native.Robot(fr3), "fetch": native.Robot(fetch)}


def _run(fn, robot, q, width, shift):
    """The kernel's rows written `shift` floats into a guarded buffer."""
    n = len(q)
    buf = native.DeviceBuffer.from_array(np.full(n * width + 8, GUARD, np.float32))
    dq = native.DeviceBuffer.from_array(q)
    native.check(fn(robot.h, dq.ptr, n, buf.ptr + 4 * shift, None), fn.__name__)
    out = buf.to_array(np.float32, (n * width + 8,))
    assert np.all(out[:shift] == GUARD) and np.all(out[shift + n * width:] == GUARD)
    return out[shift:shift + n * width]


@pytest.mark.parametrize("name", ["fr3", "fetch"])
@pytest.mark.parametrize("n,shift", [(1, 0), (7, 1), (31, 3), (33, 2), (63, 0), (64, 1), (65, 0), (257, 3)])
def test_ragged_rows(name, n, shift, robots, request):
    m, orc, r = request.getfixturevalue(name), request.getfixturevalue("orc_" + name), robots[name]
    q = workloads.uniform_configs(m, n, np.random.default_rng(n))
    L = native.lib()
    c = _run(L.mp_fk_spheres, r, q, 3 * m.S, shift).reshape(n, m.S, 3)
    assert np.array_equal(c, orc.fk32(q))
    p = _run(L.mp_fk_link_poses, r, q, 16 * m.L, shift).reshape(n, m.L, 4, 4)
    assert np.array_equal(p, orc.link_poses32(q))


@pytest.mark.parametrize("dof", [1, 3, 7, 8, 9, 16])
@pytest.mark.parametrize("n,nq", [(1, 1), (255, 3), (256, 2), (257, 5), (4096, 1), (4097, 33), (20011, 4)])
def test_nearest_nodes(dof, n, nq):
    rng = np.random.default_rng(100 * dof + n)
    tree = rng.uniform(-2, 2, (n, dof)).astype(np.float32)
    tree[n // 2:] = tree[:n - n // 2]  # every distance twice: ties go to the lower index
    if n > 300:
        tree[5::97] = np.nan  # unwritten slots are never selected
    q = rng.uniform(-2, 2, (nq, dof)).astype(np.float32)
    got = native.nn_argmin(tree, q, capacity=n + 11)
    for k in range(nq):
        d = np.sum((tree.astype(np.float64) - q[k].astype(np.float64)) ** 2, axis=1)
        d[np.isnan(d)] = np.inf
        assert got[k] == oracle.nn(tree, q[k])
        # float32 sums of `dof` terms: the chosen node is a nearest one to within their rounding, and
        # the first of its equals
        assert d[got[k]] <= d.min() * (1 + 2 * (dof + 2) * 2.0 ** -24) + 1e-30
        assert got[k] == np.nonzero((tree == tree[got[k]]).all(axis=1))[0][0]


def test_no_nodes_and_no_numbers():
    q = np.zeros((3, 7), np.float32)
    assert np.array_equal(native.nn_argmin(np.zeros((0, 7), np.float32), q), [-1, -1, -1])
    assert np.array_equal(native.nn_argmin(np.full((300, 7), np.nan, np.float32), q), [0x7fffffff] * 3)


@pytest.mark.parametrize("n,nq", [(9, (1 << 22) + 5), (4100, (1 << 22) + 2), (4100, 9000001)])
def test_nearest_nodes_of_millions_of_queries(n, nq):
    # coordinates on a grid: distances are whole numbers, exact in float32, with many ties
    rng = np.random.default_rng(n)
    tree = rng.integers(-40, 41, (n, 2)).astype(np.float32)
    at = rng.integers(-45, 46, (nq, 2))
    side = np.arange(-45, 46)
    grid = np.stack(np.meshgrid(side, side, indexing="ij"), axis=-1).reshape(-1, 2)
    want = np.concatenate([np.argmin(((g[:, None, :] - tree[None]) ** 2).sum(2), axis=1) for g in np.array_split(grid, 64)])
    got = native.nn_argmin(tree, at.astype(np.float32))
    assert np.array_equal(got, want[(at[:, 0] + 45) * 91 + at[:, 1] + 45])
