"""Cases for timing this package's public entry points: FK and collision checks of batches of
configurations, motions, nearest neighbours, planning queries and the device roadmap.

Workloads are the package's own (workloads.py: FR3 and Fetch, box / cylinder / capsule / sphere
scenes) with inputs drawn from a seed.  Batches of configurations live in device memory, as a program
that keeps its states on the GPU has them; planning queries start from and end in host memory,
which is where the planner's calls take and leave them.
"""
import math

import numpy as np
import torch

from isaac_sim_ros2_humble_amd import native, workloads
from isaac_sim_ros2_humble_amd.model import load_robot

RES = 0.02           # motion resolution (rad), the planner's default
TREE_CAPACITY = 65536
PASSES = 20          # of the roadmap planner: nearly every task is solved in three
# launch shapes that the package's tuner picks on an MI355X: batches, and one query per launch
BATCH_SHAPE = {"team_waves": 2, "waves": 1024, "teams_per_query": 32, "lanes_per_iteration": 32}
SINGLE_SHAPE = {"team_waves": 4, "waves": 256, "lanes_per_iteration": 64}

_robots = {}


def robot(name):
    """Model and native handle of a robot; a program creates each once."""
    if name not in _robots:
        model = load_robot(name)
        _robots[name] = (model, native.Robot(model))
    return _robots[name]


# --------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # validity and sphere centres of a million sampled states in a cluttered cube: building a
        # roadmap or a reachability map offline (the package's FK + collision benchmark)
        {"name": "check_fr3_1m", "kind": "check", "robot": "fr3", "n": 1 << 20, "obstacles": 64, "centres": True, "states": "uniform"},
        # re-checking densified paths at 0.005 rad, verdicts only: neighbouring states lie close together
        {"name": "check_fetch_paths", "kind": "check", "robot": "fetch", "n": 100003, "obstacles": 120, "centres": False, "states": "paths"},
        # the states of one planner step or one goal sampler: the smallest call, latency counts
        {"name": "check_fr3_small", "kind": "check", "robot": "fr3", "n": 257, "obstacles": 20, "centres": False, "states": "uniform"},
        # per-constraint penetration costs, as an optimiser of trajectories or goals reads them
        {"name": "costs_fr3", "kind": "costs", "robot": "fr3", "n": 200001, "obstacles": 64},
        # sphere centres alone, for a caller with a world model of its own
        {"name": "fk_fr3_1m", "kind": "fk", "robot": "fr3", "n": 1 << 20},
        # 4x4 pose of every link, for attaching objects, cameras or task-space constraints
        {"name": "poses_fetch", "kind": "poses", "robot": "fetch", "n": 150001},
        # motion checks between free states, as a roadmap's edges or a path shortcutter's candidates
        {"name": "edges_fr3", "kind": "edges", "robot": "fr3", "m": 5003, "obstacles": 64, "length": 6.0},
        # nearest nodes of a large tree to a batch of samples
        {"name": "nn_tree", "kind": "nn", "nodes": 50021, "queries": 256, "dof": 7},
        # planning queries one launch each, the latency a robot waits for
        {"name": "solve_fr3_each", "kind": "solve", "robot": "fr3", "queries": 16, "obstacles": 20},
        # 256 mixed queries in one launch: the package's headline throughput workload
        {"name": "batch_mixed_256", "kind": "batch", "robot": "mixed", "queries": 256},
        # reproducible planning (one team per query): the same paths for the same seeds
        {"name": "exclusive_mixed_64", "kind": "exclusive", "robot": "mixed", "queries": 64},
        # roadmap planning from creation to the graph read back, evaluation settings of the RRG planner
        {"name": "roadmap_fr3", "kind": "roadmap", "robot": "fr3", "tasks": 4, "samples": 60, "travel": 6.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["check", "check", "check", "costs", "fk", "poses", "edges", "edges", "nn", "nn", "solve", "batch",
                       "exclusive", "roadmap"])
    arm = rng.choice(["fr3", "fetch"])
    if kind == "check":
        return {"kind": kind, "robot": arm, "n": _log(rng, 1, 500000), "obstacles": _log(rng, 5, 200),
                "centres": rng.random() < 0.3, "states": rng.choice(["uniform", "paths"])}
    if kind == "costs":
        return {"kind": kind, "robot": arm, "n": _log(rng, 1, 200000), "obstacles": _log(rng, 5, 200)}
    if kind == "fk" or kind == "poses":
        return {"kind": kind, "robot": arm, "n": _log(rng, 1, 500000)}
    if kind == "edges":
        return {"kind": kind, "robot": arm, "m": _log(rng, 10, 5000), "obstacles": _log(rng, 5, 200),
                "length": round(rng.uniform(0.3, 6.0), 2)}
    if kind == "nn":
        return {"kind": kind, "nodes": _log(rng, 10, TREE_CAPACITY), "queries": _log(rng, 1, 256), "dof": rng.choice([6, 7, 8])}
    if kind == "solve":
        return {"kind": kind, "robot": arm, "queries": _log(rng, 2, 16), "obstacles": _log(rng, 5, 60)}
    if kind == "batch":
        return {"kind": kind, "robot": rng.choice(["fr3", "fetch", "mixed"]), "queries": _log(rng, 16, 256)}
    if kind == "exclusive":
        return {"kind": kind, "robot": rng.choice(["fr3", "fetch", "mixed"]), "queries": _log(rng, 4, 64)}
    return {"kind": kind, "robot": "fr3", "tasks": _log(rng, 1, 4), "samples": _log(rng, 16, 250),
            "travel": round(rng.uniform(1.0, 6.0), 2)}


# ------------------------------------------------------------------------------------------- inputs
def _bounds(model):
    return (torch.tensor(model.active_lower.astype(np.float64), device="cuda"),
            torch.tensor(model.active_upper.astype(np.float64), device="cuda"))


def _uniform(model, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    lo, hi = _bounds(model)
    return (lo + torch.rand(n, model.dof, generator=g, device="cuda", dtype=torch.float64) * (hi - lo)).float()


def _path_states(model, n, seed):
    """States along a piecewise-linear tour through random configurations, 0.005 rad apart."""
    knots = _uniform(model, 4 + n // 400, seed).double()
    seg = knots[1:] - knots[:-1]
    cum = torch.cat([torch.zeros(1, device="cuda", dtype=torch.float64), torch.cumsum(seg.norm(dim=1), 0)])
    s = torch.remainder(torch.arange(n, device="cuda", dtype=torch.float64) * 0.005, cum[-1] * 0.999999)
    k = (torch.searchsorted(cum, s, right=True) - 1).clamp(0, len(seg) - 1)
    t = (s - cum[k]) / (cum[k + 1] - cum[k])
    return (knots[k] + t[:, None] * seg[k]).float()


def _scene(model, obstacles, seed):
    """64 obstacles: the FK + collision benchmark's cube with capsules; otherwise a mixed scene."""
    if obstacles == 64:
        return workloads.c2_scene(seed=seed)
    lo, hi, keep = workloads.workspace(model)
    return workloads.random_scene(np.random.default_rng(seed), obstacles, lo, hi, keep)


def _free_motions(model, rob, scene, m, length, rng):
    """m motions of at most `length` rad between collision-free states."""
    a_all, b_all, have = [], [], 0
    while have < m:
        q = workloads.uniform_configs(model, 1 << 14, rng)
        q = q[native.check_states(rob, scene, q).astype(bool)]
        h = len(q) // 2
        a, b = q[:h], q[h:2 * h]
        d = np.linalg.norm(b - a, axis=1, keepdims=True)
        b = (a + (b - a) * np.minimum(1.0, length / d)).astype(np.float32)
        ok = native.check_states(rob, scene, b).astype(bool)
        a_all.append(a[ok])
        b_all.append(b[ok])
        have += int(ok.sum())
    return np.concatenate(a_all)[:m], np.concatenate(b_all)[:m]


def _pairs(model, rob, nscene, rng, count, batch):
    """Up to `count` collision-free (start, goal) pairs, half of them with a blocked straight line."""
    return workloads.sample_pairs(model, nscene, rng, lambda m, s, q: native.check_states(rob, s, q),
                                  lambda m, s, a, b: native.check_edges(rob, s, a, b, RES)[0], count, batch=batch, max_rounds=4)


def _queries(which, count, rng):
    """Planning queries over scenes with 5 to 200 obstacles, two per scene."""
    out = []
    while len(out) < count:
        name = which if which != "mixed" else ("fr3", "fetch")[int(rng.integers(2))]
        model, rob = robot(name)
        lo, hi, keep = workloads.workspace(model)
        ns = native.Scene(workloads.random_scene(rng, workloads.log_uniform_count(rng), lo, hi, keep))
        got = _pairs(model, rob, ns, rng, 2, 1024)
        if len(got) == 2:
            out += [(rob, ns, s, g) for s, g in got]
    return out[:count]


def _request(queries, max_path=4096):
    rob, sc, st, gl = zip(*queries)
    return native.BatchRequest(list(rob), list(sc), list(st), list(gl), max_path=max_path)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    native.init()
    if kind in ("check", "costs", "fk", "poses"):
        model, rob = robot(case["robot"])
        n = case["n"]
        q = (_path_states if case.get("states") == "paths" else _uniform)(model, n, seed)
        s = {"kind": kind, "robot": rob, "q": q, "n": n}
        if kind == "fk":
            s["out"] = torch.empty(n, model.S, 3, device="cuda")
        elif kind == "poses":
            s["out"] = torch.empty(n, model.L, 4, 4, device="cuda")
        else:
            s["scene"] = native.Scene(_scene(model, case["obstacles"], seed))
            s["verdict"] = torch.empty(n, device="cuda", dtype=torch.uint8)
            if kind == "costs":
                s["parts"] = torch.empty(len(native.COST_KINDS), n, device="cuda")
                s["cost"] = torch.empty(n, device="cuda")
            else:
                s["centres"] = torch.empty(n, model.S, 3, device="cuda") if case["centres"] else None
        return s
    if kind == "edges":
        model, rob = robot(case["robot"])
        scene = native.Scene(_scene(model, case["obstacles"], seed))
        a, b = _free_motions(model, rob, scene, case["m"], case["length"], rng)
        return {"kind": kind, "robot": rob, "scene": scene, "m": case["m"], "a": torch.from_numpy(a).cuda(),
                "b": torch.from_numpy(b).cuda(), "ok": torch.empty(case["m"], device="cuda", dtype=torch.uint8),
                "len": torch.empty(case["m"], device="cuda")}
    if kind == "nn":
        g = torch.Generator(device="cuda").manual_seed(seed)
        tree = torch.zeros(case["dof"], TREE_CAPACITY, device="cuda")
        tree[:, :case["nodes"]] = torch.rand(case["dof"], case["nodes"], generator=g, device="cuda") * 5.8 - 2.9
        q = torch.rand(case["queries"], case["dof"], generator=g, device="cuda") * 5.8 - 2.9
        return {"kind": kind, "tree": tree, "q": q, "nodes": case["nodes"], "dof": case["dof"],
                "idx": torch.empty(case["queries"], device="cuda", dtype=torch.int32)}
    if kind == "roadmap":
        model, rob = robot(case["robot"])
        tasks = []
        while len(tasks) < case["tasks"]:
            c = rng.uniform([-0.8, -0.8, 0.0], [0.8, 0.8, 1.2], size=(20, 3))
            c = c[np.hypot(c[:, 0], c[:, 1]) > 0.3]
            r = rng.uniform(0.03, 0.1, size=len(c))
            ns = native.Scene(workloads.Scene(spheres=np.concatenate([c, r[:, None]], axis=1).astype(np.float32)))
            pair = _pairs(model, rob, ns, rng, 2, 1024)[-1:]
            if pair:
                tasks.append((ns, pair[0][0], pair[0][1]))
        return {"kind": kind, "robot": rob, "tasks": tasks, "samples": case["samples"], "travel": case["travel"], "seed": seed % 1000}
    if kind == "solve":
        model, rob = robot(case["robot"])
        if case["robot"] == "fr3" and case["obstacles"] == 20:
            scene = native.Scene(workloads.c1_scene(seed=seed))
        else:
            scene = native.Scene(_scene(model, case["obstacles"], seed))
        queries = [(rob, scene, a, b) for a, b in _pairs(model, rob, scene, rng, 2 * case["queries"], 4096)]
    else:
        queries = _queries(case["robot"], case["queries"] + (8 if kind == "batch" else 0), rng)
    if kind == "exclusive":
        params = native.default_params(seed=seed % 1000, exclusive=1, max_iterations=3000, max_path=512, team_waves=2,
                                       lanes_per_iteration=32)
        return {"kind": kind, "request": _request(queries, 512), "params": params}
    # queries that the reproducible mode solves, with room for an unlucky run: which of them are solved
    # does not depend on the teams' timing (their paths do)
    found = _request(queries).solve(native.default_params(seed=seed % 1000 + 7, exclusive=1, team_waves=2,
                                                          lanes_per_iteration=32)).code == 1
    queries = [q for q, f in zip(queries, found) if f]
    want = min(case["queries"], len(queries))
    shape = SINGLE_SHAPE if kind == "solve" else BATCH_SHAPE
    return {"kind": kind, "request": _request(queries[:want]),
            "params": native.default_params(seed=seed % 1000, max_iterations=40000, **shape)}


# ---------------------------------------------------------------------------------------- one pass
def _p(t):
    return None if t is None else t.data_ptr()


def _rows(a, most):
    """`a` in a buffer of `most` rows, as a caller with room for the largest roadmap keeps it."""
    out = np.zeros((most,) + a.shape[1:], a.dtype)
    out[:len(a)] = a
    return out


def run(s):
    L, kind = native.lib(), s["kind"]
    if kind == "check":
        native.check(L.mp_check_states(s["robot"].h, s["scene"].h, _p(s["q"]), s["n"], _p(s["verdict"]), _p(s["centres"]), None),
                     "mp_check_states")
        return {"verdict": s["verdict"], "centres": s["centres"]}
    if kind == "costs":
        native.check(L.mp_constraint_costs(s["robot"].h, s["scene"].h, _p(s["q"]), s["n"], _p(s["parts"]), _p(s["cost"]),
                                           _p(s["verdict"]), None), "mp_constraint_costs")
        return {"parts": s["parts"], "cost": s["cost"], "verdict": s["verdict"]}
    if kind == "fk":
        native.check(L.mp_fk_spheres(s["robot"].h, _p(s["q"]), s["n"], _p(s["out"]), None), "mp_fk_spheres")
        return {"centres": s["out"]}
    if kind == "poses":
        native.check(L.mp_fk_link_poses(s["robot"].h, _p(s["q"]), s["n"], _p(s["out"]), None), "mp_fk_link_poses")
        return {"poses": s["out"]}
    if kind == "edges":
        native.check(L.mp_check_edges(s["robot"].h, s["scene"].h, _p(s["a"]), _p(s["b"]), s["m"], RES, _p(s["ok"]), _p(s["len"]),
                                      None), "mp_check_edges")
        return {"ok": s["ok"], "len": s["len"]}
    if kind == "nn":
        native.check(L.mp_nn_argmin(_p(s["tree"]), s["nodes"], TREE_CAPACITY, s["dof"], _p(s["q"]), len(s["q"]), _p(s["idx"]), None),
                     "mp_nn_argmin")
        return {"idx": s["idx"]}
    if kind == "roadmap":
        out = []
        for k, (scene, start, goal) in enumerate(s["tasks"]):
            rm = native.Roadmap(s["robot"], scene, start[None], goal[None], samples_per_iteration=s["samples"],
                                max_travel_distance=s["travel"], resolution=RES, seed=s["seed"] + k)
            for _ in range(PASSES):
                if rm.iterate():
                    break
            g = rm.read()
            rm.close()
            most = 2 + 2 * PASSES * s["samples"]
            out.append({"solved": g["solved"], "passes": g["passes"]} | {
                f: _rows(g[f], most) for f in ("vertices", "groups", "edges", "weights", "start_members", "goal_members")})
        return out
    req, params = s["request"], s["params"]
    if kind == "exclusive":
        r = req.solve(params)
        return {"code": r.code, "iterations": r.iterations, "start_tree": r.start_tree, "goal_tree": r.goal_tree,
                "checked": r.configs_checked, "waypoints": r.num_waypoints, "paths": req.block}
    # the teams of a query race, so a path's inner waypoints are another sample of the same search on
    # each run; its status and its two ends are not
    r = req.solve_each(params) if kind == "solve" else req.solve(params)
    rows = req.block.reshape(req.nq, req.stride)
    at = np.arange(16)
    inside = (at < req.dof[:, None]) & (r.code == 1)[:, None]
    last = np.maximum(r.num_waypoints - 1, 0)[:, None] * req.dof[:, None] + at
    return {"code": r.code, "first": np.where(inside, rows[:, :16], 0),
            "last": np.where(inside, np.take_along_axis(rows, last, axis=1), 0)}


# ----------------------------------------------------------------------------------------- the work
def _state_flops(model, obstacles):
    """What one state's check cannot do without: its FK, its spheres, a look at each obstacle."""
    return sum({1: 130, 2: 87, 5: 63}.get(int(t), 0) for t in model.joint_types[1:]) + 18 * model.S + 11 * obstacles


def work(case):
    kind = case["kind"]
    if kind == "nn":
        return {"bytes": 4 * case["dof"] * (case["nodes"] + case["queries"]) + 4 * case["queries"],
                "flops": 3 * case["dof"] * case["nodes"] * case["queries"]}
    model = load_robot("fr3" if case["robot"] == "mixed" else case["robot"])
    if kind in ("check", "costs", "fk", "poses"):
        out = {"check": 1 + (12 * model.S if case.get("centres") else 0), "costs": 4 * 7 + 1, "fk": 12 * model.S,
               "poses": 64 * model.L}[kind]
        per = _state_flops(model, case.get("obstacles", 0)) - (18 * model.S if kind == "poses" else 0)
        return {"bytes": case["n"] * (4 * model.dof + out), "flops": case["n"] * per}
    if kind == "edges":  # half of the longest motion on average; a blocked one ends early
        return {"bytes": case["m"] * (8 * model.dof + 5),
                "flops": case["m"] * case["length"] / 4 / RES * _state_flops(model, case["obstacles"])}
    # planning: the states along a path of some 5 rad have to be checked for every query
    count = case["tasks"] if kind == "roadmap" else case["queries"]
    return {"bytes": count * (288 + 20 * 4 * model.dof), "flops": count * 5.0 / RES * _state_flops(model, 20)}


# ------------------------------------------------------------------------------- results in 64 bits
def _frames(model, q):
    """Link poses [L] as (rotation [n,3,3], translation [n,3]) in float64."""
    n, out, a = len(q), [], 0
    for i in range(model.L):
        if i == 0:
            out.append((torch.eye(3, device="cuda", dtype=torch.float64).expand(n, 3, 3), torch.zeros(n, 3, device="cuda", dtype=torch.float64)))
            continue
        R, t = out[int(model.parents[i])]
        kind = int(model.joint_types[i])
        if kind == 0:
            out.append((R, t))
            continue
        O = torch.tensor(model.joint_origins[i].reshape(4, 4), device="cuda", dtype=torch.float64)
        t = t + R @ O[:3, 3]
        R = R @ O[:3, :3]
        if kind != 5:
            if model.active[i]:
                v, a = q[:, a].double(), a + 1
            else:
                v = torch.full((n,), float(model.defaults[i]), device="cuda", dtype=torch.float64)
            ax = torch.tensor(model.joint_axes[i], device="cuda", dtype=torch.float64)
            if kind == 2:
                t = t + (R @ ax) * v[:, None]
            else:
                ax = ax / ax.norm()
                z = torch.zeros((), device="cuda", dtype=torch.float64)
                K = torch.stack([torch.stack([z, -ax[2], ax[1]]), torch.stack([ax[2], z, -ax[0]]), torch.stack([-ax[1], ax[0], z])])
                Rq = torch.eye(3, device="cuda", dtype=torch.float64) + torch.sin(v)[:, None, None] * K + (1 - torch.cos(v))[:, None, None] * (K @ K)
                R = torch.bmm(R.contiguous(), Rq.contiguous())
        out.append((R, t))
    return out


def _centres(model, frames):
    return torch.stack([frames[int(l)][1] + frames[int(l)][0] @ torch.tensor(model.sphere_pos[s], device="cuda", dtype=torch.float64)
                        for s, l in enumerate(model.sphere_link)], dim=1)


def _costs(model, scene, c):
    """Per-constraint penetration costs [6][n] of sphere centres c [n,S,3]."""
    r = torch.tensor(model.sphere_radius, device="cuda", dtype=torch.float64)
    zero = torch.zeros(len(c), device="cuda", dtype=torch.float64)
    rows = [zero.clone() for _ in range(6)]
    for ob in torch.tensor(scene.spheres, dtype=torch.float64).cuda():
        rows[0] += (r + ob[3] - (c - ob[:3]).norm(dim=2)).clamp(min=0).sum(1)
    for k, obs in ((1, scene.boxes), (2, scene.cylinders)):
        for ob in torch.tensor(obs, dtype=torch.float64).cuda():
            local = (c - ob[:3]) @ ob[3:12].reshape(3, 3)
            if k == 1:
                d = (local - local.maximum(ob[12:15]).minimum(ob[15:18])).norm(dim=2)
            else:
                dx, dz = local[..., :2].norm(dim=2) - ob[12], local[..., 2].abs() - ob[13] / 2
                d = torch.hypot(dx.clamp(min=0), dz.clamp(min=0)) + dx.maximum(dz).clamp(max=0)
            rows[k] += (r - d).clamp(min=0).sum(1)
    for ob in torch.tensor(scene.capsules, dtype=torch.float64).cuda():
        v = ob[3:6] - ob[:3]
        t = (((c - ob[:3]) @ v) / (v @ v)).clamp(0, 1)
        rows[3] += (r + ob[6] - (c - ob[:3] - t[..., None] * v).norm(dim=2)).clamp(min=0).sum(1)
    links = model.sphere_link
    for i in range(model.S):
        j = [j for j in range(i + 1, model.S) if links[j] != links[i] and model.enabled[links[i], links[j]]]
        if j:
            rows[4] += (r[i] + r[j] - (c[:, j] - c[:, i:i + 1]).norm(dim=2)).clamp(min=0).sum(1)
    return torch.stack(rows)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("check", "costs", "fk", "poses", "edges") or (kind == "check" and not case["centres"]):
        return None
    s = prepare(case, seed)
    torch.cuda.synchronize()
    if kind == "edges":
        return {"ok": None, "len": (s["a"].double() - s["b"].double()).norm(dim=1)}
    model, _ = robot(case["robot"])
    got = []
    for q in s["q"].split(1 << 16):
        f = _frames(model, q)
        if kind == "poses":
            T = torch.zeros(len(q), model.L, 4, 4, device="cuda", dtype=torch.float64)
            for i, (R, t) in enumerate(f):
                T[:, i, :3, :3], T[:, i, :3, 3], T[:, i, 3, 3] = R, t, 1.0
            got.append(T)
        elif kind == "costs":
            got.append(_costs(model, s["scene"].scene, _centres(model, f)))
        else:
            got.append(_centres(model, f))
    if kind == "costs":
        parts = torch.cat(got, dim=1)
        return {"parts": parts, "cost": parts.sum(0), "verdict": None}
    v = torch.cat(got)
    return {"verdict": None, "centres": v} if kind == "check" else {"centres" if kind == "fk" else "poses": v}
