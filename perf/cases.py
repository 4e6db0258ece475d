"""Performance cases of the collision-check library.

Each case is one call (or one short sequence) that a program using gpuprm_amd
makes: exact point checks and edge checks of one scene, batches of scenes, the
radius search, the planner, and the surrogate model's inference and gradients.
Scenes are the library's seeded workloads (1: 4-DOF arm, 8 boxes; 2: 6-DOF
arm, 16 hulls of 12 points; 3: 7-DOF arm, 32 hulls of 16 points; 5: 7-DOF arm,
8..128 hulls of 8..24 points).  ``listed()`` names the cases, ``draw(rng)``
gives further ones of the same ranges, ``prepare`` makes the inputs,
``run`` makes the call, ``work`` counts what it cannot do without, and
``exact`` gives computed numbers in 64 bits.
"""
import math
import tempfile

import numpy as np
import torch

import gpuprm_amd

SCENE_SEED = 2024
DQ = 0.01
NDOF = {1: 4, 2: 6, 3: 7, 5: 7}
# obstacles of the fixed-size workloads; workload 5 draws 8..128
OBSTACLES = {1: 8, 2: 16, 3: 32, 5: 68}
HIDDEN = 256


def listed():
    return [
        # a planner that checks its step's candidates one at a time: each a host
        # array in, a code out
        {"name": "point_single_4dof_32", "kind": "single", "workload": 1, "n": 32},
        # one planner step's candidates, an odd count, resident in HBM
        {"name": "points_7dof_3001", "kind": "points", "workload": 3, "n": 3001},
        # the 4-DOF scene's usual batch
        {"name": "points_4dof_65536", "kind": "points", "workload": 1, "n": 65536},
        # labelling configurations for the surrogate, the largest call
        {"name": "points_7dof_4m", "kind": "points", "workload": 3, "n": 1 << 22},
        # one step of the reference's planner at its default of 32 new nodes:
        # edges as host arrays, through copies and wait
        {"name": "edges_host_4dof_32", "kind": "edges_host", "workload": 1, "n": 32, "length": 1.0},
        # a planner step's candidate edges within its connection radius
        {"name": "edges_local_7dof_20011", "kind": "edges_local", "workload": 3, "n": 20011, "length": 0.5},
        # a whole roadmap: the k nearest neighbours of 16,384 free vertices
        {"name": "edges_roadmap_6dof_16384", "kind": "edges_knn", "workload": 2, "n": 16384, "k": 10},
        # many scenes in one graph-replayed batch, 1k-64k configurations each
        {"name": "batch_points_16_scenes", "kind": "batch", "workload": 5, "scenes": 16, "least": 1000, "most": 65536},
        # neighbour lists of a roadmap's vertices
        {"name": "radius_6dof_20000", "kind": "radius", "ndof": 6, "n": 20000, "radius": 1.1},
        # a planning task from start to goal
        {"name": "plan_6dof_2048", "kind": "plan", "workload": 2, "num": 2048, "radius": 1.0},
        # the surrogate ranks many configurations
        {"name": "predict_7dof_1m", "kind": "predict", "workload": 3, "n": 1 << 20},
        # forward, loss and backward of a training batch, gradients read back
        {"name": "gradients_6dof_32768", "kind": "gradients", "workload": 2, "n": 32768},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "points", "points", "edges_host", "edges_local", "edges_knn", "batch", "radius",
                       "plan", "predict", "gradients"])
    wl = rng.choice([1, 2, 3])
    if kind == "single":
        return {"kind": kind, "workload": wl, "n": _spread(rng, 16, 64)}
    if kind == "points":
        return {"kind": kind, "workload": wl, "n": _spread(rng, 16, 1 << 22)}
    if kind == "edges_host":
        return {"kind": kind, "workload": wl, "n": _spread(rng, 24, 2048), "length": round(rng.uniform(0.5, 1.5), 3)}
    if kind == "edges_local":
        return {"kind": kind, "workload": wl, "n": _spread(rng, 100, 20011), "length": round(rng.uniform(0.2, 1.0), 3)}
    if kind == "edges_knn":
        return {"kind": kind, "workload": rng.choice([1, 2]), "n": _spread(rng, 500, 16384), "k": rng.choice([5, 8, 10])}
    if kind == "batch":
        return {"kind": kind, "workload": 5, "scenes": rng.randint(2, 16), "least": 1000,
                "most": _spread(rng, 2000, 65536)}
    if kind == "radius":
        nd = rng.choice([4, 6, 7])
        n = _spread(rng, 500, 20000)
        # about eight neighbours a vertex: the ball's volume over the cube's
        ball = math.pi ** (nd / 2) / math.gamma(nd / 2 + 1)
        return {"kind": kind, "ndof": nd, "n": n, "radius": round((8 * (2 * math.pi) ** nd / (n * ball)) ** (1 / nd), 3)}
    if kind == "plan":
        return {"kind": kind, "workload": 2, "num": _spread(rng, 512, 2048), "radius": 1.0}
    if kind == "predict":
        return {"kind": kind, "workload": wl, "n": _spread(rng, 64, 1 << 20)}
    return {"kind": kind, "workload": wl, "n": _spread(rng, 256, 32768)}


_dirs, _spaces = {}, {}


def _scene_dir(workload, seed):
    if (workload, seed) not in _dirs:
        _dirs[workload, seed] = gpuprm_amd.generate_scene(workload, seed, tempfile.mkdtemp(prefix="gprm_perf_"))
    return _dirs[workload, seed]


def _space(workload, seed=SCENE_SEED):
    """The scene's checker, which a program makes once and keeps."""
    if (workload, seed) not in _spaces:
        sp = gpuprm_amd.RobotConfigspace(_scene_dir(workload, seed), DQ, 1 << 20)
        sp.init(0, 1)
        _spaces[workload, seed] = sp
    return _spaces[workload, seed]


def _uniform(g, shape):
    return (torch.rand(shape, generator=g, device="cuda") * 2 - 1) * math.pi


def _free(space, g, n):
    """n collision-free configurations (ndof, n), uniform by rejection."""
    out, have = [], 0
    while have < n:
        q = _uniform(g, (space.dim(), max(4096, 2 * n)))
        code = torch.zeros(q.shape[1], dtype=torch.int32, device="cuda")
        space.indicator_dev(q, code)
        out.append(q[:, code == 0])
        have += out[-1].shape[1]
    return torch.cat(out, dim=1)[:, :n].contiguous()


def _local_edges(space, g, n, length):
    """n edges of at most `length` between free configurations, their ends
    uniform in a ball around their starts."""
    nd = space.dim()
    S, E, have = [], [], 0
    while have < n:
        a = _free(space, g, 2 * n)
        d = torch.randn(a.shape, generator=g, device="cuda")
        r = length * torch.rand(a.shape[1], generator=g, device="cuda") ** (1.0 / nd)
        b = (a + d / d.norm(dim=0) * r).clamp(-math.pi, math.pi).contiguous()
        code = torch.zeros(b.shape[1], dtype=torch.int32, device="cuda")
        space.indicator_dev(b, code)
        S.append(a[:, code == 0])
        E.append(b[:, code == 0])
        have += S[-1].shape[1]
    return torch.cat(S, dim=1)[:, :n].contiguous(), torch.cat(E, dim=1)[:, :n].contiguous()


def _knn_count(n, k):
    return 11 * n * k // 20


def _knn_edges(space, g, n, k):
    """Undirected k-nearest-neighbour edges of n free configurations: of their
    0.6 n k or so, an evenly spread 0.55 n k, so that calls of one size hold
    as many edges."""
    V = _free(space, g, n)
    X = V.t().double()
    nbr = []
    for i in range(0, n, 1024):
        d2 = sum((X[i:i + 1024, None, c] - X[None, :, c]) ** 2 for c in range(X.shape[1]))
        j = torch.arange(d2.shape[0], device="cuda")
        d2[j, j + i] = math.inf
        nbr.append(torch.topk(d2, k, dim=1, largest=False).indices)
    J = torch.cat(nbr).flatten()
    I = torch.arange(n, device="cuda").repeat_interleave(k)
    key = torch.unique(torch.minimum(I, J) * n + torch.maximum(I, J))
    m = _knn_count(n, k)
    key = key[torch.arange(m, device="cuda") * key.shape[0] // m]
    return V[:, key // n].contiguous(), V[:, key % n].contiguous()


def _model(case, seed, batch):
    """A surrogate as training leaves it: weights a few times their initial
    scale, so that probabilities are spread over (0, 1)."""
    m = gpuprm_amd.Surrogate(ndof=NDOF[case["workload"]], batch=batch, seed=seed)
    m.set_params(2.0 * m.get_params())
    return m


def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = {"kind": kind}
    if kind in ("single", "points", "edges_host", "edges_local", "edges_knn", "plan"):
        s["space"] = _space(case["workload"])
        nd = s["space"].dim()
    if kind == "single":
        s["q"] = list(_uniform(g, (case["n"], nd)).cpu().numpy())
    elif kind == "points":
        s["q"] = _uniform(g, (nd, case["n"]))
        s["res"] = torch.zeros(case["n"], dtype=torch.int32, device="cuda")
    elif kind == "edges_host":
        a, b = _local_edges(s["space"], g, case["n"], case["length"])
        s["qs"], s["qe"] = a.cpu().numpy().ravel(), b.cpu().numpy().ravel()
        s["res"] = np.zeros(case["n"], np.int32)
        s["n"] = case["n"]
    elif kind in ("edges_local", "edges_knn"):
        if kind == "edges_local":
            s["qs"], s["qe"] = _local_edges(s["space"], g, case["n"], case["length"])
        else:
            s["qs"], s["qe"] = _knn_edges(s["space"], g, case["n"], case["k"])
        s["res"] = torch.zeros(s["qs"].shape[1], dtype=torch.int32, device="cuda")
    elif kind == "batch":
        sizes = np.random.default_rng(case["scenes"]).integers(case["least"], case["most"] + 1, case["scenes"])
        s["batch"] = gpuprm_amd.SceneBatch([_space(5, 1000 + i) for i in range(case["scenes"])])
        s["qs"] = [_uniform(g, (7, int(n))) for n in sizes]
        s["res"] = [torch.zeros(int(n), dtype=torch.int32, device="cuda") for n in sizes]
    elif kind == "radius":
        s["nodes"] = _uniform(g, (case["ndof"], case["n"]))
        s["hi"] = np.full(case["ndof"], np.pi, np.float32)
        s["radius"] = case["radius"]
        # the lists in arrays of a fixed size, -1 beyond the pairs found
        s["cap"] = 32 * case["n"]
        s["out"] = (np.full(s["cap"], -1, np.int32), np.full(s["cap"], -1, np.int32), np.zeros(s["cap"], np.float32))
    elif kind == "plan":
        # start and goal: free, and well apart
        V = _free(s["space"], g, 64).t().cpu().numpy()
        d = np.linalg.norm(V - V[0], axis=1)
        s["start"], s["goal"] = V[0], V[int(np.argmax(d > 4.0)) or int(np.argmax(d))]
        s["path"] = np.zeros((1024, nd), np.float32)  # zeros beyond the path
        s["args"] = dict(num=case["num"], D=case["radius"], max_nodes=1 << 18, max_steps=300, seed=seed)
    elif kind == "predict":
        s["model"] = _model(case, seed, 64)
        s["q"] = _uniform(g, (NDOF[case["workload"]], case["n"]))
        s["out"] = torch.zeros(case["n"], dtype=torch.float32, device="cuda")
    elif kind == "gradients":
        s["model"] = _model(case, seed, case["n"])
        s["q"] = _uniform(g, (NDOF[case["workload"]], case["n"]))
        s["codes"] = torch.zeros(case["n"], dtype=torch.int32, device="cuda")
        _space(case["workload"]).indicator_dev(s["q"], s["codes"])
    else:
        raise ValueError(kind)
    return s


def run(s):
    kind = s["kind"]
    if kind == "single":
        return np.array([s["space"].indicator(q) for q in s["q"]])
    if kind == "points":
        s["space"].indicator_dev(s["q"], s["res"])
        return s["res"]
    if kind == "edges_host":
        s["space"].indicator2(s["qs"], s["qe"], s["res"], s["n"], s["n"])
        return s["res"] != 0  # the decision: which colliding sample's code is left open
    if kind in ("edges_local", "edges_knn"):
        st = s["space"].indicator2_dev(s["qs"], s["qe"], s["res"])
        return s["res"] != 0, int(st.samples_total)
    if kind == "batch":
        s["batch"].indicator_dev(s["qs"], s["res"], use_graph=True)
        return s["res"]
    if kind == "radius":
        found = gpuprm_amd.radius_neighbours(s["nodes"], s["nodes"], -s["hi"], s["hi"], s["radius"], cap=s["cap"])
        for to, x in zip(s["out"], found):
            to[:len(x)] = x
        return s["out"]
    if kind == "plan":
        r, path = s["space"].prm_solve(s["start"], s["goal"], **s["args"])
        if path is not None:
            s["path"][:len(path)] = path
        return {"path": s["path"], "length": r.path_len, "found": r.found, "steps": r.steps,
                "nodes": r.nodes_left + r.nodes_right, "edges_free": r.edges_free, "point_checks": r.point_checks}
    if kind == "predict":
        s["model"].predict(s["q"], s["out"])
        return s["out"]
    return s["model"].gradients(s["q"], s["codes"])


# Operations that any exact check needs: per joint the sine and cosine and
# one frame product, per pair of polytopes at least one separating direction
# (a difference, two projections, a comparison).
_JOINT, _PAIR = 110, 20


def _check_flops(workload):
    nd = NDOF[workload]
    pairs = nd * OBSTACLES[workload] + (nd - 1) * (nd - 2) // 2
    return nd * _JOINT + pairs * _PAIR


def work(case):
    kind = case["kind"]
    if kind == "radius":
        nd, n = case["ndof"], case["n"]
        ball = math.pi ** (nd / 2) / math.gamma(nd / 2 + 1) * case["radius"] ** nd
        found = n * (1 + n * ball / (2 * math.pi) ** nd)
        return {"bytes": 4 * nd * n + 12 * found, "flops": 3 * nd * found}
    wl = case["workload"]
    nd = NDOF[wl]
    if kind in ("predict", "gradients"):
        n = case["n"]
        forward = 2.0 * n * (nd * HIDDEN + 2 * HIDDEN * HIDDEN + HIDDEN)
        weights = nd * HIDDEN + 2 * HIDDEN * HIDDEN + 4 * HIDDEN + 1
        if kind == "predict":
            return {"bytes": 4.0 * n * (nd + 1) + 2 * weights, "flops": forward}
        return {"bytes": 4.0 * n * (nd + 1) + 6 * weights, "flops": 3 * forward}
    if kind in ("single", "points"):
        return {"bytes": 4.0 * case["n"] * (nd + 1), "flops": 1.0 * case["n"] * _check_flops(wl)}
    if kind == "batch":
        n = case["scenes"] * 0.5 * (case["least"] + case["most"])
        return {"bytes": 4.0 * n * (nd + 1), "flops": n * _check_flops(wl)}
    if kind == "plan":
        # at least one step's candidates and one edge of each
        n = case["num"]
        return {"bytes": 4.0 * n * (nd + 1), "flops": n * (1 + 0.5 * case["radius"] / DQ) * _check_flops(wl)}
    if kind == "edges_knn":
        # mean length: the ball that holds half of the k neighbours
        edges = _knn_count(case["n"], case["k"])
        ball = math.pi ** (nd / 2) / math.gamma(nd / 2 + 1)
        length = (0.5 * case["k"] * 2 * (2 * math.pi) ** nd / (case["n"] * ball)) ** (1 / nd)
    else:
        edges, length = case["n"], case["length"] * nd / (nd + 1)
    return {"bytes": 4.0 * edges * (2 * nd + 1), "flops": edges * (1 + length / DQ) * _check_flops(wl)}


def _mlp64(model, q, ndof):
    """(inputs, weights, biases, pre-activations, activations) in 64 bits."""
    P = torch.from_numpy(model.get_params()).double().cuda()
    sizes = [(HIDDEN, 16), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN,), (1,)]
    parts, at = [], 0
    for sh in sizes:
        k = math.prod(sh)
        parts.append(P[at:at + k].reshape(sh))
        at += k
    W, b = parts[0::2], parts[1::2]
    x = torch.zeros(q.shape[1], 16, dtype=torch.float64, device="cuda")
    x[:, :ndof] = q.t().double() / math.pi
    pre, act = [], [x]
    for l in range(3):
        pre.append(act[-1] @ W[l].t() + b[l])
        act.append(pre[-1] * torch.sigmoid(pre[-1]))
    return W, b, pre, act


def exact(case, seed):
    kind = case["kind"]
    if kind == "radius":
        # the distances of the pairs closer than the radius, by (query, node)
        X = prepare(case, seed)["nodes"].t().double()
        out = []
        for i in range(0, X.shape[0], 2048):
            d2 = torch.zeros(min(2048, X.shape[0] - i), X.shape[0], dtype=torch.float64, device="cuda")
            for c in range(X.shape[1]):
                d2 += (X[i:i + 2048, None, c] - X[None, :, c]) ** 2
            out.append(d2[d2 < float(np.float32(case["radius"]) * np.float32(case["radius"]))])
        out.append(torch.zeros(32 * case["n"] - sum(len(x) for x in out), dtype=torch.float64, device="cuda"))
        return None, None, torch.cat(out)
    if kind == "predict":
        s = prepare(case, seed)
        out = []
        for i in range(0, case["n"], 1 << 17):
            W, b, _, act = _mlp64(s["model"], s["q"][:, i:i + (1 << 17)], NDOF[case["workload"]])
            out.append(torch.sigmoid(act[3] @ W[3] + b[3]))
        return torch.cat(out)
    if kind == "gradients":
        s = prepare(case, seed)
        W, b, pre, act = _mlp64(s["model"], s["q"], NDOF[case["workload"]])
        z = act[3] @ W[3] + b[3]
        y = (s["codes"] != 0).double()
        loss = (torch.clamp(z, min=0) - z * y + torch.log1p(torch.exp(-z.abs()))).mean()
        dz = (torch.sigmoid(z) - y) / case["n"]
        grads = [(act[3] * dz[:, None]).sum(0), dz.sum().reshape(1)]
        dH = dz[:, None] * W[3][None, :]
        for l in (2, 1, 0):
            sg = torch.sigmoid(pre[l])
            dA = dH * (sg * (1 + pre[l] * (1 - sg)))
            grads = [dA.t() @ act[l], dA.sum(0)] + grads
            dH = dA @ W[l]
        return torch.cat([x.flatten() for x in grads]), loss
    return None
