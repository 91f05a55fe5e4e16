"""The measured workloads: what programs that use this framework have it do,
through its public entry points, with sizes from the smallest frame to the
largest batch.

A case is a dict of plain values.  Its kind is

  "scene"       a batch of worlds stepped `steps` times, then read back:
                the state of every body of every world (and, with `overlay`,
                the contacts and boxes the demo draws);
  "infer"       the warm-start network on `rows` feature rows on the GPU
                (device addresses in and out, nothing allocated);
  "forward"     the same network on `rows` rows of host memory;
  "gradient"    the gradient of its loss over `rows` rows of host memory;
  "train"       `steps` Adam steps on mini-batches of `batch` rows of a
                training set that lies on the GPU; the updated weights.

`prepare` makes worlds from the seed and steps them untimed (`settle`) into
the regime the case stands for; `run` is one pass on them and continues from
where the last one ended, as a simulation does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from shapes_amd import engine, scenes


SOLVERS = {"ordered": engine.SOLVER_ORDERED_F64, "coloured": engine.SOLVER_COLORED_F32}
WARMS = {"zero": engine.WARM_ZERO, "learned": engine.WARM_LEARNED}
BROADPHASES = {"auto": engine.BROADPHASE_AUTO, "scan": engine.BROADPHASE_SCAN,
               "grid": engine.BROADPHASE_GRID, "grid1": engine.BROADPHASE_GRID_1,
               "grid16": engine.BROADPHASE_GRID_16}
PILE_LAYERS = 60   # piles start as columns of at most this many bodies
SHAPES = [(14, 128), (128,), (128, 128), (128,), (128, 128), (128,), (128, 2), (2,)]


def _scene(name, scene, size, solver, iterations, settle, steps, **kw):
    c = {"name": name, "kind": "scene", "scene": scene, "size": size, "worlds": 1,
         "solver": solver, "iterations": iterations, "warm": "zero", "threads": 0,
         "broadphase": "auto", "settle": settle, "steps": steps, "graph": False,
         "overlay": False}
    c.update(kw)
    return c


def listed():
    return [
        # one frame of an interactive program: the 55-box pyramid, drop-in
        # solver, one update, the bodies read back to draw them
        _scene("pyramid_55_frame", "pyramid", 10, "ordered", 4, 150, 1),
        # the same frame of the mixed circle and box scene with the demo's
        # overlays on: contacts of the world as it stands, and its boxes
        _scene("balls_100_overlay", "balls", 10, "ordered", 2, 100, 1, overlay=True),
        # the reference's own benchmark: 900 boxes in columns, 10 steps
        _scene("stacks_900_run", "stacks", 30, "ordered", 2, 50, 10),
        # one large settled pile with the drop-in solver
        _scene("pile_8192_ordered", "pile", 8192, "ordered", 8, 400, 5, graph=True),
        # the same pile with the coloured solver, 1024 lanes as the autotuner picks
        _scene("pile_8192_coloured", "pile", 8192, "coloured", 8, 400, 20, graph=True,
               threads=1024),
        # the largest single world: its velocities do not fit on one CU
        _scene("pile_32768_coloured", "pile", 32768, "coloured", 4, 500, 10, graph=True,
               threads=1024),
        # a batch of rollouts of small uneven worlds (8 to 1024 bodies) with
        # the drop-in solver, all final states read back
        _scene("worlds_512_ordered", "worlds", 1024, "ordered", 6, 170, 50, graph=True,
               worlds=512),
        # more of them with the coloured solver, one wavefront per world
        _scene("worlds_2048_coloured", "worlds", 1024, "coloured", 6, 170, 100, graph=True,
               worlds=2048, threads=64, broadphase="grid1"),
        # piles in a batch, coloured solver with the learned warm start: the
        # headline configuration of the benchmark with fewer, smaller piles
        _scene("piles_256_learned", "piles", 8192, "coloured", 4, 300, 10, graph=True,
               worlds=256, threads=1024, broadphase="grid1", warm="learned"),
        # the network alone: a step's cache misses on the GPU (odd count)
        {"name": "infer_4099", "kind": "infer", "rows": 4099},
        # evaluating the model on a held-out set in host memory
        {"name": "forward_100003", "kind": "forward", "rows": 100003},
        # training: mini-batches of 4096 as the training program uses
        {"name": "train_4096", "kind": "train", "rows": 262144, "batch": 4096, "steps": 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "small", "pile", "pile", "worlds", "worlds", "piles", "infer",
                       "host", "train"])
    if kind == "small":
        scene = rng.choice(["pyramid", "balls", "stacks"])
        size = {"pyramid": rng.randint(3, 20), "balls": rng.randint(4, 20),
                "stacks": rng.randint(8, 40)}[scene]
        c = _scene("", scene, size, rng.choice(["ordered", "ordered", "coloured"]),
                   rng.randint(2, 8), rng.randint(0, 200), rng.choice([1, 1, 2, 5, 10]),
                   overlay=rng.random() < 0.3, graph=rng.random() < 0.3)
    elif kind == "pile":
        ordered = rng.random() < 0.4
        c = _scene("", "pile", _log(rng, 500, 12000 if ordered else 30000),
                   "ordered" if ordered else "coloured", rng.randint(2, 8),
                   rng.randint(150, 400), rng.randint(1, 8), graph=True,
                   threads=0 if ordered else rng.choice([0, 256, 512, 1024]))
    elif kind == "worlds":
        ordered = rng.random() < 0.4
        c = _scene("", "worlds", rng.randint(200, 1024), "ordered" if ordered else "coloured",
                   rng.randint(2, 8), rng.randint(60, 170), rng.randint(10, 60), graph=True,
                   worlds=_log(rng, 16, 512 if ordered else 1500),
                   threads=0 if ordered else rng.choice([0, 64, 64, 256]),
                   broadphase=rng.choice(["auto", "grid1", "grid"]))
    elif kind == "piles":
        c = _scene("", "piles", rng.randint(3000, 8000), "coloured", rng.randint(2, 6),
                   rng.randint(150, 300), rng.randint(2, 8), graph=True,
                   worlds=_log(rng, 8, 200), threads=rng.choice([512, 1024]),
                   broadphase="grid1", warm=rng.choice(["zero", "learned"]))
    elif kind == "infer":
        c = {"kind": "infer", "rows": _log(rng, 1, 65536)}
    elif kind == "host":
        c = {"kind": rng.choice(["forward", "gradient"]), "rows": _log(rng, 1, 100000)}
    else:
        c = {"kind": "train", "rows": _log(rng, 8192, 262144),
             "batch": 64 * rng.randint(1, 96), "steps": rng.randint(1, 20)}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ scenes

def _widen(w):
    """The floor (body 0) twice as wide: bodies stay on it however long a
    run goes on."""
    w.hull_x[:4] *= 2.0
    return w


def _pile(rng, count, spacing, vel):
    cols = max(2, int(math.ceil(count / PILE_LAYERS)))
    if count < 20 * PILE_LAYERS:
        cols = max(2, int(math.ceil(math.sqrt(count))))
    return _widen(scenes.grid_world(rng, count, cols, spacing, 1.1, 0.0, vel=vel))


def _counts(lo, hi, n):
    """Log-uniform body counts, the same for every seed (the bodies differ)."""
    rng = np.random.Generator(np.random.Philox(lo))
    return np.rint(np.exp(rng.uniform(np.log(lo), np.log(hi), n))).astype(int)


def _worlds_of(case, seed):
    """(worlds, config) of a scene case."""
    rng = np.random.Generator(np.random.Philox(seed))
    size, it = case["size"], case["iterations"]
    cfg = scenes.SceneConfig(iterations=it)
    if case["scene"] == "pyramid":
        sc = scenes.pyramid(seed=seed, rows=size, iterations=it)
        return sc.worlds, sc.config
    if case["scene"] in ("balls", "stacks"):
        sc = (scenes.balls(dims=(size, size), iterations=it) if case["scene"] == "balls"
              else scenes.reference_stacks(dims=(size, size)))
        w = sc.worlds[0]
        w.vx[1:] += rng.uniform(-0.05, 0.05, w.n - 1)  # seeded: the scenes themselves are fixed
        return sc.worlds, scenes.SceneConfig(**{**sc.config.__dict__, "iterations": it})
    if case["scene"] == "pile":
        if size > 16384:  # the largest piles step at the pile batches' 1/120
            cfg = scenes.SceneConfig(iterations=it, dt=1.0 / 120.0)
        return [_pile(rng, size, 2.05, 1.0)], cfg
    if case["scene"] == "worlds":
        return [_widen(scenes.grid_world(rng, int(c), max(2, int(math.ceil(math.sqrt(c)))), 2.1,
                                         2.0, 0.5)) for c in _counts(8, size, case["worlds"])], cfg
    cfg = scenes.SceneConfig(iterations=it, dt=1.0 / 120.0)
    return [_widen(scenes.grid_world(rng, int(c), int(math.ceil(c / 20)), 2.05, 1.05, 0.0, vel=0.2))
            for c in _counts(2048, size, case["worlds"])], cfg


def _batch(case, worlds, cfg, solver, threads):
    b = engine.make_batch(worlds, cfg, solver=SOLVERS[solver], warm_start=WARMS[case["warm"]],
                          max_pairs_per_body=0 if case["scene"] != "piles" else 4,
                          broadphase=BROADPHASES[case["broadphase"]], solver_threads=threads)
    if case["warm"] == "learned":
        b.set_mlp(np.load(engine.HERE + "/warmstart_mlp.npy"))
    return b


def _prepare_scene(case, seed):
    worlds, cfg = _worlds_of(case, seed)
    settle = case["settle"]
    if case["scene"] == "pile" and case["solver"] == "ordered" and settle:
        # a large pile settles with the coloured solver; the drop-in solver
        # takes over its state and warm-start cache
        b = _batch(case, worlds, cfg, "coloured", 1024)
        b.step_async(settle, use_graph=True)
        b.sync()
        w, s, (keys, lam) = worlds[0], b.bodies(0), b.cache(0)
        b.close()
        w.px, w.py, w.theta, w.vx, w.vy, w.omega = (s[:, k].copy() for k in range(6))
        b = _batch(case, worlds, cfg, case["solver"], case["threads"])
        b.set_cache(0, keys, lam)
        settle = 2
    else:
        b = _batch(case, worlds, cfg, case["solver"], case["threads"])
    if case["graph"]:
        b.step_async(settle, use_graph=True)
        b.sync()
    elif settle:
        b.step(settle)
    return {"case": case, "batch": b}


def _run_scene(state):
    case, b = state["case"], state["batch"]
    if case["graph"]:
        b.step_async(case["steps"], use_graph=True)
        b.sync()
    else:
        b.step(case["steps"])
    out = {"bodies": np.concatenate([b.bodies(w) for w in range(b.n_worlds)])}
    if case["overlay"]:
        b.probe_contacts()
        out.update(b.contacts())
        # into the drawing program's arrays, which have a fixed length
        for k, a in out.items():
            if k != "bodies":
                out[k] = np.zeros((4 * b.sizes[0] + 64,) + a.shape[1:], a.dtype)
                out[k][:len(a)] = a[:len(out[k])]
        out["slots"], out["boxes"] = b.aabbs()
    return out


def _scene_sizes(case):
    """(bodies, vertices, contacts) a scene has, as far as its sizes say."""
    n = case["size"]
    mean = lambda lo, hi: (hi - lo) / math.log(hi / lo)  # noqa: E731  log-uniform counts
    bodies = {"pyramid": n * (n + 1) // 2, "balls": n * n, "stacks": n * n, "pile": n,
              "worlds": case["worlds"] * mean(8, n), "piles": case["worlds"] * mean(2048, n)}
    nb = float(bodies[case["scene"]])
    verts = {"pyramid": 4.0, "stacks": 4.0, "balls": 2.0, "worlds": 4.75}.get(case["scene"], 5.5)
    conts = {"balls": 1.5}.get(case["scene"], 2.0)
    return nb, nb * verts, nb * conts


# ----------------------------------------------------------------- network

def _features(rng, n):
    """Rows as contact generation makes them: unit normal, 10 x depth,
    closing velocities, log1p of the inverse masses and inertias of 3-8-gons,
    lever arms, mean friction."""
    a = rng.uniform(0, 2 * np.pi, n)
    f = np.empty((n, 14))
    f[:, 0], f[:, 1] = np.cos(a), np.sin(a)
    f[:, 2] = 10.0 * np.minimum(rng.exponential(0.03, n), 0.5)
    f[:, 3] = -np.abs(rng.standard_t(3, n)) * 0.6
    f[:, 4] = rng.standard_t(3, n) * 0.6
    r = rng.uniform(0.3, 1.0, (n, 2))
    m = 2.2 * r * r
    f[:, 5:7] = np.log1p(1.0 / m)
    f[:, 7:9] = np.log1p(1.0 / (0.4 * m * r * r))
    static = rng.uniform(size=n) < 0.05  # the floor
    f[static, 6] = 0.0
    f[static, 8] = 0.0
    b = rng.uniform(0, 2 * np.pi, (n, 2))
    f[:, 9], f[:, 10] = r[:, 0] * np.cos(b[:, 0]), r[:, 0] * np.sin(b[:, 0])
    f[:, 11], f[:, 12] = r[:, 1] * np.cos(b[:, 1]), r[:, 1] * np.sin(b[:, 1])
    f[:, 13] = rng.uniform(0.2, 0.8, n)
    return np.clip(f, -20.0, 20.0).astype(np.float32)


def _targets(rng, f):
    n = np.maximum(0.0, -1.1 * f[:, 3] + 0.3 * f[:, 2] + 0.1 * rng.standard_normal(len(f)))
    t = np.clip(-0.7 * f[:, 4], -f[:, 13] * n, f[:, 13] * n)
    return np.stack([n, t], axis=1).astype(np.float32)


def _init_params(rng):
    """He-normal hidden weights, small output layer, zero biases."""
    parts = []
    for k, s in enumerate(SHAPES):
        if len(s) == 2:
            parts.append((rng.normal(0.0, math.sqrt(2.0 / s[0]), s) * (0.1 if k == 6 else 1.0)).ravel())
        else:
            parts.append(np.zeros(s))
    return np.concatenate(parts).astype(np.float32)


def _net_inputs(case, seed):
    rng = np.random.default_rng(seed)
    d = {"params": _init_params(rng), "feats": _features(rng, case["rows"])}
    if case["kind"] in ("gradient", "train"):
        d["targets"] = _targets(rng, d["feats"])
    if case["kind"] == "train":
        d["indices"] = rng.integers(0, case["rows"], case["steps"] * case["batch"]).astype(np.int32)
    return d


_STREAM = None


def _stream():
    """The one stream of the program's network calls on device memory."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


def prepare(case, seed):
    if case["kind"] == "scene":
        return _prepare_scene(case, seed)
    d = _net_inputs(case, seed)
    d["case"], d["net"] = case, engine.Mlp(d["params"])
    if case["kind"] == "infer":
        d["d_feats"] = torch.from_numpy(d["feats"]).cuda()
        d["d_out"] = torch.zeros((case["rows"], 2), device="cuda")
        d["stream"] = _stream().cuda_stream
    elif case["kind"] == "train":
        d["net"].set_data(d["feats"], d["targets"])
    return d


def run(state):
    case = state["case"]
    if case["kind"] == "scene":
        return _run_scene(state)
    net = state["net"]
    if case["kind"] == "infer":
        net.forward_noalloc(state["d_feats"].data_ptr(), case["rows"], state["d_out"].data_ptr(),
                            state["stream"])
        return state["d_out"]
    if case["kind"] == "forward":
        return net.forward(state["feats"])
    if case["kind"] == "gradient":
        grad, loss = net.gradient(state["feats"], state["targets"])
        return {"grad": grad, "loss": loss}
    net.train(state["indices"], case["batch"], 1e-3)
    return net.params()


def work(case):
    """Bytes: per step each body's state (48 B) read and written, its inverse
    masses, friction and restitution (32 B) and its hull read, each contact's
    cached key and impulses (24 B) read and written; the states read back.
    Operations: a contact's update is about 100 per sweep, a pair's separating
    axes about 4 per vertex pair.  Network: rows in and out, the weights, and
    two operations per weight and row (six with the gradient)."""
    if case["kind"] == "scene":
        nb, nv, nc = _scene_sizes(case)
        per = nb * (96 + 32) + nv * 16 + nc * 48
        flops = nc * 100 * (case["iterations"] + 1) + nb * 3 * 250
        return {"bytes": case["steps"] * per + 48 * nb, "flops": case["steps"] * flops}
    n, p = case["rows"], 35202
    if case["kind"] == "train":
        n = case["batch"] * case["steps"]
        return {"bytes": n * (32 + 8 + 4) + case["steps"] * p * 24, "flops": 6.0 * p * n}
    if case["kind"] == "gradient":
        return {"bytes": n * 64 + p * 8, "flops": 6.0 * p * n}
    return {"bytes": n * 64 + p * 4, "flops": 2.0 * p * n}


# ------------------------------------------------------- values in 64 bits

def _split(flat):
    out, o = [], 0
    for s in SHAPES:
        k = int(np.prod(s))
        out.append(flat[o:o + k].reshape(s))
        o += k
    return out


def _net64(p, x):
    w1, b1, w2, b2, w3, b3, w4, b4 = _split(p)
    silu = torch.nn.functional.silu
    return silu(silu(silu(x @ w1 + b1) @ w2 + b2) @ w3 + b3) @ w4 + b4


def exact(case, seed):
    """The network's outputs, gradients and updated weights in 64 bits.  A
    scene's steps have no such value here: their trajectories amplify every
    rounding, and the drop-in solver's results are defined to the bit by the
    order of its operations."""
    if case["kind"] == "scene":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    d = _net_inputs(case, seed)
    p = torch.from_numpy(d["params"]).to(dev, torch.float64)
    x = torch.from_numpy(d["feats"]).to(dev, torch.float64)
    if case["kind"] in ("infer", "forward"):
        return torch.cat([_net64(p, c) for c in x.split(16384)])
    t = torch.from_numpy(d["targets"]).to(dev, torch.float64)
    if case["kind"] == "gradient":
        p.requires_grad_(True)
        total = 0.0
        for xc, tc in zip(x.split(16384), t.split(16384)):
            loss = ((_net64(p, xc) - tc) ** 2).sum() / len(x)
            loss.backward()
            total += float(loss.detach())
        return {"grad": p.grad, "loss": total}
    idx = torch.from_numpy(d["indices"].astype(np.int64)).to(dev).reshape(case["steps"], -1)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for s in range(case["steps"]):
        q = p.clone().requires_grad_(True)
        ((_net64(q, x[idx[s]]) - t[idx[s]]) ** 2).sum().div(case["batch"]).backward()
        m = 0.9 * m + 0.1 * q.grad
        v = 0.999 * v + 0.001 * q.grad ** 2
        p = p - 1e-3 * (m / (1 - 0.9 ** (s + 1))) / ((v / (1 - 0.999 ** (s + 1))).sqrt() + 1e-8)
    return p
