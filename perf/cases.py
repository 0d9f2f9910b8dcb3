"""What the speed of this framework is measured on: the calls that a program which simulates
reaction-diffusion systems makes, from the smallest to the largest sizes in use.

A stepping case is one stretch of a simulation between two snapshots: `steps` accepted steps of every
realization through `Context.run`, then every realization's counts and statistics on the host.  A pass goes
on where the last one ended, as a run that writes snapshots does.  The training case is one call of
`Context.mlp_train`, which returns the trained weights and the losses.
"""
from __future__ import annotations

import functools
import math

import numpy as np

from pliscuda_amd import capi, learned
from pliscuda_amd import workloads as W

INF = float("inf")


# --------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------


def _steps(name, net, grid, nx, ny, nz, steps, **more):
    return {"name": name, "do": "steps", "net": net, "grid": grid, "nx": nx, "ny": ny, "nz": nz, "steps": steps,
            "realizations": 1, "learned": False, **more}


def listed():
    return [
        # the smallest use: one small box stepped for a long time (teaching models, unit tests, parameter
        # scans by a script); nothing but the latency of a step counts
        _steps("abc_box_4", "abc", "reflecting", 4, 4, 4, 400),
        # diffusion from few molecules per subvolume (5,125 subvolumes as in the reference's benchmark): most
        # steps end at a critical event, many short steps
        _steps("diffusion_low_5125", "diffusion", "reflecting", 41, 25, 5, 400),
        # a signalling network (32 species, 62 reactions, two compartments) along a rod of 60 subvolumes: the
        # shape of the reference's chemotaxis benchmark
        _steps("cascade_rod_60", "cascade", "reflecting", 60, 1, 1, 50),
        # an ensemble of small boxes for statistics: 64 realizations of the 8^3 A-B-C grid
        _steps("abc_ensemble_64x8", "abc", "reflecting", 8, 8, 8, 400, realizations=64),
        # a cell with two compartments of different rates on a grid of odd sides
        _steps("abc_cell_37x29x23", "abc2", "reflecting", 37, 29, 23, 200),
        # transport with drift: hops along x are likelier one way, so the topology is not symmetric
        _steps("abc_drift_45x31x20", "abc", "drift", 45, 31, 20, 100),
        # the bistable model on one 64^3 periodic grid
        _steps("schlogl_64", "schlogl", "periodic", 64, 64, 64, 200),
        # an ensemble of uneven grids of 16..48 a side in one context (2.7 M subvolumes)
        _steps("schlogl_batch_64", "schlogl", "periodic", 16, 0, 48, 40, realizations=64),
        # the headline: 1,048,576 subvolumes of a weighted random mesh, 5 species, 8 reactions
        _steps("brusselator_mesh_1M", "brusselator", "mesh", 128, 128, 64, 200),
        # uneven random meshes in one context, as parameter studies on real geometries hold them
        _steps("brusselator_batch_32", "brusselator", "mesh", 8, 0, 32, 150, realizations=32),
        # learned tau on a 262,144-subvolume mesh: proposals by the network inside the leap pass
        _steps("learned_mesh_262k", "brusselator", "mesh", 64, 64, 64, 100, learned=True),
        # training the network on the records of a plain run
        {"name": "train_65536", "do": "train", "records": 262144, "batch": 65536, "steps": 30, "gelu": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: what is run as often as it is listed, sizes over their whole ranges."""
    kind = rng.choice(["box", "diffusion", "cascade", "ensemble", "cell", "drift", "grid", "batch", "mesh",
                       "mesh_batch", "learned", "train"])
    steps = rng.randint(40, 200)
    if kind == "train":
        batch = 64 * _log(rng, 64, 1024)
        return {"do": "train", "records": _log(rng, 20000, 262144), "batch": batch, "steps": rng.randint(10, 30),
                "gelu": rng.random() < 0.7}
    if kind in ("mesh", "learned"):  # the meshes are built on even sides
        n = _log(rng, 4096, 262144)
        a = 2 * rng.randint(2, 1 + int(n ** (1 / 3) / 2))
        b = 2 * rng.randint(2, 1 + int(n ** (1 / 3) / 2))
        c = _steps("", "brusselator", "mesh", a, b, 2 * max(2, n // (2 * a * b)), steps, learned=kind == "learned")
    elif kind == "mesh_batch":
        c = _steps("", "brusselator", "mesh", 2 * rng.randint(3, 6), 0, 2 * rng.randint(7, 16), steps,
                   realizations=_log(rng, 2, 32))
    elif kind == "batch":
        lo = rng.randint(5, 20)
        c = _steps("", "schlogl", "periodic", lo, 0, rng.randint(lo + 1, 40), steps // 2, realizations=_log(rng, 2, 64))
    elif kind == "cascade":
        c = _steps("", "cascade", "reflecting", rng.randint(20, 400), 1, 1, rng.randint(20, 50))
    else:
        n = {"box": (27, 2000), "diffusion": (500, 40000), "ensemble": (64, 4000), "cell": (1000, 60000),
             "drift": (1000, 60000), "grid": (2000, 262144)}[kind]
        n = _log(rng, *n)
        a = rng.randint(3, 2 + int(n ** (1 / 3) * 1.3))
        b = rng.randint(3, 2 + int(n ** (1 / 3)))
        net = {"box": "abc", "diffusion": "diffusion", "ensemble": "abc", "cell": "abc2", "drift": "abc",
               "grid": "schlogl"}[kind]
        grid = {"drift": "drift", "grid": "periodic"}.get(kind, "reflecting")
        c = _steps("", net, grid, a, b, max(3, n // (a * b)), steps,
                   realizations=_log(rng, 8, 128) if kind == "ensemble" else 1)
    del c["name"]
    return c


# --------------------------------------------------------------------------
# models
# --------------------------------------------------------------------------


def _cascade():
    """32 species in a chain of bindings and conversions, 62 reactions; every fourth species diffuses."""
    sp = [f"X{i}" for i in range(32)]
    reactions, k = [], []
    for i in range(30):
        if i % 3 == 0:
            lhs, rhs, kf, kb = {sp[i]: 1, sp[i + 1]: 1}, {sp[i + 2]: 1}, 1e-3, 0.5
        else:
            lhs, rhs, kf, kb = {sp[i]: 1}, {sp[i + 1]: 1}, 0.3, 0.2
        reactions += [(lhs, rhs), (rhs, lhs)]
        k += [kf, kb]
    reactions += [({}, {sp[0]: 1}), ({sp[31]: 1}, {})]
    k += [5.0, 0.1]
    d = [2.5 if i % 4 == 0 else 0.0 for i in range(32)]
    return W.network(sp, reactions, [k, [0.5 * v for v in k]], [d, [0.5 * v for v in d]], n_compartments=2)


@functools.lru_cache(maxsize=None)
def _network(name):
    """(network, Poisson means of the initial counts or None for the bistable model's uniform start, epsilon)"""
    if name == "abc":
        return W.abc_network(), [50.0, 50.0, 50.0], 0.03
    if name == "abc2":
        one = W.abc_network()
        reactions = [({"A": 1, "B": 1}, {"C": 1}), ({"C": 1}, {"A": 1, "B": 1}), ({}, {"A": 1})]
        return W.network(one["species"], reactions, [[0.01, 0.1, 1.0], [0.02, 0.05, 3.0]],
                         [[0.5, 0.5, 0.1], [0.2, 0.8, 0.0]], n_compartments=2), [50.0, 50.0, 20.0], 0.03
    if name == "diffusion":
        return W.network(["A"], [({"A": 1}, {"A": 1})], [0.0], [50.0]), [19.5], 0.05
    if name == "cascade":
        return _cascade(), [40.0] * 32, 0.05
    if name == "schlogl":
        return W.schlogl_network(), None, 0.03
    means = np.random.Generator(np.random.PCG64(W.SEED_BRUSS + 2)).uniform(20.0, 200.0, size=5)
    return W.brusselator_network(W.SEED_BRUSS), list(means), 0.03


@functools.lru_cache(maxsize=None)
def _topology(grid, nx, ny, nz):
    """One topology: a program loads its geometry from a file, so it is not made from the inputs' seed."""
    if grid == "mesh":
        return W.random_mesh(nx, ny, nz, 1000 * nx + 100 * ny + nz)
    topo = dict(W.cubic_grid(nx, ny, nz, periodic=grid == "periodic"))
    if grid == "drift":  # hops to higher subvolume ids along x are likelier
        src = np.repeat(np.arange(topo["N"], dtype=np.int64), np.diff(topo["row_ptr"].astype(np.int64)))
        step = topo["col"].astype(np.int64) - src
        topo["w"] = np.where(step == 1, 1.3, np.where(step == -1, 0.7, 1.0)).astype(np.float32)
    return topo


def _topologies(case):
    """The realizations' topologies.  ny = 0: a batch of uneven sides between nx and nz."""
    n = case["realizations"]
    if case["ny"]:
        topo = _topology(case["grid"], case["nx"], case["ny"], case["nz"])
        if case["net"] in ("abc2", "cascade"):  # an outer and an inner compartment along x
            x = np.arange(topo["N"]) % case["nx"]
            topo = dict(topo, comp=((x >= case["nx"] // 3) & (x < case["nx"] - case["nx"] // 3)).astype(np.int32))
        return [topo] * n
    rng = np.random.Generator(np.random.PCG64(case["nx"] * 97 + case["nz"]))
    if case["grid"] == "mesh":
        sides = 2 * rng.integers(case["nx"] // 2, case["nz"] // 2 + 1, size=(n, 3))
        return [_topology("mesh", int(a), int(b), int(c)) for a, b, c in sides]
    return [_topology(case["grid"], int(s), int(s), int(s)) for s in rng.integers(case["nx"], case["nz"] + 1, size=n)]


def _counts(case, topos, seed):
    net, means, _ = _network(case["net"])
    if means is None:
        return [W.uniform_state(t["N"], 80, 600, seed * 1009 + r) for r, t in enumerate(topos)]
    return [W.poisson_state(net["S"], t["N"], means, seed * 1009 + r) for r, t in enumerate(topos)]


def _context(case, seed):
    net, _, eps = _network(case["net"])
    topos = _topologies(case)
    return capi.Context(net, topos, _counts(case, topos, seed), eps=eps, nc=10, seed=seed)


@functools.lru_cache(maxsize=None)
def _saved_network(nx, ny, nz):
    """The weights that a program loads from a file: fitted to the records of a plain run on this mesh.  The
    hidden layers keep their initial weights, the output layer is the ridge solution in 64 bits."""
    case = _steps("", "brusselator", "mesh", nx, ny, nz, 1)
    with _context(case, 77) as ctx:
        feats, ylog, _ = learned.collect_records(ctx, snapshots=4, stride=4, per_snapshot=4096, seed=1)
        rate = learned.calibrate_viol_rate([ctx.stats(0)], [ctx.N[0]])
    norm = learned.fit_norm(feats, ylog)
    w = learned.init_weights(3)
    h = _hidden(w.astype(np.float64), norm.astype(np.float64), feats.astype(np.float64), True)[-1]
    A = np.concatenate([h, np.ones((len(h), 1))], axis=1)
    y = (ylog.astype(np.float64) - norm[24]) / norm[25]
    sol = np.linalg.solve(A.T @ A + 1e-2 * len(h) * np.eye(65), A.T @ y)
    w[5248:5376] = np.stack([sol[:64], np.zeros(64)], axis=1).ravel().astype(np.float32)
    w[5376:5378] = [sol[64], -2.0]
    return w, norm, rate


# --------------------------------------------------------------------------
# prepare / run
# --------------------------------------------------------------------------


def _training_data(case, seed):
    """Records as a plain run gives them: log counts, log propensities, an order, the previous log tau; the
    targets are a smooth function of them with noise."""
    rng = np.random.Generator(np.random.PCG64(seed))
    n = case["records"]
    f = np.empty((n, 12), dtype=np.float32)
    f[:, :5] = np.log1p(rng.poisson(rng.uniform(20.0, 200.0, size=5), size=(n, 5)))
    f[:, 5:10] = np.log1p(np.exp(f[:, :5]) * rng.uniform(0.5, 8.0, size=5) + rng.random((n, 5)))
    f[:, 10] = rng.integers(1, 4, size=n)
    f[:, 11] = rng.normal(-7.0, 0.3, size=n)
    ylog = (-0.8 * f[:, 5] + 0.3 * f[:, 1] - 0.2 * f[:, 2] * f[:, 0] / 4.0 + 0.05 * rng.standard_normal(n)).astype(np.float32)
    crit = (rng.random(n) < 0.16).astype(np.float32)
    norm = learned.fit_norm(f, ylog)
    return f, learned.standardize_y(ylog, norm), crit, norm


def prepare(case, seed):
    if case["do"] == "train":
        f, y, c, norm = _training_data(case, seed)
        topo = _topology("reflecting", 4, 4, 4)
        ctx = capi.Context(W.abc_network(), [topo], [W.poisson_state(3, topo["N"], 50.0, seed)], seed=seed)
        ctx.mlp_activation(1 if case["gelu"] else 0)
        return {"do": "train", "ctx": ctx, "feats": f, "y": y, "crit": c, "norm": norm, "w0": learned.init_weights(seed),
                "steps": case["steps"], "batch": case["batch"], "seed": seed}
    ctx = _context(case, seed)
    if case["learned"]:
        w, norm, rate = _saved_network(case["nx"], case["ny"], case["nz"])
        ctx.mlp_set(w, norm)
        ctx.set_tau_mode(True, kappa=1.0, theta=learned.THETA, viol_rate_max=rate)
    return {"do": "steps", "ctx": ctx, "steps": case["steps"], "made": 0}


def run(state):
    ctx = state["ctx"]
    if state["do"] == "train":
        ctx.mlp_set(state["w0"], state["norm"])
        losses = ctx.mlp_train(state["feats"], state["y"], state["crit"], state["steps"], state["batch"], 1e-3, state["seed"])
        return {"weights": ctx.mlp_get(), "losses": losses}
    state["made"] += state["steps"]
    ctx.run(INF, step_limit=state["made"])
    counts = [ctx.get_state(r).view(np.int32) for r in range(ctx.n)]
    stats = [ctx.stats(r) for r in range(ctx.n)]
    whole = ("steps", "leapbacks", "firings", "subvolume_leaps", "crit_events", "learned_steps", "learned_rejects", "violations")
    return {"counts": counts[0] if ctx.n == 1 else np.concatenate(counts),
            "t": np.array([s["t"] for s in stats]), "tau": np.array([s["tau"] for s in stats]),
            "stats": np.array([[s[f] for f in whole] for s in stats], dtype=np.int64)}


def work(case):
    """Bytes: the records once and each minibatch's rows; counts read and written and the topology read in each
    step.  Flops: the network forward and backward; propensities, their changes and the hops' means in each step."""
    if case["do"] == "train":
        rows = case["steps"] * case["batch"]
        return {"bytes": 56.0 * (case["records"] + rows), "flops": rows * 6.0 * (12 * 64 + 64 * 64 + 64 * 2)}
    net = _network(case["net"])[0]
    S, R = net["S"], net["R"]
    topos = _topologies(case)
    N = sum(t["N"] for t in topos)
    E = sum(len(t["col"]) for t in topos)
    edge = 8 if topos[0].get("w") is not None else 4
    flops = N * (8.0 * R + 20.0 * S) + E * 6.0 * S
    if case["learned"]:
        flops += N * 2.0 * (12 * 64 + 64 * 64 + 64 * 2)
    return {"bytes": case["steps"] * (8.0 * S * N + 4.0 * N + edge * float(E)), "flops": case["steps"] * flops}


# --------------------------------------------------------------------------
# exact
# --------------------------------------------------------------------------


def _gelu(z):
    """The library's GELU, max(z, 0) - |z| max(0, p(|z|)) with a cubic p, and its derivative."""
    c1, c2, c3 = (float(np.float32(v)) for v in (-0.47735822, 0.15120307, -0.01585033))
    a = np.abs(z)
    p = 0.5 + a * (c1 + a * (c2 + a * c3))
    q = np.where(p > 0.0, p + a * (c1 + a * (2.0 * c2 + a * 3.0 * c3)), 0.0)
    return np.maximum(z, 0.0) - a * np.maximum(p, 0.0), np.where(z > 0.0, 1.0 - q, q)


def _act(z, gelu):
    return _gelu(z) if gelu else (np.maximum(z, 0.0), (z > 0.0).astype(np.float64))


def _layers(w):
    return (w[:1024].reshape(16, 64)[:12], w[1024:1088], w[1088:5184].reshape(64, 64), w[5184:5248],
            w[5248:5376].reshape(64, 2), w[5376:5378])


def _hidden(w, norm, feats, gelu):
    w1, b1, w2, b2, _, _ = _layers(w)
    x = (feats - norm[:12]) / norm[12:24]
    h1, g1 = _act(x @ w1 + b1, gelu)
    h2, g2 = _act(h1 @ w2 + b2, gelu)
    return x, h1, g1, g2, h2


def _loss_grad(w, norm, feats, y, crit, gelu):
    _, _, w2, _, w3, b3 = _layers(w)
    x, h1, g1, g2, h2 = _hidden(w, norm, feats, gelu)
    o = h2 @ w3 + b3
    loss = (o[:, 0] - y) ** 2 + np.logaddexp(0.0, o[:, 1]) - crit * o[:, 1]
    do = np.stack([2.0 * (o[:, 0] - y), 1.0 / (1.0 + np.exp(-o[:, 1])) - crit], axis=1) / len(y)
    dz2 = (do @ w3.T) * g2
    dz1 = (dz2 @ w2.T) * g1
    g = np.zeros(5378)
    g[:768] = (x.T @ dz1).ravel()
    g[1024:1088] = dz1.sum(0)
    g[1088:5184] = (h1.T @ dz2).ravel()
    g[5184:5248] = dz2.sum(0)
    g[5248:5376] = (h2.T @ do).ravel()
    g[5376:] = do.sum(0)
    return loss.mean(), g


def _philox_row(sample, step, seed, n):
    """The record that a minibatch's sample takes: Philox4x32-10 (Salmon et al., SC'11) of (sample, step)."""
    c = [sample.astype(np.uint64), np.full(sample.shape, step, np.uint64), np.full(sample.shape, 0x4D4C50, np.uint64),
         np.zeros(sample.shape, np.uint64)]
    k0, k1, low = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF, np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & low, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return ((c[1] << np.uint64(32)) | c[0]) % np.uint64(n)


def exact(case, seed):
    """Training in 64 bits.  A trajectory is made of random draws: no value but its own for it."""
    if case["do"] != "train":
        return None
    f, y, c, norm = (v.astype(np.float64) for v in _training_data(case, seed))
    w = learned.init_weights(seed).astype(np.float64)
    m, v = np.zeros(5378), np.zeros(5378)
    losses = np.empty(case["steps"])
    for t in range(case["steps"]):
        row = _philox_row(np.arange(case["batch"]), t, seed, case["records"]).astype(np.int64)
        losses[t], g = _loss_grad(w, norm, f[row], y[row], c[row], case["gelu"])
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1.0 - 0.9 ** (t + 1))) / (np.sqrt(v / (1.0 - 0.999 ** (t + 1))) + 1e-8)
    return {"weights": w, "losses": losses}
