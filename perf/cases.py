"""The workloads this package is timed on: what a user's program calls, over
the range of sizes, rules and options that this repository's tests, benchmark
and command line use.

``listed`` gives the fixed cases, ``draw`` more of the same ranges;
``prepare`` makes what a program holds before the call (instances, contexts,
network, inputs), ``run`` is one pass through the public entry points,
``work`` the bytes and operations that pass cannot do without, and ``exact``
its floating-point results in 64 bits from numpy alone where the outputs are
computed numbers (tours and trails are the outcome of a random search and
have no such value).
"""
from __future__ import annotations

import math

import numpy as np

import cvrp_aco_ocl_amd as ca
from cvrp_aco_ocl_amd import decompose as dc
from cvrp_aco_ocl_amd import prior as pr

NF, H = pr.NF, 64
# parameter vector of the prior network: W1[64][12], b1, W2[64][64], b2, w3, b3
O_B1 = H * NF
O_W2 = O_B1 + H
O_B2 = O_W2 + H * H
O_W3 = O_B2 + H
O_B3 = O_W3 + H

DIST = {"float": ca.DIST_FLOAT, "nint": ca.DIST_NINT}
SELECT = {"iroulette": (ca.SEL_IROULETTE, ca.RNG_PARK_MILLER), "knn": (ca.SEL_KNN, ca.RNG_PHILOX)}
SEARCH = {"none": 0, "2opt": ca.LS_2OPT, "2opt+swap": ca.LS_2OPT | ca.LS_SWAP,
          "full": ca.LS_2OPT | ca.LS_SWAP | ca.LS_RELOCATE,
          "full-random": ca.LS_2OPT_RANDOM | ca.LS_SWAP | ca.LS_RELOCATE}


def listed():
    return [
        # the smallest: a 50-customer set of the kind the literature starts with,
        # unrounded distances, route-length limit and service time, a short try
        # under the reference's rules (command line defaults): latency, launches
        dict(name="try_51_limit", kind="colony", customers=50, geometry="uniform", per_route=9, dist="float",
             limit=True, ants=51, rule="iroulette", k=0, search="2opt", tau0="first", iterations=5,
             tuned=False),
        # 100 uniform customers, reference rules, one ant per customer (the
        # seed-distribution workload of the tests)
        dict(name="try_101_reference", kind="colony", customers=100, geometry="uniform", per_route=13,
             dist="nint", limit=False, ants=100, rule="iroulette", k=0, search="2opt", tau0="nn",
             iterations=10, tuned=False),
        # a mid-sized set with a route-length limit and unrounded distances,
        # candidate roulette, full local search, launch shape not tuned
        dict(name="limit_242_float", kind="colony", customers=241, geometry="uniform", per_route=9,
             dist="float", limit=True, ants=242, rule="knn", k=20, search="full", tau0="nn", iterations=5,
             tuned=False),
        # the 481-node clustered instance of the benchmark: 480 ants, k = 30
        dict(name="clustered_481", kind="colony", customers=480, geometry="clustered", per_route=16,
             dist="nint", limit=False, ants=480, rule="knn", k=30, search="full", tau0="first",
             iterations=20, tuned=True),
        # the benchmark's main workload, 1001 nodes, 256 ants, k = 32, its trail
        # saved at the end of the run
        dict(name="mixed_1001", kind="colony", customers=1000, geometry="mixed", per_route=12, dist="nint",
             limit=False, ants=256, rule="knn", k=32, search="full", tau0="first", iterations=20,
             tuned=True, trail=True),
        # the same instance under the reference's rules
        dict(name="mixed_1001_reference", kind="colony", customers=1000, geometry="mixed", per_route=12,
             dist="nint", limit=False, ants=256, rule="iroulette", k=0, search="full", tau0="first",
             iterations=10, tuned=True),
        # many instances in one context (labelling, evaluation, serving)
        dict(name="batch_256", kind="batch", count=256, ants=64, k=16, search="full", iterations=5,
             tuned=True),
        # a large instance: master colony without local search, then one
        # decomposition round with the default sub-colonies
        dict(name="decompose_3001", kind="decompose", customers=3000, ants=256, k=16, iterations=1,
             sub_ants=64, sub_iterations=75),
        # setting up a solver for a new instance: lists, heuristic, tables
        dict(name="setup_1001", kind="setup", customers=1000, geometry="mixed", dist="nint", k=32, ants=64),
        # the learned prior of one instance, as a dense multiplier
        dict(name="prior_build_501", kind="prior_build", customers=500, k=16, exponent=0.5),
        # one gradient of the prior's loss at the training batch size
        dict(name="prior_gradient", kind="prior_gradient", customers=1024, k=16, edges=16384),
        # a short training run of the prior, 16384 edges per step
        dict(name="prior_train", kind="prior_train", customers=4096, k=16, edges=65536, batch=16384, epochs=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["colony"] * 6 + ["batch"] * 2 + ["decompose", "setup", "prior_build", "prior_gradient",
                                                        "prior_train"])
    if kind == "colony":
        customers = _log_int(rng, 40, 1000)
        rule = rng.choice(["iroulette", "knn", "knn"])
        return dict(kind=kind, customers=customers, geometry=rng.choice(["uniform", "clustered", "mixed"]),
                    per_route=rng.randint(6, 24), dist=rng.choice(["nint", "nint", "float"]),
                    limit=rng.random() < 0.25, ants=_log_int(rng, 24, 512) if rule == "knn" else
                    _log_int(rng, 24, 256), rule=rule, k=0 if rule == "iroulette" else rng.randint(8, 32),
                    search=rng.choice(["2opt", "2opt+swap", "full", "full", "full", "full-random"]),
                    tau0=rng.choice(["first", "nn"]), iterations=rng.randint(3, 10),
                    tuned=rng.random() < 0.7, trail=rng.random() < 0.1)
    if kind == "batch":
        return dict(kind=kind, count=_log_int(rng, 4, 160), ants=rng.choice([32, 48, 64]),
                    k=rng.choice([8, 12, 16, 20]), search=rng.choice(["2opt", "full", "full"]),
                    iterations=rng.randint(2, 5), tuned=rng.random() < 0.6)
    if kind == "decompose":
        return dict(kind=kind, customers=_log_int(rng, 400, 2500), ants=rng.choice([64, 128, 256]),
                    k=rng.choice([12, 16]), iterations=rng.randint(1, 2), sub_ants=rng.choice([32, 64]),
                    sub_iterations=rng.randint(20, 75))
    if kind == "setup":
        return dict(kind=kind, customers=_log_int(rng, 40, 1400), geometry=rng.choice(["uniform", "mixed"]),
                    dist=rng.choice(["nint", "float"]), k=rng.randint(8, 32), ants=rng.choice([32, 64]))
    if kind == "prior_build":
        return dict(kind=kind, customers=_log_int(rng, 50, 1000), k=rng.choice([8, 12, 16]),
                    exponent=rng.choice([0.5, 1.0, 2.0]))
    edges = _log_int(rng, 500, 65536)
    if kind == "prior_gradient":
        return dict(kind=kind, customers=max(17, (edges + 15) // 16), k=16, edges=edges)
    return dict(kind=kind, customers=max(17, (edges + 15) // 16), k=16, edges=edges,
                batch=rng.choice([1024, 4096, 16384]), epochs=rng.randint(1, 3))


# ------------------------------------------------------------- inputs ----

def _clusters(r, count, nclust, sigma):
    centres = r.uniform(0.0, 1000.0, size=(nclust, 2))
    pts = centres[r.integers(0, nclust, size=count)] + r.normal(0.0, sigma, size=(count, 2))
    return np.clip(np.rint(pts), 0.0, 1000.0)


def _coords(geometry, customers, r):
    """Customers in [0,1000]^2: uniform, 8 Gaussian clusters (sigma 6), or
    half uniform and half in 10 clusters (sigma 25); depot at the centre,
    or anywhere for the clustered ones."""
    if geometry == "uniform":
        pts = r.integers(0, 1001, size=(customers, 2)).astype(np.float64)
    elif geometry == "clustered":
        pts = _clusters(r, customers, 8, 6.0)
    else:
        half = customers // 2
        pts = np.concatenate([r.integers(0, 1001, size=(half, 2)).astype(np.float64),
                              _clusters(r, customers - half, 10, 25.0)])
    depot = r.integers(0, 1001, size=2).astype(np.float64) if geometry == "clustered" else np.array([500.0, 500.0])
    return np.concatenate([depot[None], pts])


def _instance(case, seed):
    r = np.random.default_rng(seed)
    xy = _coords(case["geometry"], case["customers"], r)
    dem = np.concatenate([[0], r.integers(1, 101, size=case["customers"])]).astype(np.int32)
    cap = max(int(math.ceil(case.get("per_route", 12) * dem[1:].mean())), int(dem.max()))
    limit, service = math.inf, 0.0
    if case.get("limit"):
        # a vehicle reaches every customer alone; full routes are longer than the limit now and then
        far = float(np.hypot(*(xy - xy[0]).T).max())
        service = 10.0
        limit = float(math.ceil(2.6 * far + 6 * service))
    return ca.Instance.from_coords(xy[:, 0], xy[:, 1], dem, cap, DIST[case["dist"]], max_dist=limit,
                                   service_time=service)


def _batch(case, seed):
    """Uneven instances: 50 to 500 customers, uniform or 4 to 12 clusters,
    5 to 40 routes."""
    r = np.random.default_rng(seed)
    xs, dems, caps = [], [], []
    for _ in range(case["count"]):
        c = int(r.integers(50, 501))
        pts = (r.integers(0, 1001, size=(c, 2)).astype(np.float64) if r.random() < 0.5 else
               _clusters(r, c, int(r.integers(4, 13)), float(r.uniform(10.0, 60.0))))
        xs.append(np.concatenate([r.integers(0, 1001, size=(1, 2)).astype(np.float64), pts]))
        dem = np.concatenate([[0], r.integers(1, 51, size=c)]).astype(np.int32)
        dems.append(dem)
        caps.append(max(int(math.ceil(dem.sum() / int(r.integers(5, 41)))), int(dem.max())))
    dist = ca.Instance.distances_batch([p[:, 0] for p in xs], [p[:, 1] for p in xs], ca.DIST_NINT)
    return [ca.Instance(n=len(p), x=p[:, 0].copy(), y=p[:, 1].copy(), demand=d, capacity=q, dist=m)
            for p, d, q, m in zip(xs, dems, caps, dist)]


def _edge_set(case, seed):
    """Coordinates, demands, distances, candidate lists (ties to the lower
    index) and capacity of a clustered instance, in numpy."""
    r = np.random.default_rng(seed)
    xy = _coords("clustered", case["customers"], r)
    dem = np.concatenate([[0], r.integers(1, 101, size=case["customers"])]).astype(np.int32)
    cap = max(int(math.ceil(dem.sum() / 30)), int(dem.max()))
    d = np.sqrt((xy[:, None, 0] - xy[None, :, 0]) ** 2 + (xy[:, None, 1] - xy[None, :, 1]) ** 2)
    d = np.floor(d + 0.5)
    key = d.copy()
    key[:, 0] = np.inf
    np.fill_diagonal(key, np.inf)
    nn = np.argsort(key, axis=1, kind="stable")[:, :case["k"]].astype(np.int32)
    return xy, dem, cap, d, nn


def _features64(xy, dem, cap, d, nn, k):
    n = len(xy)
    rad = np.hypot(xy[:, 0] - xy[0, 0], xy[:, 1] - xy[0, 1])
    ang = np.arctan2(xy[:, 1] - xy[0, 1], xy[:, 0] - xy[0, 0]) / np.pi
    kd = d[np.arange(n), nn[:, k - 1]]
    i, q = np.repeat(np.arange(n), k), np.tile(np.arange(k), n)
    j = nn[:, :k].reshape(-1)
    mkd, big = kd.mean(), rad.max()
    return np.stack([d[i, j] / mkd, q / k, dem[i] / cap, dem[j] / cap, ang[i], ang[j], rad[i] / big,
                     rad[j] / big, kd[i] / mkd, kd[j] / mkd, (d[0, i] + d[0, j] - d[i, j]) / big,
                     (nn[j][:, :k] == i[:, None]).any(axis=1).astype(np.float64)], axis=1)


def _edges(case, seed):
    """Features and labels of about 10% positives, nearer candidates first,
    as the tours of solved instances give them."""
    # the features of clustered instances of 500 customers, as many as the edges need
    f = []
    for s in range(-(-case["edges"] // (501 * case["k"]))):
        c = dict(case, customers=min(500, case["customers"]))
        f.append(_features64(*_edge_set(c, seed * 1000 + s), case["k"]))
    f = np.concatenate(f)
    while len(f) < case["edges"]:
        f = np.concatenate([f, f])
    f = np.ascontiguousarray(f[:case["edges"]], np.float32)
    r = np.random.default_rng(seed + 7)
    y = (r.random(len(f)) < 0.55 * np.exp(-5.0 * f[:, 1])).astype(np.float32)
    w = r.uniform(-1, 1, pr.NPARAM).astype(np.float32)
    w[:O_B1] *= math.sqrt(6 / (NF + H))
    w[O_W2:O_B2] *= math.sqrt(6 / (H + H))
    w[O_W3:O_B3] *= math.sqrt(6 / (H + 1))
    w[O_B1:O_W2] = w[O_B2:O_W3] = w[O_B3] = 0.0
    return f, y, w


# ---------------------------------------------------------------- passes ----

def _colony(case, insts, seed):
    sel, rng = SELECT[case.get("rule", "knn")]
    tau0 = ca.TAU0_NN_TOUR if case.get("tau0", "nn") == "nn" else ca.TAU0_FIRST_COLONY
    g = ca.GpuACO(insts, n_ants=case["ants"], k=case["k"], selection=sel, rng=rng,
                  ls_flags=SEARCH[case.get("search", "none")], tau0_rule=tau0, seed=seed + 1)
    if case.get("tuned"):
        g.init_aco()
        g.autotune(reps=2)
    return g


def prepare(case, seed):
    kind = case["kind"]
    if kind == "colony":
        return dict(kind=kind, g=_colony(case, _instance(case, seed), seed), iterations=case["iterations"],
                    trail=case.get("trail", False))
    if kind == "batch":
        return dict(kind=kind, g=_colony(case, _batch(case, seed), seed), iterations=case["iterations"])
    if kind == "decompose":
        inst = _instance(dict(case, geometry="mixed", per_route=75, dist="nint"), seed)
        return dict(kind=kind, inst=inst, g=_colony(dict(case, tau0="first"), inst, seed),
                    iterations=case["iterations"], sub_iterations=case["sub_iterations"],
                    sub=dc.sub_params(n_ants=case["sub_ants"], seed=seed + 5))
    if kind == "setup":
        return dict(kind=kind, inst=_instance(case, seed), case=case, seed=seed)
    if kind == "prior_build":
        xy, dem, cap, d, nn = _edge_set(case, seed)
        inst = ca.Instance(n=len(xy), x=xy[:, 0].copy(), y=xy[:, 1].copy(), demand=dem, capacity=cap,
                           dist=d.astype(np.float32))
        return dict(kind=kind, inst=inst, nn=nn, net=pr.PriorNet.load(), k=case["k"],
                    exponent=case["exponent"])
    f, y, w = _edges(case, seed)
    return dict(kind=kind, f=f, y=y, w=w, net=pr.PriorNet(params=w), case=case, seed=seed)


def _padded(tour, n):
    """A tour in an array of 2n entries (its longest possible form)."""
    out = np.zeros(2 * n, np.int32)
    out[:len(tour)] = tour
    return out


def run(state):
    kind = state["kind"]
    if kind == "colony":
        # one try: initial colony, iterations, the best tour, the last colony's
        # tours (a program that goes on, or restarts, keeps these) and the trail
        g = state["g"]
        g.init_aco()
        g.run(state["iterations"])
        tour, length = g.best()
        tours, sizes, lengths = g.ants()
        # a tour's buffer past its end is not part of the answer
        tours[np.arange(tours.shape[1])[None, :] >= sizes[:, None]] = 0
        out = {"tour": _padded(tour, g.n), "length": length, "tours": tours, "sizes": sizes,
               "lengths": lengths}
        if state["trail"]:
            out["tau"], out["info"] = g.pheromone()
        return out
    if kind == "batch":
        g = state["g"]
        g.init_aco()
        g.run(state["iterations"])
        best = [g.best(b) for b in range(g.B)]
        return {"tours": np.stack([_padded(t, 501) for t, _ in best]),
                "lengths": np.array([v for _, v in best], np.float32)}
    if kind == "decompose":
        g = state["g"]
        g.init_aco()
        g.run(state["iterations"])
        tour, length = g.best()
        merged, mlen, subs, replaced = dc.decompose_round(g, state["inst"], params=state["sub"],
                                                          sub_iterations=state["sub_iterations"])
        return {"tour": _padded(tour, g.n), "length": length, "merged": _padded(merged, g.n),
                "merged_length": mlen, "subs": subs, "replaced": replaced}
    if kind == "setup":
        with _colony(state["case"], state["inst"], state["seed"]) as g:
            return g.setup_arrays()
    if kind == "prior_build":
        return state["net"].build(state["inst"], state["nn"], state["k"], exponent=state["exponent"])
    if kind == "prior_gradient":
        g, loss = state["net"].gradient(state["f"], state["y"], 3.0)
        return {"grad": g, "loss": loss}
    # every pass trains the same network from the same start
    net, c = state["net"], state["case"]
    net.set_params(state["w"])
    losses = net.train(state["f"], state["y"], epochs=c["epochs"], batch=c["batch"], pos_weight=3.0,
                       shuffle_seed=state["seed"] + 11)
    return {"params": net.params(), "losses": losses}


def work(case):
    """Matrices and tours read and written once per step; every construction
    step's candidates weighed once, every position's nearest partners once."""
    kind = case["kind"]
    n = case.get("customers", 0) + 1

    def colony(n, m, k, search, iterations):
        step_bytes = 16 * n * n + 8 * n * k + 16 * m * n
        step_ops = m * n * (6 * k if k else 4 * n) + (m * n * 256 if search != "none" else 0)
        return iterations * step_bytes, iterations * step_ops

    if kind == "colony":
        b, f = colony(n, case["ants"], case["k"], case["search"], case["iterations"])
    elif kind == "batch":
        b, f = colony(296, case["ants"], case["k"], case["search"], case["iterations"])
        b, f = b * case["count"], f * case["count"]
    elif kind == "decompose":
        b, f = colony(n, case["ants"], case["k"], "none", case["iterations"] + 1)
        subs = max(1, case["customers"] // 150)
        sb, sf = colony(151, case["sub_ants"], 16, "full", case["sub_iterations"])
        b, f = b + subs * sb, f + subs * sf
    elif kind == "setup":
        b, f = n * n * (4 + 4 + 8 + 2 + 2), 10 * n * n * math.log2(n)
    else:
        per_edge = 2 * (NF * H + H * H + H)
        if kind == "prior_build":
            b, f = 8 * n * n, n * case["k"] * per_edge
        elif kind == "prior_gradient":
            b, f = case["edges"] * (4 * NF + 4) + 8 * pr.NPARAM, 3 * case["edges"] * per_edge
        else:
            b = case["edges"] * (4 * NF + 4) + 8 * pr.NPARAM
            f = 3 * case["epochs"] * case["edges"] * per_edge
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------ 64 bits ----

def _net64(w, x):
    w = np.asarray(w, np.float64)
    W1, b1 = w[:O_B1].reshape(H, NF), w[O_B1:O_W2]
    W2, b2 = w[O_W2:O_B2].reshape(H, H), w[O_B2:O_W3]
    z1 = x @ W1.T + b1
    h1 = np.maximum(z1, 0)
    z2 = h1 @ W2.T + b2
    h2 = np.maximum(z2, 0)
    return z1, h1, z2, h2, h2 @ w[O_W3:O_B3] + w[O_B3]


def _gradient64(w, x, y, pos):
    z1, h1, z2, h2, z = _net64(w, x)
    we = np.where(y > 0.5, pos, 1.0)
    loss = np.mean(we * (np.logaddexp(0.0, z) - y * z))
    g = we * (1.0 / (1.0 + np.exp(-z)) - y) / len(z)
    d2 = g[:, None] * np.asarray(w[O_W3:O_B3], np.float64) * (z2 > 0)
    d1 = (d2 @ np.asarray(w[O_W2:O_B2], np.float64).reshape(H, H)) * (z1 > 0)
    return np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), g @ h2,
                           [g.sum()]]), loss


def _train64(case, f, y, w, seed):
    """Adam over shuffled batches (a Fisher-Yates order per epoch from one
    SplitMix64 stream), cosine step size from 3e-3 to 3e-4."""
    mask, s = (1 << 64) - 1, (seed + 11) & ((1 << 64) - 1)
    p, m, v = w.astype(np.float64), np.zeros(len(w)), np.zeros(len(w))
    x, losses, step = f.astype(np.float64), [], 0
    nb = -(-len(f) // case["batch"])
    total = nb * case["epochs"]
    for _ in range(case["epochs"]):
        perm = list(range(len(f)))
        for i in range(len(f) - 1, 0, -1):
            s = (s + 0x9E3779B97F4A7C15) & mask
            z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            j = (z ^ (z >> 31)) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        perm, ep = np.array(perm), []
        for b in range(nb):
            at = perm[b * case["batch"]:(b + 1) * case["batch"]]
            lr = 3e-4 + 0.5 * (3e-3 - 3e-4) * (1.0 + math.cos(math.pi * step / max(total - 1, 1)))
            step += 1
            g, loss = _gradient64(p, x[at], y[at], 3.0)
            ep.append(loss)
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            p = p - lr * (m / (1 - 0.9 ** step)) / (np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
        losses.append(np.mean(ep))
    return p, np.array(losses)


def exact(case, seed):
    kind = case["kind"]
    if kind == "setup":
        r = np.random.default_rng(seed)
        xy = _coords(case["geometry"], case["customers"], r)
        d = np.sqrt((xy[:, None, 0] - xy[None, :, 0]) ** 2 + (xy[:, None, 1] - xy[None, :, 1]) ** 2)
        if case["dist"] == "nint":
            d = np.floor(d + 0.5)
        key = d.copy()
        key[:, 0] = np.inf
        np.fill_diagonal(key, np.inf)
        key.sort(axis=1)
        return {"heur": 1.0 / (d + 0.1) ** 2, "d0": d[:, 0].copy(), "nnk": None,
                "nnkd": key[:, :case["k"]].copy(), "nnls": None, "nnd": key[:, :len(d) - 2].copy(),
                "nnpos": None, "dist16": None}
    if kind == "prior_build":
        xy, dem, cap, d, nn = _edge_set(case, seed)
        w = np.fromfile(pr.WEIGHTS_PATH, np.float32)
        z = _net64(w, _features64(xy, dem, cap, d, nn, case["k"]))[-1]
        out = np.full(d.shape, 0.05 ** case["exponent"])
        np.put_along_axis(out, nn.astype(np.int64),
                          ((1.0 / (1.0 + np.exp(-z))) ** case["exponent"]).reshape(nn.shape), axis=1)
        return out
    if kind == "prior_gradient":
        f, y, w = _edges(case, seed)
        g, loss = _gradient64(w, f.astype(np.float64), y.astype(np.float64), 3.0)
        return {"grad": g, "loss": float(loss)}
    if kind == "prior_train":
        f, y, w = _edges(case, seed)
        p, losses = _train64(case, f, y.astype(np.float64), w, seed)
        return {"params": p, "losses": losses}
    return None
