"""The calls whose speed is measured: connected components of a graph that is held on the GPU, one by one and in
batches, with each variant, schedule and deviate stream that programs use, and the training of the model behind the
learned centre proposals.

Every case is a whole call of the Python entry points: the handle (DeviceGraph, DeviceBatch, Mlp) is what a program keeps
between calls, and the labels come back to host memory as they do for the command-line programs.  Graphs are drawn from
the seed by the package's own generators; sizes are those of bench.py and the tests, or odd ones near them.

Outputs are labels and counts that the graph and the seed alone decide.  The number of sweeps is left out: sweeps work in
place, so it can differ from call to call.  With learned centres the number of levels is left out too: the features sample
rows whose entries stand in no fixed order from the second level on.
"""
import math

import numpy as np

import components_amd as ca


def _rmat(scale, **kw):
    return dict(kind="graph", graph="rmat", n=1 << scale, m=16 << scale, **kw)


def listed():
    return [
        # the smallest calls: a sparse random graph with every option at its default (in-place sweeps, reference draw)
        dict(name="gnm_small_default", kind="graph", graph="gnm_undirected", n=1 << 14, m=1 << 15, variant="exp",
             rounds=False, hashed=False),
        # ordinary: G(n,m) of 2^20 vertices, the benchmark's schedule and stream
        dict(name="gnm_2p20_rounds", kind="graph", graph="gnm_undirected", n=1 << 20, m=1 << 22, variant="exp",
             rounds=True, hashed=True),
        # high diameter, short rows, many clusters a level: the percolated 3D grid
        dict(name="grid3d_256_rounds", kind="graph", graph="grid_3d", n=256, p=0.3, variant="exp", rounds=True,
             hashed=True),
        # a geometric graph of an odd size, defaults
        dict(name="rgg2d_default", kind="graph", graph="rgg_2d", n=2000003, d=8.0, variant="exp", rounds=False,
             hashed=False),
        # the largest: skewed degrees, the headline workload
        dict(name="rmat24_rounds", **_rmat(24, variant="exp", rounds=True, hashed=True)),
        # skewed degrees with the command-line program's defaults
        dict(name="rmat20_default", **_rmat(20, variant="exp", rounds=False, hashed=False)),
        # the learned form on a hyperbolic graph
        dict(name="rhg20_learned", kind="learned", graph="rhg", n=1 << 20, d=16.0, gamma=2.8),
        # the other programs: shortcuts on a percolated 2D grid, local contraction on an odd-sized random graph
        dict(name="grid2d_shortcut", kind="graph", graph="grid_2d", n=1500, m=1100, p=0.6, variant="shortcut",
             rounds=False, hashed=False),
        dict(name="gnm_local", kind="graph", graph="gnm_undirected", n=700001, m=2100003, variant="local",
             rounds=False, hashed=False),
        # thousands of small graphs in the persistent kernel, the default launch shape
        dict(name="batch_small", kind="batch", graphs=4096, lo=8.0, hi=12.0, block=256, groups=4, split=0),
        # a mix of small and large graphs, the large ones together in the device-wide path, as the autotuner picks
        dict(name="batch_mixed", kind="batch", graphs=1024, lo=8.0, hi=16.0, block=512, groups=1, split=4096),
        # training of the model on a dataset of traces
        dict(name="mlp_train", kind="train", rows=300007, batch=8192, steps=50),
    ]


# (draw() keeps to sparse graphs: a connected one has the same labels whatever its seed.)
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["graph"] * 6 + ["batch"] * 2 + ["learned", "train"])
    if kind == "train":
        return dict(kind="train", rows=_log_int(rng, 20000, 500000), batch=16 * rng.randint(64, 1024),
                    steps=rng.randint(10, 60))
    if kind == "batch":
        if rng.random() < 0.5:
            return dict(kind="batch", graphs=_log_int(rng, 64, 4096), lo=8.0, hi=rng.uniform(9.0, 12.0),
                        block=rng.choice([256, 512]), groups=rng.choice([1, 2, 4]), split=0)
        return dict(kind="batch", graphs=_log_int(rng, 64, 1024), lo=8.0, hi=rng.uniform(13.0, 16.0), block=512,
                    groups=1, split=4096)
    if kind == "learned":
        if rng.random() < 0.5:
            return dict(kind="learned", graph="rhg", n=_log_int(rng, 30000, 1 << 20), d=rng.uniform(8.0, 20.0),
                        gamma=rng.uniform(2.5, 3.0))
        return dict(kind="learned", graph="rmat", n=1 << rng.randint(16, 21), m=0, d=16.0, gamma=0.0)
    c = dict(kind="graph")
    graph = rng.choice(["gnm_undirected", "gnm_undirected", "grid_3d", "grid_2d", "rgg_2d", "rmat", "rmat"])
    if graph == "gnm_undirected":
        n = _log_int(rng, 1000, 4000000)
        c.update(graph=graph, n=n, m=int(n * rng.uniform(1.0, 2.0 if n < 20000 else 4.0)))
    elif graph == "grid_3d":
        c.update(graph=graph, n=rng.randint(12, 200), p=rng.uniform(0.25, 0.5))
    elif graph == "grid_2d":
        c.update(graph=graph, n=rng.randint(40, 2000), m=rng.randint(40, 2000), p=rng.uniform(0.5, 0.75))
    elif graph == "rgg_2d":
        c.update(graph=graph, n=_log_int(rng, 2000, 3000000), d=rng.uniform(4.0, 7.0))
    else:
        scale = rng.randint(12, 22)
        c.update(graph=graph, n=1 << scale, m=int((1 << scale) * rng.uniform(4.0, 16.0)))
    c["variant"] = rng.choice(["exp"] * 5 + ["shortcut", "local"])
    c["rounds"] = c["variant"] == "exp" and rng.random() < 0.5
    c["hashed"] = c["rounds"] or rng.random() < 0.3
    return c


def _size(case):
    """(vertices, undirected edges) of the case's graph, about."""
    g, n = case["graph"], case["n"]
    if g == "grid_3d":
        return n ** 3, int(3 * n ** 3 * case["p"])
    if g == "grid_2d":
        return n * case["m"], int(2 * n * case["m"] * case["p"])
    if g in ("rgg_2d", "rhg"):
        return n, int(n * case["d"] / 2)
    if g == "rmat":
        return n, case["m"] or 16 * n
    return n, case["m"]


def _host_or_device_graph(case, seed):
    """The handle of the case's graph: generated in HBM where the library does that, else on the host and copied."""
    g, n, s = case["graph"], case["n"], seed % (1 << 30) + 1
    if g == "rmat":
        return ca.DeviceGraph.generate("rmat", n=n, m=case["m"] or 16 * n, seed=s, rmat_a=0.57, rmat_b=0.19, rmat_c=0.19)
    if g == "grid_3d":
        return ca.DeviceGraph.generate(g, nx=n, ny=n, nz=n, p=case["p"], seed=s)
    if g == "grid_2d":
        return ca.DeviceGraph.generate(g, nx=n, ny=case["m"], p=case["p"], seed=s)
    if g == "gnm_undirected":
        return ca.DeviceGraph.generate(g, n=n, m=case["m"], seed=s)
    if g == "rgg_2d":
        return ca.DeviceGraph(ca.generate(g, n=n, r=math.sqrt(case["d"] / (math.pi * n)), seed=s))
    return ca.DeviceGraph(ca.generate(g, n=n, gamma=case["gamma"], d=case["d"], seed=s))


def _batch(case, seed):
    """A mix of G(n,m), 2D geometric graphs and percolated grids, sizes spread over [2^lo, 2^hi] on a log scale and
    average degrees over [2, 16]; sizes, degrees and types are the case's alone, so that every seed has as many vertices."""
    rng, graphs = np.random.default_rng(4), []
    count = case["graphs"]
    sizes = np.rint(2.0 ** (case["lo"] + (case["hi"] - case["lo"]) * (rng.permutation(count) + 0.5) / count)).astype(int)
    degrees = rng.uniform(2.0, 16.0, count)
    for k in range(count):
        n, d, s = int(sizes[k]), float(degrees[k]), (seed * 8191 + k) % (1 << 30) + 1
        if k % 3 == 0:
            graphs.append(ca.generate("gnm_undirected", n=n, m=int(n * d / 2), seed=s))
        elif k % 3 == 1:
            graphs.append(ca.generate("rgg_2d", n=n, r=math.sqrt(d / (math.pi * n)), seed=s))
        else:
            side = int(round(math.sqrt(n)))
            graphs.append(ca.generate("grid_2d", nx=side, ny=side, p=min(1.0, d / 4), seed=s))
    return ca.BatchGraphs.pack(graphs)


def _model():
    """A model trained on traces of small graphs, as the benchmark trains its own on larger ones."""
    mlp = ca.Mlp(seed=1)
    for name, kw in (("gnm_undirected", dict(n=1 << 15, m=1 << 17, seed=1)),
                     ("rmat", dict(n=1 << 15, m=16 << 15, seed=3, rmat_a=0.57, rmat_b=0.19, rmat_c=0.19))):
        g = ca.DeviceGraph.generate(name, **kw)
        mlp.collect(g, stride=4, seed=11, seq_limit=0, stream=ca.STREAM_HASHED)
        g.close()
    mlp.train(steps=200, batch=4096)
    return mlp


def _rows(case, seed):
    """Feature rows and targets of the kind that traces hold: log2 degrees of a heavy-tailed graph, a clustering rate of
    quarters, a small round index; a target that grows with the neighbours' degrees."""
    rng = np.random.default_rng(seed)
    n = case["rows"]
    deg = np.floor(rng.pareto(1.8, n) * 4 + 1)
    mean = np.floor(rng.pareto(1.5, n) * 6 + 1)
    mx = mean * (1 + rng.random(n) * 3)
    X = np.stack([np.log2(1 + deg), np.log2(1 + mean), np.log2(1 + mx), np.log2(1 + deg * mean),
                  rng.integers(0, 3, n) / 2.0, rng.integers(0, 3, n)], 1).astype(np.float32)
    y = (0.8 * X[:, 2] + 0.3 * X[:, 0] + rng.random(n)).astype(np.float32)
    return X, y


def _weights(seed):
    """Weights that training starts from: uniform, scaled by the layers' widths; no biases."""
    rng = np.random.default_rng(seed + 1)
    u = lambda n, lim: rng.uniform(-lim, lim, n)  # noqa: E731
    return np.concatenate([u(6 * 64, 1.0), np.zeros(64), u(64 * 64, math.sqrt(6 / 64)), np.zeros(64),
                           u(64, math.sqrt(3 / 64)), np.zeros(1)]).astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "train":
        mlp = ca.Mlp(seed=1)
        mlp.set_weights(_weights(seed))
        mlp.add_dataset(*_rows(case, seed))
        return dict(case=case, mlp=mlp, seed=seed % 1000 + 1)
    if case["kind"] == "batch":
        b = ca.DeviceBatch(_batch(case, seed))
        b.set_tuning(block=case["block"], groups_per_cu=case["groups"], use_graph=True, split_vertices=case["split"])
        return dict(case=case, batch=b, kw=dict(seed=seed % 1000 + 1001, stream=ca.STREAM_HASHED))
    g = _host_or_device_graph(case, seed)
    kw = dict(seed=seed % 1000 + 1001, seq_limit=max(g.m // 256, 4096))
    if case["kind"] == "learned":
        mlp = _model()
        g.set_mlp(mlp)
        kw.update(variant="exp", use_bfs=True, stream=ca.STREAM_HASHED, learned=True)
    else:
        kw.update(variant=case["variant"], use_bfs=case["rounds"],
                  stream=ca.STREAM_HASHED if case["hashed"] else ca.STREAM_REFERENCE)
    return dict(case=case, graph=g, kw=kw)


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        st = state["mlp"].train(steps=case["steps"], batch=case["batch"], seed=state["seed"])
        return dict(weights=state["mlp"].get_weights(), first_loss=st["first_loss"], last_loss=st["last_loss"])
    if case["kind"] == "batch":
        labels, st = state["batch"].run(**state["kw"])
        return dict(labels=labels, components=st["components"], levels=st["levels_sum"], radius=st["radius_sum"])
    labels, st = state["graph"].find_components(**state["kw"])
    out = dict(labels=labels, components=st["components"])
    if case["kind"] == "graph":
        out.update(levels=st["levels"], radius=st["radius_sum"])
    return out


def work(case):
    if case["kind"] == "train":
        rows = case["batch"] * case["steps"]
        # forward, and two products of the backward pass, for each sampled row
        return dict(bytes=28.0 * min(case["rows"], rows) + 8.0 * ca.MLP_PARAMS,
                    flops=3.0 * 2.0 * rows * (6 * 64 + 64 * 64 + 64))
    if case["kind"] == "batch":
        n = case["graphs"] * (2 ** case["hi"] - 2 ** case["lo"]) / ((case["hi"] - case["lo"]) * math.log(2))
        m2 = 7.5 * n  # average degree over the batch's types
    else:
        n, m = _size(case)
        m2 = 2.0 * m
    # offsets and neighbour ids read, labels written
    flops = 2.0 * n * (6 * 64 + 64 * 64 + 64) if case["kind"] == "learned" else 0.0
    return dict(bytes=8.0 * (n + 1) + 4.0 * m2 + 4.0 * n, flops=flops)


# The samples of a training step come from counter-based SplitMix64 streams (Steele, Lea, Flood 2014).
def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
    return z ^ (z >> np.uint64(31))


def _samples(seed, step, batch, rows):
    """Row numbers of one step: 64-bit draws reduced to [0, rows) by a multiplication."""
    with np.errstate(over="ignore"):
        s = np.array([seed], np.uint64)
        base = _mix(_mix(s ^ np.uint64(12 << 40)) + np.uint64(12))
        i = np.arange(batch, dtype=np.uint64) + np.uint64(step * batch + 1)
        z = _mix(base + i * np.uint64(0x9e3779b97f4a7c15))
        lo, hi = z & np.uint64(0xffffffff), z >> np.uint64(32)
        r = np.uint64(rows)
        return ((hi * r + ((lo * r) >> np.uint64(32))) >> np.uint64(32)).astype(np.int64)


def exact(case, seed):
    """The trained weights and the losses in 64 bits, nothing rounded to bf16; the other cases return whole numbers."""
    if case["kind"] != "train":
        return None
    X, y = (a.astype(np.float64) for a in _rows(case, seed))
    w = _weights(seed).astype(np.float64)
    m, v = np.zeros_like(w), np.zeros_like(w)
    cut = np.cumsum([6 * 64, 64, 64 * 64, 64, 64])
    losses = []
    for step in range(case["steps"]):
        W1, b1, W2, b2, w3, b3 = np.split(w, cut)
        W1, W2 = W1.reshape(6, 64), W2.reshape(64, 64)
        rows = _samples(seed % 1000 + 1, step, case["batch"], case["rows"])
        x = X[rows]
        h1 = np.maximum(x @ W1 + b1, 0)
        h2 = np.maximum(h1 @ W2 + b2, 0)
        diff = h2 @ w3 + b3 - y[rows]
        losses.append(0.5 * float(np.mean(diff ** 2)))
        ds = diff / case["batch"]
        d2 = np.outer(ds, w3) * (h2 > 0)
        d1 = (d2 @ W2.T) * (h1 > 0)
        g = np.concatenate([(x.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0), h2.T @ ds, [ds.sum()]])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        w = w - 3e-3 * (m / (1 - 0.9 ** (step + 1))) / (np.sqrt(v / (1 - 0.999 ** (step + 1))) + 1e-8)
    return dict(weights=w, first_loss=losses[0], last_loss=losses[-1])
