"""The work that users of cudatree_amd have it do, as measurable cases.

A case is a dict of plain values.  Three kinds of work are covered:

``fit``      grow a forest: transpose, presort and value codes of the training
             set, bootstrap, every level of every tree, canonical trees in the
             caller's host arrays.  ``path`` "host" goes through
             RandomForestClassifier with numpy arrays (upload and label
             compaction included), "device" through the C-ABI with the
             training set already in device memory.
``predict``  labels and votes of a fitted forest.  ``path`` "host" / "proba":
             RandomForestClassifier on numpy rows; "device" / "noalloc": the
             device-pointer entry points on resident rows.
``serve``    a burst of small requests through the serving loop.

The data sets follow the generators of cudatree_amd.datasets (same layouts and
distributions), drawn on the device where the program holds them there:
``digits`` (small integers, many ties), ``tabular`` (class-conditional Gaussian
mixtures beside one-hot groups), ``gauss`` (continuous clusters), ``zipf``
(many skewed classes, 256 levels per feature) and ``wide`` (few rows, thousands
of mostly uninformative features).

Trees, labels and votes are whole numbers, and a threshold is the float32
midpoint of two input values; no forest can be grown in 64-bit numpy without
this package's node order, so ``exact`` has no values to give.
"""
import ctypes
import math

import numpy as np
import torch

from cudatree_amd import RandomForestClassifier, _lib, datasets

_DEV = "cuda:0"


def listed():
    return [
        # The package's introductory example: a digits-sized set from numpy
        # arrays, 50 trees; latency of many small levels.
        _fit("fit_digits_host", "digits", 1797, 64, 10, 50, path="host"),
        # An everyday table from numpy arrays with an odd size, leaves of a
        # minimum size, a depth cap and no bootstrap; 16-bit row entries.
        _fit("fit_table_host", "tabular", 50021, 37, 4, 30, path="host", bootstrap=False, mss=20, max_depth=18),
        # The headline workload: covtype-shaped table resident in HBM.
        _fit("fit_covtype", "tabular", 581012, 54, 7, 50),
        # Many continuous features and classes, a large forest.
        _fit("fit_gauss", "gauss", 200000, 256, 20, 200),
        # The largest: a million samples, 100 skewed classes, quantised
        # features full of ties.
        _fit("fit_zipf", "zipf", 1000000, 64, 100, 100),
        # Short and wide (4,096 features, 16-bit row entries).
        _fit("fit_wide", "wide", 20000, 4096, 5, 100),
        # One small scoring request from numpy: latency.
        _predict("predict_16_host", "tabular", 581012, 54, 7, 50, 16, path="host"),
        # Class probabilities of a batch from numpy, 100 classes.
        _predict("proba_20k_host", "zipf", 100003, 64, 100, 30, 20011, path="proba"),
        # A small resident batch where the caller forbids allocation.
        _predict("predict_1k_noalloc", "tabular", 581012, 54, 7, 50, 1000, path="noalloc"),
        # Bulk scoring of a held-out set resident in HBM.
        _predict("predict_100k", "tabular", 581012, 54, 7, 50, 100000),
        # A large request on a large serving forest.
        _predict("predict_64k_500t", "tabular", 581012, 54, 7, 500, 65536, max_depth=24),
        # A client that hands the serving loop 2,000 gathered small requests.
        dict(_predict("serve_burst", "tabular", 581012, 54, 7, 200, 2000, max_depth=24), kind="serve", largest=64),
    ]


def _fit(name, data, N, F, K, T, path="device", bootstrap=True, mss=1, max_depth=0):
    return {"name": name, "kind": "fit", "data": data, "N": N, "F": F, "K": K, "T": T, "m": int(math.ceil(F ** 0.5)),
            "path": path, "bootstrap": bootstrap, "mss": mss, "max_depth": max_depth}


def _predict(name, data, N, F, K, T, R, path="device", max_depth=0):
    c = _fit(name, data, N, F, K, T, max_depth=max_depth)
    c.update(kind="predict", path=path, R=R)
    return c


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges; its cost stays below the largest
    listed one's (rows x features x trees of a fit, rows x trees of a predict)."""
    kind = rng.choice(["fit", "fit", "fit", "predict", "predict", "serve"])
    if kind == "fit":
        data = rng.choice(["digits", "tabular", "tabular", "gauss", "zipf", "wide"])
        N = _log_int(rng, 1000, 1000000)
        F = _log_int(rng, 8, 256)
        if data == "wide":
            N, F = _log_int(rng, 500, 20000), _log_int(rng, 257, 4096)
        if data == "tabular":
            F = max(F, 16)
        K = _log_int(rng, 2, 20 if data != "zipf" else 100)
        N = max(500, min(N, 60000000 // F))
        T = _log_int(rng, 5, 200)
        T = max(1, min(T, int(2.5e9 // (N * F))))
        path = rng.choice(["host", "device"]) if N * F <= 8000000 else "device"
        c = _fit("", data, N, F, K, T, path=path, bootstrap=rng.random() < 0.8,
                 mss=rng.choice([1, 1, 2, 10, 50]), max_depth=rng.choice([0, 0, 0, 8, 20]))
    else:
        data = rng.choice(["digits", "tabular", "gauss", "zipf"])
        N = _log_int(rng, 2000, 400000)
        F = _log_int(rng, 16, 128)
        K = _log_int(rng, 2, 20 if data != "zipf" else 100)
        T = _log_int(rng, 5, 500)
        T = max(1, min(T, int(2.0e9 // (N * F))))
        depth = rng.choice([0, 0, 12, 24])
        if kind == "predict":
            path = rng.choice(["host", "proba", "device", "device", "noalloc"])
            hi = {"host": 50000, "proba": 50000, "device": 100000, "noalloc": (1 << 20) // K}[path]
            c = _predict("", data, N, F, K, T, _log_int(rng, 1, min(hi, 100000)), path=path, max_depth=depth)
        else:
            c = dict(_predict("", data, N, F, K, T, _log_int(rng, 50, 4000), max_depth=depth), kind="serve",
                     largest=rng.choice([16, 64, 256]))
    del c["name"]
    return c


# ---- inputs ---------------------------------------------------------------------
def _data(case, seed, rows, dev):
    """(X, y) of `rows` samples on `dev`, every class present."""
    data, F, K = case["data"], case["F"], case["K"]
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def rand(*s):
        return torch.rand(*s, generator=g, device=dev)

    def randn(*s):
        return torch.randn(*s, generator=g, device=dev)

    def randint(hi, *s):
        return torch.randint(0, hi, s, generator=g, device=dev)

    if data == "tabular":
        # class shares falling as in covtype's table, then a tail
        p = torch.tensor([datasets.COVTYPE_PROPORTIONS[k] if k < 7 else 0.01 for k in range(K)], device=dev,
                         dtype=torch.float32)
    elif data == "zipf":
        p = 1.0 / torch.arange(1, K + 1, device=dev, dtype=torch.float32) ** 1.1
    else:
        p = torch.ones(K, device=dev)
    cum = torch.cumsum(p / p.sum(), 0)
    y = torch.clamp(torch.searchsorted(cum, rand(rows)), max=K - 1)
    y[:K] = torch.arange(K, device=dev)[:rows]
    if data == "digits":
        centroid = randint(17, K, F).float()
        X = torch.clamp(torch.round(centroid[y] + 3.0 * randn(rows, F)), 0, 16)
    elif data == "tabular":
        C = min(10, F)
        X = torch.zeros(rows, F, device=dev)
        mean, sig = 4000.0 * rand(K, C, 2), 4000.0 * (0.05 + 0.1 * rand(K, C, 2))
        comp = randint(2, rows, C)
        cols = torch.arange(C, device=dev)[None, :]
        X[:, :C] = mean[y[:, None], cols, comp] + sig[y[:, None], cols, comp] * randn(rows, C)
        lo = C
        while lo < F:
            width = min(4 if lo == C else 40, F - lo)
            w = -torch.log(rand(K, width).clamp_min(1e-9))  # Dirichlet(1) shares per class
            cc = torch.cumsum(w / w.sum(1, keepdim=True), 1)
            cat = torch.clamp((rand(rows)[:, None] > cc[y]).sum(1), max=width - 1)
            X[torch.arange(rows, device=dev), lo + cat] = 1.0
            lo += width
    elif data == "gauss":
        centroids = 2.0 * randn(K, 3, F)
        X = centroids[y, randint(3, rows)]
        X += randn(rows, F)
    elif data == "zipf":
        centroids = randn(K, F)
        X = centroids[y]
        X += randn(rows, F)
        a, b = X.min(0).values, X.max(0).values
        X = torch.floor((X - a) / (b - a) * 255.0 + 0.5)
    else:
        X = randn(rows, F)
        s = min(64, F)
        X[:, :s] += (randint(2, K, s).float() - 0.5)[y]
    return X.contiguous(), y.to(torch.int32).contiguous()


def _opts(case, seed):
    o = _lib.default_opts()
    o.seed = seed * 7919 + 17
    o.max_features = case["m"]
    o.min_samples_split = case["mss"]
    o.max_depth = case["max_depth"]
    o.bootstrap = int(case["bootstrap"])
    return o


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _device_fit(ctx, case, X, y, opts):
    ds = ctypes.c_void_p()
    forest = ctypes.c_void_p()
    _lib.check(ctx.lib.cta_dataset_create_device(ctx.h, _ptr(X), _ptr(y), X.shape[0], case["F"], case["K"], 0,
                                                 ctypes.byref(ds)))
    try:
        _lib.check(ctx.lib.cta_fit(ctx.h, ds, case["T"], None, None, ctypes.byref(opts), ctypes.byref(forest)))
    finally:
        ctx.lib.cta_dataset_destroy(ds)
    return _lib.Forest(ctx, forest)


def prepare(case, seed):
    ctx = _lib.default_context(0)
    st = {"case": case, "ctx": ctx}
    if case["kind"] == "fit":
        X, y = _data(case, seed, case["N"], _DEV)
        if case["path"] == "host":
            st["clf"] = RandomForestClassifier(case["T"], max_features=case["m"], min_samples_split=case["mss"],
                                               bootstrap=case["bootstrap"], max_depth=case["max_depth"] or None,
                                               random_state=seed)
            X, y = X.cpu().numpy(), y.cpu().numpy().astype(np.int64)
        else:
            st["opts"] = _opts(case, seed)
        st["X"], st["y"] = X, y
        cap = _capacity(case)
        st["out"] = {k: np.zeros(cap, dt) for k, dt in _NODE_ARRAYS}
        st["out"]["tree_off"] = np.zeros(case["T"] + 1, np.int64)
        torch.cuda.synchronize()
        return st
    # a fitted forest and rows it has not seen, of the same distribution
    if case["kind"] == "serve":
        # the request sizes go with the case, the rows with the seed
        r = np.random.default_rng([case["R"], case["largest"]])
        sizes = np.exp(r.uniform(0, np.log(case["largest"] + 1), size=case["R"])).astype(np.int64)
        sizes = np.clip(sizes, 1, case["largest"])
        R = int(sizes.sum())
    else:
        R = case["R"]
    X, y = _data(case, seed, case["N"] + R, _DEV)
    rows = X[case["N"]:].contiguous()
    X, y = X[:case["N"]].contiguous(), y[:case["N"]].contiguous()
    torch.cuda.synchronize()
    if case["path"] in ("host", "proba") and case["kind"] == "predict":
        st["clf"] = RandomForestClassifier(case["T"], max_features=case["m"], max_depth=case["max_depth"] or None,
                                           random_state=seed).fit(X.cpu().numpy(), y.cpu().numpy())
        st["rows"] = rows.cpu().numpy()
        return st
    forest = _device_fit(ctx, case, X, y, _opts(case, seed))
    if case["kind"] == "serve":
        st["rows"], st["sizes"] = rows.cpu().numpy(), sizes
        st["server"] = _lib.Server()
        st["fid"] = st["server"].add_forest(forest)
    else:
        st["forest"], st["rows"] = forest, rows
        st["labels"] = torch.empty(R, dtype=torch.int32, device=_DEV)
        st["votes"] = torch.empty(R, case["K"], dtype=torch.int32, device=_DEV) if case["path"] == "device" else None
        torch.cuda.synchronize()
    return st


# ---- one pass -------------------------------------------------------------------
_NODE_ARRAYS = (("feature", np.int32), ("threshold", np.float32), ("left", np.uint32), ("right", np.uint32),
                ("value", np.uint32), ("n_samples", np.uint32), ("depth", np.uint32))


def _capacity(case):
    """Entries of the program's node arrays: twice the in-bag samples holds
    any forest; large forests of these data sets stay well below that."""
    n = int(case["N"] * (0.66 if case["bootstrap"] else 1.0)) * case["T"]
    share = {"digits": 0.6, "tabular": 0.6, "gauss": 0.6, "wide": 1.6,
             "zipf": 0.6 if case["F"] >= 32 else 1.4}[case["data"]]
    return 2 * n + case["T"] if n <= 1000000 else int(share * n)


def _export(st, forest):
    """The trees in the node arrays that the program keeps from fit to fit
    (zero past the last node)."""
    o = st["out"]
    if forest.n_nodes > len(o["feature"]):
        raise MemoryError("%d nodes exceed the program's arrays" % forest.n_nodes)

    def p(k, t):
        return o[k].ctypes.data_as(ctypes.POINTER(t))

    _lib.check(forest.lib.cta_forest_export(
        forest.h, p("tree_off", ctypes.c_int64), p("feature", ctypes.c_int32), p("threshold", ctypes.c_float),
        p("left", ctypes.c_uint32), p("right", ctypes.c_uint32), p("value", ctypes.c_uint32),
        p("n_samples", ctypes.c_uint32), p("depth", ctypes.c_uint32)))
    return o


def run(st):
    case, ctx = st["case"], st["ctx"]
    if case["kind"] == "fit":
        if case["path"] == "host":
            trees = st["clf"].fit(st["X"], st["y"]).export_trees()
            for k, v in trees.items():
                st["out"][k][:len(v)] = v
            return st["out"]
        forest = _device_fit(ctx, case, st["X"], st["y"], st["opts"])
        out = _export(st, forest)
        forest.close()
        return out
    if case["kind"] == "serve":
        tickets, labels = st["server"].submit_rows(st["fid"], st["rows"], st["sizes"])
        status = st["server"].wait_many(tickets)
        return {"labels": labels, "status": status}
    if case["path"] == "host":
        return st["clf"].predict(st["rows"])
    if case["path"] == "proba":
        return st["clf"].predict_proba(st["rows"])
    rows, labels, votes, forest = st["rows"], st["labels"], st["votes"], st["forest"]
    if case["path"] == "noalloc":
        _lib.check(ctx.lib.cta_predict_device_noalloc(ctx.h, forest.h, _ptr(rows), rows.shape[0], case["F"],
                                                      _ptr(labels)))
        return labels
    _lib.check(ctx.lib.cta_predict_device(ctx.h, forest.h, _ptr(rows), rows.shape[0], case["F"], _ptr(labels),
                                          _ptr(votes)))
    return {"labels": labels, "votes": votes}


# ---- accounting -----------------------------------------------------------------
# nodes per in-bag sample of fully grown trees of each data set, about
_NODES = {"digits": 0.05, "tabular": 0.06, "gauss": 0.05, "zipf": 0.3, "wide": 0.45}


def _tree(case):
    """(in-bag samples, nodes, mean leaf depth) of one tree, about."""
    n = case["N"] * (0.632 if case["bootstrap"] else 1.0)
    nodes = max(3.0, _NODES[case["data"]] * n / max(1.0, case["mss"] / 2.0))
    depth = 1.4 * math.log2(nodes + 1)
    if case["max_depth"]:
        depth = min(depth, case["max_depth"])
        nodes = min(nodes, 2.0 ** min(case["max_depth"] + 1, 60))
    return n, nodes, depth


def work(case):
    """Bytes: the training set (or the rows and the node table) read once, the
    trees (or labels and votes) written once.  Operations: about ten per
    in-bag sample, evaluated feature and level of a fit (rank, two running
    sums, the score and its comparison); two per (row, tree, level) of a walk."""
    n, nodes, depth = _tree(case)
    F, K, T = case["F"], case["K"], case["T"]
    if case["kind"] == "fit":
        return {"bytes": float(case["N"] * (F * 4 + 4) + T * nodes * 28), "flops": float(10 * T * n * case["m"] * depth)}
    R = case["R"]
    if case["kind"] == "serve":
        R = int(case["R"] * (case["largest"] / math.log(case["largest"] + 1)))
    out = 4 + (K * 4 if case["path"] in ("device", "proba") else 0)
    return {"bytes": float(R * (F * 4 + out) + min(T * nodes, R * T * depth) * 16), "flops": float(2 * R * T * depth)}


def exact(case, seed):
    """No 64-bit counterpart: trees, labels and votes are whole numbers that
    stay equal, and thresholds are float32 midpoints of input values."""
    return None
