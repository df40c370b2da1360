"""The fit's own choice between sorted rows and sample lists (needs an MI355X),
seen in the context's kernel statistics: by the sizes, by how the features'
values are spread, and that either search is the one that ran."""
import numpy as np
import pytest

import helpers
from cudatree_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return _lib.default_context(0)


def opts(m, seed=5, **kw):
    o = _lib.default_opts()
    o.max_features = m
    o.seed = seed
    o.bootstrap = 1
    for k, v in kw.items():
        setattr(o, k, v)
    return o


def profiled(ctx, ds, T, o, ids=None):
    """(forest, kernel statistics) of one fit."""
    ctx.reset_stats()
    ctx.set_profiling(True)
    try:
        f = _lib.Forest.fit(ctx, ds, T, o, ids).export()
    finally:
        ctx.set_profiling(False)
    return f, ctx.kernel_stats()


def search_of(stats):
    """Row scans take chunk histograms, list fits have none."""
    return "rows" if "k_scan_hist" in stats else "lists"


def dense(N, F, K, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    y = rng.integers(0, K, size=N)
    X = rng.standard_normal((N, F), dtype=np.float32) + (y[:, None] * 0.3).astype(np.float32)
    return X, y


def with_counts(N, F, K, share, rare, seed):
    """`share` of the features are zeros with small counts in `rare` of the
    samples, more in some classes than in others; the rest are continuous."""
    X, y = dense(N, F, K, seed)
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    k = int(round(share * F))
    lam = rare * (0.2 + 1.6 * rng.random((K, k)))
    X[:, :k] = (rng.random((N, k)) < lam[y]) * rng.integers(1, 9, size=(N, k))
    return X[:, rng.permutation(F)].copy(), y


def test_statistics_name_the_search(ctx):
    """The scans of either search have entries of their own, and only the row
    scan's, whose bytes are counted, gives a rate."""
    N, F, K, T, m = 6000, 40, 5, 4, 7
    X, y = dense(N, F, K, 6)
    ds = _lib.Dataset(ctx, X, y, K)
    print("statistics", flush=True)
    _, rows = profiled(ctx, ds, T, opts(m, search=_lib.CTA_SEARCH_ROWS))
    _, lists = profiled(ctx, ds, T, opts(m, search=_lib.CTA_SEARCH_LISTS))
    assert rows["k_scan"]["alg_bytes"] > 0 and "k_list_scan" not in rows
    assert lists["k_list_scan"]["ms"] > 0 and lists["k_list_scan"]["alg_bytes"] == 0 and "k_scan" not in lists


@pytest.mark.parametrize("share,rare,want", [(1.0, 0.003, "rows"),    # long chains of large nodes
                                             (1.0, 0.2, "lists"),
                                             (0.6, 0.0003, "rows"),   # constant in nearly every node
                                             (0.6, 0.02, "lists"),
                                             (0.0, 0.0, "lists")])
def test_choice_by_rare_values(ctx, share, rare, want):
    N, F, K, T, m = 20000, 300, 5, 40, 18
    X, y = with_counts(N, F, K, share, rare, 7)
    ds = _lib.Dataset(ctx, X, y, K)
    print("choice by rare values", share, rare, flush=True)
    _, st = profiled(ctx, ds, T, opts(m))
    assert search_of(st) == want


def test_constant_columns_are_not_read(ctx):
    """As many columns of one value beside the others leave the selection's time
    about where it was: such a column was read through in every node that drew
    it."""
    N, F, K, T, m = 30000, 250, 5, 20, 16
    X, y = dense(N, F, K, 8)
    Z = np.ones((N, 2 * F), np.float32)
    Z[:, ::2] = X
    ms = []
    for A in (X, Z):
        ds = _lib.Dataset(ctx, A, y, K)
        o = opts(m, search=_lib.CTA_SEARCH_LISTS)
        print("constant columns", A.shape, flush=True)
        profiled(ctx, ds, T, o)
        ms.append(profiled(ctx, ds, T, o)[1]["k_select"]["ms"])
    print(ms)
    assert ms[1] < 3.0 * ms[0], ms


@pytest.mark.parametrize("N,F,T,kw,want", [
    (20000, 1000, 50, {"max_depth": 1}, "rows"), (20000, 1000, 50, {"max_depth": 2, "bootstrap": 0}, "rows"),
    (20000, 1000, 50, {"max_depth": 8}, "lists"), (20000, 1000, 50, {"min_samples_split": 9000}, "rows"),
    (20000, 1000, 50, {"min_samples_split": 200}, "lists"),
    (3000, 400, 20, {"max_depth": 3}, "rows"), (3000, 400, 20, {"max_depth": 8}, "lists"),
    (3000, 190, 20, {}, "lists"), (3000, 179, 20, {}, "rows")])  # (both sides of 10 m)
def test_choice_by_depth(ctx, N, F, T, kw, want):
    """Trees of few levels spare too little for the list search's tables."""
    X, y = dense(N, F, 5, 9)
    m = 18 if F < 400 else int(np.ceil(F ** 0.5))
    ds = _lib.Dataset(ctx, X, y, 5)
    print("choice by depth", N, F, T, kw, flush=True)
    f, st = profiled(ctx, ds, T, opts(m, **kw))
    assert search_of(st) == want
    g, st = profiled(ctx, ds, T, opts(m, search=_lib.CTA_SEARCH_ROWS if want == "lists" else _lib.CTA_SEARCH_LISTS, **kw))
    assert search_of(st) != want and helpers.forest_diff(f, g) is None


def test_choice_by_in_bag_sets(ctx):
    """Few samples in-bag: rows of them are cheap to move after the compaction."""
    N, F, T, m = 100000, 100, 50, 2
    X, y = dense(N, F, 5, 10)
    rng = np.random.Generator(np.random.PCG64(11))
    ids = [np.sort(rng.choice(N, 50, replace=False)).astype(np.uint32) for _ in range(T)]
    ds = _lib.Dataset(ctx, X, y, 5)
    print("choice by in-bag sets", flush=True)
    assert search_of(profiled(ctx, ds, T, opts(m), ids)[1]) == "rows"
    assert search_of(profiled(ctx, ds, T, opts(m))[1]) == "lists"


@pytest.mark.parametrize("N,F,K,levels,T,R,want", [
    (40000, 300, 2, 0, 60, 4, "rows"), (40000, 300, 2, 0, 60, 6, "lists"),      # R (F - 8 m) (K + 11) from 10,500
    (40000, 300, 100, 0, 60, 2, "lists"),
    (32768, 300, 2, 0, 60, 2, "lists"),                                          # no node of more than 32,768
    (100000, 100, 5, 17, 40, 2, "rows"), (100000, 100, 5, 17, 40, 8, "lists")])  # few values: R F N from 2^26
def test_choice_by_trees_at_a_time(ctx, N, F, K, levels, T, R, want):
    """Few trees at a time leave too few workgroups for large nodes."""
    X, y = dense(N, F, K, 12)
    if levels:
        X = np.clip(np.round(X * 2 + levels // 2), 0, levels - 1).astype(np.float32)
    m = 17 if not levels else 10
    ds = _lib.Dataset(ctx, X, y, K)
    print("choice by trees at a time", N, F, K, levels, R, flush=True)
    f, st = profiled(ctx, ds, T, opts(m, trees_per_batch=R))
    assert search_of(st) == want
    g, st = profiled(ctx, ds, T, opts(m, trees_per_batch=T))
    assert search_of(st) == "lists" and helpers.forest_diff(f, g) is None


def test_choice_by_the_memory_for_trees(ctx):
    """The same where the workspace limit holds one tree at a time."""
    N, F, K, T, m = 40000, 300, 2, 60, 17
    X, y = dense(N, F, K, 13)
    c = _lib.Context(0)
    ds = _lib.Dataset(c, X, y, K)
    print("choice by the memory for trees", flush=True)
    want, st = profiled(c, ds, T, opts(m))
    assert search_of(st) == "lists"
    c.release_workspace()
    _lib.check(c.lib.cta_ctx_set_workspace_limit(c.h, 140 << 20))
    f, st = profiled(c, ds, T, opts(m))
    assert search_of(st) == "rows" and helpers.forest_diff(f, want) is None
    ds.close()
    c.close()


@pytest.mark.parametrize("kw,R,want", [({"min_samples_split": 200}, 4, "rows"), ({"min_samples_split": 200}, 30, "lists"),
                                       ({"max_depth": 7}, 8, "rows"), ({"max_depth": 7}, 9, "lists"), ({}, 4, "lists")])
def test_choice_by_cut_trees_at_a_time(ctx, kw, R, want):
    """Few trees at a time without their small nodes."""
    N, F, T, m = 8000, 500, 30, 17
    X, y = dense(N, F, 5, 14)
    ds = _lib.Dataset(ctx, X, y, 5)
    print("choice by cut trees at a time", kw, R, flush=True)
    f, st = profiled(ctx, ds, T, opts(m, trees_per_batch=R, **kw))
    assert search_of(st) == want
    g, st = profiled(ctx, ds, T, opts(m, **kw))
    assert search_of(st) == "lists" and helpers.forest_diff(f, g) is None


@pytest.mark.parametrize("T,want", [(5, "rows"), (12, "lists")])
def test_choice_by_partly_rare_few_values(ctx, T, want):
    """Features of 17 levels beside zeros in 0 to 100% of the samples: a share of
    them is rare enough to drag the constant tests of a large set."""
    N, F, m = 350000, 98, 10
    rng = np.random.Generator(np.random.PCG64(15))
    y = rng.integers(0, 2, size=N)
    X = np.clip(np.round(rng.standard_normal((N, F), dtype=np.float32) * 2 + 8 + y[:, None]), 0, 16)
    X *= rng.random((N, F), dtype=np.float32) < rng.random(F, dtype=np.float32) ** 2
    ds = _lib.Dataset(ctx, X.astype(np.float32), y, 2)
    print("choice by partly rare few values", T, flush=True)
    f, st = profiled(ctx, ds, T, opts(m))
    assert search_of(st) == want
    g, _ = profiled(ctx, ds, T, opts(m, search=_lib.CTA_SEARCH_ROWS if want == "lists" else _lib.CTA_SEARCH_LISTS))
    assert helpers.forest_diff(f, g) is None
