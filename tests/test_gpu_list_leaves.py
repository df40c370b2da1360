"""Leaves labelled by their first sample in feature 0's presorted order (needs an
MI355X): children below min_samples_split and whole trees that are such a
leaf.  The list search keeps samples in another order and has to find it: its
forests equal the oracle's, and finding it in large leaves costs no more than a
few times the row search's children step."""
import numpy as np
import pytest

import helpers
import oracle
from cudatree_amd import _lib
from test_gpu_search_choice import profiled

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return _lib.default_context(0)


@pytest.fixture(scope="module")
def orc():
    return oracle.get()


def levels(N, F, K, L, seed):
    """Features of L levels, the last four of two, feature 0 of many values."""
    rng = np.random.Generator(np.random.PCG64(seed))
    y = rng.integers(0, K, size=N)
    X = np.clip(np.floor(rng.standard_normal((N, F)) * L / 6 + L / 2 + (y[:, None] % 3)), 0, L - 1).astype(np.float32)
    X[:, -4:] = X[:, -4:] > L / 2
    X[:, 0] = np.floor(rng.standard_normal(N) * 50)
    return X, y


@pytest.mark.parametrize("N,F,mss,boot,idx_bits", [(63, 9, 30, False, 0), (700, 9, 500, True, 0),
                                                   (5000, 12, 2500, False, 32), (5000, 12, 1200, True, 16),
                                                   (40001, 8, 20000, False, 0), (40001, 8, 9000, True, 0),
                                                   (70001, 6, 60000, False, 0)])
def test_leaves_below_min_samples_split(ctx, orc, N, F, mss, boot, idx_bits):
    X, y = levels(N, F, 5, 40, N)
    ids = [np.unique(np.random.default_rng([N, t]).integers(0, N, N)).astype(np.uint32) for t in range(3)] if boot else None
    ds = _lib.Dataset(ctx, X, y, 5, idx_bits=idx_bits)
    o = _lib.default_opts()
    o.seed, o.max_features, o.search, o.min_samples_split = 3, 3, _lib.CTA_SEARCH_LISTS, mss
    print("first-sample leaves", N, F, mss, boot, flush=True)
    got = _lib.Forest.fit(ctx, ds, 3, o, ids).export()
    want = orc.fit(X, y, 5, 3, 3, boot_ids=ids, seed=3, min_samples_split=mss)
    assert helpers.forest_diff(got, want) is None
    assert (got["left"] == 0).sum() >= 3


def test_large_leaves_are_labelled_in_parallel(ctx):
    """300,000 x 64, 40 trees of leaves below 150,000 samples."""
    N, F, K, T = 300000, 64, 20, 40
    X, y = levels(N, F, K, 256, 1)
    ds = _lib.Dataset(ctx, X, y, K)
    ms = {}
    for search in (_lib.CTA_SEARCH_ROWS, _lib.CTA_SEARCH_LISTS):
        o = _lib.default_opts()
        o.seed, o.max_features, o.min_samples_split, o.search = 4, 8, N // 2, search
        print("large leaves", search, flush=True)
        profiled(ctx, ds, T, o)
        f, st = profiled(ctx, ds, T, o)
        ms[search] = (f, st["k_children"]["ms"])
    rows, lists = ms[_lib.CTA_SEARCH_ROWS], ms[_lib.CTA_SEARCH_LISTS]
    print("k_children rows %.3f lists %.3f ms" % (rows[1], lists[1]))
    assert helpers.forest_diff(rows[0], lists[0]) is None
    assert lists[1] < 4.0 * rows[1] + 0.5


@pytest.mark.parametrize("N,n,idx_bits", [(3, 0, 0), (900, 0, 16), (900, 40, 32), (30011, 0, 0), (30011, 16000, 16),
                                          (30011, 900, 0), (70001, 3, 0), (70001, 1500, 0)])
def test_whole_trees_below_min_samples_split(ctx, orc, N, n, idx_bits):
    """Every root is such a leaf; the in-bag samples (n of them, 0: all) are the
    last ones of feature 0's order in the first tree, so their first lies far
    down the presorted row, and drawn at random in the others."""
    X, y = levels(N, 9, 3, 30, N + n)
    T = 5
    ids = None
    if n:
        rng = np.random.default_rng(n)
        ids = [np.sort(np.argsort(X[:, 0], kind="stable")[-n:]).astype(np.uint32)]
        ids += [np.sort(rng.choice(N, n, replace=False)).astype(np.uint32) for _ in range(T - 1)]
    ds = _lib.Dataset(ctx, X, y, 3, idx_bits=idx_bits)
    o = _lib.default_opts()
    o.seed, o.max_features, o.search, o.min_samples_split = 3, 3, _lib.CTA_SEARCH_LISTS, N + 1
    print("whole trees below min_samples_split", N, n, flush=True)
    got = _lib.Forest.fit(ctx, ds, T, o, ids).export()
    want = orc.fit(X, y, 3, T, 3, boot_ids=ids, seed=3, min_samples_split=N + 1)
    assert helpers.forest_diff(got, want) is None
    assert len(got["feature"]) == T


def test_root_labels_far_down_the_row(ctx):
    """20 trees of the last 50 of 500,000 samples in feature 0's order: the list
    fit takes no more than a few times the row fit's setup."""
    N, n, T = 500000, 50, 20
    X, y = levels(N, 6, 5, 40, 9)
    ids = [np.sort(np.argsort(X[:, 0], kind="stable")[-n:]).astype(np.uint32)] * T
    ds = _lib.Dataset(ctx, X, y, 5)
    ms = []
    for search in (_lib.CTA_SEARCH_ROWS, _lib.CTA_SEARCH_LISTS):
        o = _lib.default_opts()
        o.seed, o.max_features, o.search, o.min_samples_split = 3, 2, search, 100
        print("root labels", search, flush=True)
        profiled(ctx, ds, T, o, ids)
        f, st = profiled(ctx, ds, T, o, ids)
        ms.append((f, st["host_setup"]["ms"]))
    print("setup rows %.3f lists %.3f ms" % (ms[0][1], ms[1][1]))
    assert helpers.forest_diff(ms[0][0], ms[1][0]) is None
    assert ms[1][1] < 4.0 * ms[0][1] + 2.0
