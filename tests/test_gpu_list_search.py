"""Split search from sample lists (needs an MI355X): forests grown with
search=CTA_SEARCH_LISTS equal the oracle's bit for bit, with root sizes on
both sides of every limit between the sorts (a wave's 64 to 1,024 samples, a
workgroup's 4,096 and 32,768, the filtered rows beyond), for features with gaps
below the candidate test's, many ties, infinities, constants and two values,
few and many classes, both index widths, and numbers of distinct values on both
sides of every limit of the counted features; and the fit's own choice grows
the forest of either search."""
import numpy as np
import pytest

import helpers
import oracle
from cudatree_amd import _lib, datasets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return _lib.default_context(0)


@pytest.fixture(scope="module")
def orc():
    return oracle.get()


def fit(ctx, case, search, idx_bits=0, **opts):
    ds = _lib.Dataset(ctx, case["X"], case["y"], case["K"], idx_bits=idx_bits)
    o = _lib.default_opts()
    o.seed = case["seed"]
    o.max_features = case["m"]
    o.min_samples_split = case["mss"]
    o.max_depth = case["max_depth"]
    o.identity_perm = int(case["identity"])
    o.search = search
    for k, v in opts.items():
        setattr(o, k, v)
    return _lib.Forest.fit(ctx, ds, case["n_trees"], o, helpers.case_boot_ids(case)).export()


def mixed(n, K, seed, F=10, m=4, n_trees=1, max_depth=4, mss=1):
    """Features: continuous; distinct values mostly closer than 1e-5; three of
    every four equal; 6 levels; 300 levels; infinities at both ends; constant;
    two-valued; nearly constant (two other values); a few hundred levels closer
    than 1e-5."""
    rng = np.random.Generator(np.random.PCG64(seed))
    y = rng.integers(0, K, size=n)
    y[:min(K, n)] = np.arange(min(K, n))
    X = rng.standard_normal((n, F)).astype(np.float32) + (y[:, None] % 7 * 0.2).astype(np.float32)
    X[:, 1] *= np.float32(3e-3 if n > 500 else 1e-5)
    X[rng.random(n) < 0.75, 2] = 0.0
    X[:, 3] = np.floor(X[:, 3] * 1.5)
    X[:, 4] = np.floor(X[:, 4] * 60)
    X[rng.random(n) < 0.01, 5] = np.inf
    X[rng.random(n) < 0.01, 5] = -np.inf
    X[:, 6] = 2.5
    X[:, 7] = rng.random(n) < 0.3
    X[:, 8] = 0.0
    X[n - 1, 8] = 1.0 if n % 2 else -1.0
    X[n // 2, 8] = 3.0
    X[:, 9] = np.floor(X[:, 9] * 40) * np.float32(4e-6)
    return {"X": X, "y": y, "K": K, "m": m, "mss": mss, "max_depth": max_depth, "identity": False, "seed": seed,
            "boot": False, "n_trees": n_trees}


def test_tiny_cases(ctx, orc):
    for s in range(60):
        case = datasets.tiny_case(s)
        print("list tiny seed=%d" % s, flush=True)
        d = helpers.forest_diff(fit(ctx, case, _lib.CTA_SEARCH_LISTS), helpers.oracle_forest(case, orc))
        assert d is None, "seed %d: %s" % (s, d)


@pytest.mark.parametrize("n,K", [(3, 2), (63, 2), (64, 4), (65, 5), (128, 3), (129, 7), (256, 2), (257, 20), (512, 4),
                                 (513, 300), (1024, 6), (1025, 3), (2048, 5), (2049, 9), (4096, 2), (4097, 4),
                                 (8192, 7), (8193, 100), (16384, 3), (16385, 6), (32768, 2),
                                 (32769, 4), (40001, 7), (70001, 20), (131072, 2)])
def test_sort_limits(ctx, orc, n, K):
    case = mixed(n, K, 1000 + n)
    print("list limits n=%d K=%d" % (n, K), flush=True)
    d = helpers.forest_diff(fit(ctx, case, _lib.CTA_SEARCH_LISTS), helpers.oracle_forest(case, orc))
    assert d is None, d


@pytest.mark.parametrize("idx_bits,opts", [(16, {}), (32, {}), (32, {"fill_global": 1, "resh_global": 1}),
                                           (16, {"scan_chunk": 64, "trees_per_batch": 2}),
                                           (16, {"scan_chunk": 1 << 20, "hist_layout": 2})])
def test_full_depth(ctx, orc, idx_bits, opts):
    """Bootstrapped trees down to their leaves, 40 features in use."""
    case = mixed(6001, 5, 77, F=40, m=7, n_trees=5, max_depth=0, mss=3)
    case["boot"] = True
    print("list full depth", idx_bits, opts, flush=True)
    d = helpers.forest_diff(fit(ctx, case, _lib.CTA_SEARCH_LISTS, idx_bits=idx_bits, **opts),
                            helpers.oracle_forest(case, orc))
    assert d is None, d


@pytest.mark.parametrize("D,K", [(64, 3), (65, 3), (128, 10), (129, 10), (256, 9), (256, 20), (257, 20), (512, 20),
                                 (513, 3), (1024, 20), (1025, 3)])
def test_counted_values(ctx, orc, D, K):
    rng = np.random.Generator(np.random.PCG64(D))
    n = 12001
    y = rng.integers(0, K, size=n)
    X = rng.integers(0, D, size=(n, 3)).astype(np.float32)
    X[:, 1] = np.minimum(np.abs(rng.standard_normal(n) * D / 8 + y * D / (2 * K)).astype(np.int64), D - 1)
    X[:D, :] = np.arange(D)[:, None]
    case = {"X": X, "y": y, "K": K, "m": 3, "mss": 1, "max_depth": 4, "identity": False, "seed": D, "boot": False,
            "n_trees": 2}
    print("list counted D=%d K=%d" % (D, K), flush=True)
    d = helpers.forest_diff(fit(ctx, case, _lib.CTA_SEARCH_LISTS), helpers.oracle_forest(case, orc))
    assert d is None, d


@pytest.mark.parametrize("n,F,m,T,levels", [(4096, 40, 4, 3, 0), (4097, 40, 4, 400, 0), (4097, 80, 6, 126, 0),
                                            (40000, 48, 4, 70, 10), (40000, 48, 4, 69, 10), (40000, 48, 4, 70, 2)])
def test_choice(ctx, n, F, m, T, levels):
    """Both sides of the size rule, few and many values (levels = 0)."""
    rng = np.random.Generator(np.random.PCG64(n + T))
    y = rng.integers(0, 3, size=n)
    X = (rng.standard_normal((n, F)) + y[:, None] * 0.3).astype(np.float32)
    if levels:
        X = np.clip(np.floor(X + levels / 2), 0, levels - 1).astype(np.float32)
    case = {"X": X, "y": y, "K": 3, "m": m, "mss": 1, "max_depth": 5, "identity": False, "seed": 3, "boot": False,
            "n_trees": T}
    print("list choice", n, F, m, T, levels, flush=True)
    auto = fit(ctx, case, _lib.CTA_SEARCH_AUTO)
    for search in (_lib.CTA_SEARCH_ROWS, _lib.CTA_SEARCH_LISTS):
        d = helpers.forest_diff(auto, fit(ctx, case, search))
        assert d is None, d
