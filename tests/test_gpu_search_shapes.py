"""Both searches at the sizes where their kernels differ (needs an MI355X), each
named by the context's kernel statistics: the row search on the shapes whose
default is the list search, against the oracle; the list search's workgroup
kernels with classes past a wave's registers and past 8 bits, bootstrapped
roots that are filtered from the presorted row, two lanes, and sample sets too
large for the LDS."""
import numpy as np
import pytest

import helpers
import oracle
from cudatree_amd import _lib, datasets
from test_gpu_search_choice import opts, profiled, search_of

pytestmark = pytest.mark.gpu

SEARCHES = (_lib.CTA_SEARCH_ROWS, _lib.CTA_SEARCH_LISTS)


@pytest.fixture(scope="module")
def ctx():
    c = _lib.default_context(0)
    yield c
    c.release_workspace()


@pytest.fixture(scope="module")
def orc():
    return oracle.get()


def gaussian():
    return datasets.gaussian_clusters() + (16,)


def zipf():
    return datasets.zipf_quantized() + (8,)


def wide():
    return datasets.wide_sparse_signal() + (64,)


# 200,000 x 256, 20 classes; 1,000,000 x 64, 100 classes; 20,000 x 4,096 (above
# the reshuffle's limit of rows for its big tasks), 5 classes
@pytest.mark.parametrize("data", [gaussian, zipf, wide])
def test_either_search_on_the_large_shapes(ctx, orc, data):
    """The first of two trees against the oracle, from rows and from lists."""
    X, y, m = data()
    K = int(y.max()) + 1
    ds = _lib.Dataset(ctx, X, y, K)
    want = orc.fit(X, y, K, 1, m, boot_ids=orc.bootstrap_forest_ids(1005, 1, len(y)), seed=1005)
    for search, name in zip(SEARCHES, ("rows", "lists")):
        print("large shapes", data.__name__, name, flush=True)
        got, st = profiled(ctx, ds, 2, opts(m, seed=1005, search=search))
        assert search_of(st) == name
        assert helpers.forest_diff(helpers.forest_slice(got, 0, 1), want) is None


def mixed(N, F, K, seed, levels):
    """Continuous features and, of every three, one of `levels` values."""
    rng = np.random.Generator(np.random.PCG64(seed))
    y = rng.integers(0, K, size=N)
    X = rng.standard_normal((N, F)).astype(np.float32) + (y[:, None] % 11 * 0.1).astype(np.float32)
    X[:, ::3] = np.clip(np.floor(X[:, ::3] * levels / 8 + levels / 2), 0, levels - 1)
    return X, y


# kernels: workgroups of 4 and 16 waves that sort, the filtered row, the counts of
# 16 and 4 waves
@pytest.mark.parametrize("N,K,levels,kernels", [
    (4000, 70, 13, ["k_list_mid"]), (4000, 300, 13, ["k_list_mid", "k_list_hist4"]),
    (20000, 100, 100, ["k_list_mid", "k_list_big", "k_list_hist"]),
    (20000, 300, 60, ["k_list_mid", "k_list_big", "k_list_hist"]),
    (60000, 100, 90, ["k_list_big", "k_list_filter", "k_list_hist"]),
    (60000, 300, 12, ["k_list_big", "k_list_filter", "k_list_hist", "k_list_hist4"]),
    (90001, 470, 30, ["k_list_filter", "k_list_hist"])])
def test_workgroup_kernels_with_many_classes(ctx, orc, N, K, levels, kernels):
    """Bootstrapped trees of six levels; the larger roots hold more than 32,768
    in-bag samples."""
    X, y = mixed(N, 9, K, N + K, levels)
    ds = _lib.Dataset(ctx, X, y, K)
    print("workgroup kernels", N, K, levels, flush=True)
    got, st = profiled(ctx, ds, 2, opts(5, seed=21, search=_lib.CTA_SEARCH_LISTS, max_depth=6))
    assert search_of(st) == "lists" and all(k in st for k in kernels), sorted(st)
    want = orc.fit(X, y, K, 2, 5, boot_ids=orc.bootstrap_forest_ids(21, 2, N), seed=21, max_depth=6)
    assert helpers.forest_diff(got, want) is None
    if "k_list_filter" in kernels:
        assert got["n_samples"][0] > 32768


def test_two_lanes(ctx, orc):
    X, y = mixed(9000, 12, 6, 31, 40)
    ds = _lib.Dataset(ctx, X, y, 6)
    print("two lanes", flush=True)
    got, st = profiled(ctx, ds, 24, opts(4, seed=22, search=_lib.CTA_SEARCH_LISTS, lanes=2))
    assert search_of(st) == "lists"
    want = orc.fit(X, y, 6, 24, 4, boot_ids=orc.bootstrap_forest_ids(22, 24, 9000), seed=22)
    assert helpers.forest_diff(got, want) is None


@pytest.mark.parametrize("N,F,K,levels", [(1400000, 4, 3, 50), (90001, 9, 1000, 30)])
def test_sizes_that_lists_do_not_take(ctx, orc, N, F, K, levels):
    """A node's sample set, or a large node's words beside the class counts of 16
    waves, is larger than the LDS: rows, also where lists are asked for."""
    X, y = mixed(N, F, K, N + K, levels)
    ds = _lib.Dataset(ctx, X, y, K)
    print("sizes that lists do not take", N, K, flush=True)
    got, st = profiled(ctx, ds, 1, opts(2, seed=23, search=_lib.CTA_SEARCH_LISTS, max_depth=5))
    assert search_of(st) == "rows"
    want = orc.fit(X, y, K, 1, 2, boot_ids=orc.bootstrap_forest_ids(23, 1, N), seed=23, max_depth=5)
    assert helpers.forest_diff(got, want) is None
