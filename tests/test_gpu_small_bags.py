"""Trees on in-bag sets far smaller than the training set (needs an MI355X): the
bootstrap compaction moves whole rows however few samples it keeps.  Forests
of both searches equal the oracle's."""
import numpy as np
import pytest

import helpers
import oracle
from cudatree_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return _lib.default_context(0)


@pytest.fixture(scope="module")
def orc():
    return oracle.get()


@pytest.mark.parametrize("search", [_lib.CTA_SEARCH_ROWS, _lib.CTA_SEARCH_LISTS])
@pytest.mark.parametrize("N,F,n,T", [(2000, 500, 2, 20), (900, 1200, 5, 4), (70000, 24, 3, 6), (5000, 40, 1, 3)])
def test_few_in_bag(ctx, orc, N, F, n, T, search):
    rng = np.random.Generator(np.random.PCG64(N))
    y = rng.integers(0, 4, size=N)
    X = rng.standard_normal((N, F)).astype(np.float32)
    ids = [np.sort(rng.choice(N, n, replace=False)).astype(np.uint32) for _ in range(T)]
    ds = _lib.Dataset(ctx, X, y, 4)
    o = _lib.default_opts()
    o.seed, o.max_features, o.search = 11, 6, search
    print("few in-bag", N, F, n, T, search, flush=True)
    got = _lib.Forest.fit(ctx, ds, T, o, ids).export()
    want = orc.fit(X, y, 4, T, 6, boot_ids=ids, seed=11)
    assert helpers.forest_diff(got, want) is None
