"""The list search's cost on features that suit it badly (needs an MI355X), seen
in the context's kernel statistics."""
import numpy as np
import pytest

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


def dense(N, F, K, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    y = rng.integers(0, K, size=N)
    X = rng.standard_normal((N, F), dtype=np.float32) + (y[:, None] * 0.3).astype(np.float32)
    return X, y


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
