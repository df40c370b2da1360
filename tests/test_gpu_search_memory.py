"""Memory and the choice of search (needs an MI355X): the list search's tables
take device memory that sorted rows do not, so a fit that may use either goes
back to rows where they do not fit, and grows the same trees."""
import ctypes

import numpy as np
import pytest

import helpers
from cudatree_amd import _lib

pytestmark = pytest.mark.gpu


def gauss(N, F, K, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    y = rng.integers(0, K, size=N)
    X = rng.standard_normal((N, F), dtype=np.float32) + (y[:, None] * 0.3).astype(np.float32)
    return X, y


def opts(m, seed=5, **kw):
    o = _lib.default_opts()
    o.max_features = m
    o.seed = seed
    o.bootstrap = 1
    for k, v in kw.items():
        setattr(o, k, v)
    return o


@pytest.mark.parametrize("spare", [1 << 20, 1 << 30])
def test_server_admits_what_sorted_rows_need(spare):
    """A job whose estimate over sorted rows fits the budget is admitted, also
    where the list search's tables do not fit beside it (the small spare)."""
    N, F, K, T, m = 3000, 400, 5, 20, 20
    X, y = gauss(N, F, K, 1)
    rows = sum(_lib.fit_estimate(N, F, K, T, opts(m, search=_lib.CTA_SEARCH_ROWS)))
    either = sum(_lib.fit_estimate(N, F, K, T, opts(m)))
    assert either > rows + (1 << 20)  # lists are the fit's own choice here, and cost more
    ctx = _lib.default_context(0)
    want = _lib.Forest.fit(ctx, _lib.Dataset(ctx, X, y, K), T, opts(m), None).export()
    print("server admission spare=%d" % spare, flush=True)
    srv = _lib.Server(hbm_budget=rows + spare)
    try:
        st, fid = srv.wait(srv.submit_fit(X, y, K, T, opts(m)))
        assert st == 0
        assert helpers.forest_diff(srv.export_forest(fid), want) is None
        s = srv.stats()
        assert s["fit_rejected"] == 0 and s["hbm_peak"] <= rows + spare and s["fit_mem_ratio_max"] <= 1.0, s
    finally:
        srv.close()


class Hog:
    """Device memory taken until about `leave` bytes are free."""

    def __init__(self, ctx, leave):
        self.held = []
        chunk = 16 << 30
        while chunk >= 1 << 20:
            if ctx.mem_info()[0] <= leave + chunk:
                chunk >>= 1
                continue
            self.held.append(helpers.DeviceArray(chunk, np.uint8))

    def free(self):
        for d in self.held:
            d.free()


def searches(ctx, fit):
    """fit()'s result and whether rows were searched, and lists, in it."""
    ctx.reset_stats()
    ctx.set_profiling(True)
    try:
        out = fit()
    finally:
        ctx.set_profiling(False)
    st = ctx.kernel_stats()
    return out, "k_scan_hist" in st, "k_select" in st and "k_scan_hist" not in st


def test_rows_where_the_list_tables_do_not_fit():
    """60,000 x 1,000, one tree's rows 240 MB, the tables 480 MB and their
    scratch 240 MB: with 600 MB free the fit's own choice is lists, and the
    trees come from rows.  Then the other way round: tables of an earlier fit
    make way for rows that need their memory."""
    N, F, K, T, m = 60000, 1000, 5, 5, 10
    X, y = gauss(N, F, K, 2)
    ctx = _lib.Context(0)
    ds = _lib.Dataset(ctx, X, y, K)
    assert ds.idx_bits == 16

    def fit(**kw):
        return _lib.Forest.fit(ctx, ds, T, opts(m, **kw), None).export()

    want = fit(search=_lib.CTA_SEARCH_ROWS)
    ctx.release_workspace()
    print("tables that do not fit", flush=True)
    free0 = ctx.mem_info()[0]
    hog = Hog(ctx, 600 << 20)
    try:
        got, rows, lists = searches(ctx, fit)
    finally:
        hog.free()
    assert rows and helpers.forest_diff(got, want) is None
    ctx.release_workspace()
    assert ctx.mem_info()[0] >= free0 - (32 << 20)  # nothing of the tables stayed
    got, rows, lists = searches(ctx, fit)
    assert lists and not rows and helpers.forest_diff(got, want) is None
    ctx.release_workspace()
    print("tables that make way", flush=True)
    hog = Hog(ctx, 200 << 20)
    try:
        got, rows, lists = searches(ctx, lambda: fit(search=_lib.CTA_SEARCH_ROWS))
    finally:
        hog.free()
    assert rows and helpers.forest_diff(got, want) is None
    ds.close()
    ctx.close()


def test_rows_where_the_list_tasks_do_not_fit_their_indices():
    """1,100 x 65,535 with every feature evaluated at 1,024 classes: the class
    counts of the list search's workgroup tasks pass 32 bits, those of the rows
    (one chunk a node) do not."""
    N, F, K = 1100, 65535, 1024
    rng = np.random.Generator(np.random.PCG64(3))
    y = rng.permutation(np.arange(N) % K)
    X = rng.integers(0, 3, size=(N, F)).astype(np.float32)
    ctx = _lib.Context(0)
    ds = _lib.Dataset(ctx, X, y, K)
    print("task indices", flush=True)
    trees = [_lib.Forest.fit(ctx, ds, 1, opts(F, search=s, bootstrap=0, max_depth=1, scan_chunk=1 << 20), None).export()
             for s in (_lib.CTA_SEARCH_ROWS, _lib.CTA_SEARCH_LISTS)]
    assert len(trees[0]["feature"]) == 3 and helpers.forest_diff(*trees) is None
    ds.close()
    ctx.close()


def limited(ctx, spare=None):
    """Sets the context's workspace limit to what it holds and `spare` bytes."""
    held = ctypes.c_uint64()
    _lib.check(ctx.lib.cta_ctx_workspace_bytes(ctx.h, ctypes.byref(held)))
    _lib.check(ctx.lib.cta_ctx_set_workspace_limit(ctx.h, held.value + spare if spare is not None else 0))
    return held.value


def test_limited_context_builds_tables_in_the_scratch_it_holds():
    """3,000 x 2,000: the scratch of the tables (24 MB) is what the dataset's
    build left, so lists need next to nothing more; and after a release a limit
    that one tree's rows fit holds the tables' scratch as well."""
    N, F, K, T, m = 3000, 2000, 5, 3, 45
    X, y = gauss(N, F, K, 4)
    ctx = _lib.Context(0)
    ds = _lib.Dataset(ctx, X, y, K)

    def fit(**kw):
        return _lib.Forest.fit(ctx, ds, T, opts(m, **kw), None).export()

    want = fit(search=_lib.CTA_SEARCH_ROWS)
    print("limited context", flush=True)
    limited(ctx, 1 << 20)
    got, rows, lists = searches(ctx, fit)
    assert lists and not rows and helpers.forest_diff(got, want) is None
    ds.close()
    limited(ctx)
    ds = _lib.Dataset(ctx, X, y, K)
    ctx.release_workspace()
    limited(ctx, 28 << 20)
    got, rows, lists = searches(ctx, fit)
    assert lists and not rows and helpers.forest_diff(got, want) is None
    assert limited(ctx) <= 20 << 20  # the scratch was given back
    ds.close()
    ctx.close()


def test_limited_context_without_room_for_list_tasks():
    """A limit at what a row fit holds: the list search's own workspaces do not
    fit it, and the rows do, as they did."""
    N, F, K, T, m = 3000, 2000, 5, 3, 45
    X, y = gauss(N, F, K, 6)
    ctx = _lib.Context(0)
    ds = _lib.Dataset(ctx, X, y, K)

    def fit(**kw):
        return _lib.Forest.fit(ctx, ds, T, opts(m, **kw), None).export()

    want = fit(search=_lib.CTA_SEARCH_ROWS)
    print("limit at what rows hold", flush=True)
    held = limited(ctx, 0)
    got, rows, _ = searches(ctx, fit)
    assert rows and helpers.forest_diff(got, want) is None
    assert limited(ctx) <= held
    ds.close()
    ctx.close()


def test_tables_make_way_for_another_training_set():
    """The tables of a fit on 60,000 x 1,000 (480 MB) stay with that training set;
    with 450 MB free, another one of 20,000 x 1,000 (700 MB while it is built) and
    its fit take their memory, and a later fit builds them again."""
    N, F, K, T, m = 60000, 1000, 5, 5, 10
    X, y = gauss(N, F, K, 7)
    ctx = _lib.Context(0)
    a = _lib.Dataset(ctx, X, y, K)

    def fit(ds):
        return _lib.Forest.fit(ctx, ds, T, opts(m), None).export()

    want, rows, lists = searches(ctx, lambda: fit(a))
    assert lists and not rows
    n = 20000
    b = _lib.Dataset(ctx, X[:n], y[:n], K)
    want_b = fit(b)
    b.close()
    fit(a)
    ctx.release_workspace()
    print("another training set", flush=True)
    hog = Hog(ctx, 450 << 20)
    try:
        b = _lib.Dataset(ctx, X[:n], y[:n], K)
        ctx.release_workspace()
        got_b = fit(b)
    finally:
        hog.free()
    assert helpers.forest_diff(got_b, want_b) is None
    got, rows, lists = searches(ctx, lambda: fit(a))
    assert lists and not rows and helpers.forest_diff(got, want) is None
    b.close()
    a.close()
    ctx.close()
