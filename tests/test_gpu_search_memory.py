"""Memory and the choice of search (needs an MI355X): the list search's tables
take device memory that sorted rows do not, so a fit that may use either goes
back to rows where they do not fit, and grows the same trees."""
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
