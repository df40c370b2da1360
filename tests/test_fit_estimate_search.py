"""cta_fit_estimate and the choice of search (host only): a fit that keeps to
sorted rows is estimated at what sorted rows need, and only a fit that may
search from sample lists is charged their tables."""
import pytest

from cudatree_amd import _lib

# (N, F, K, T, max_features): dataset and workspace bytes of a fit over sorted rows
ROWS = {
    (20000, 54, 7, 10, 7): (13241376, 220337800),
    (581012, 54, 7, 50, 7): (446819604, 25576158564),
    (200000, 256, 20, 200, 16): (724286016, 103863563584),
    (20000, 4096, 5, 100, 64): (994694816, 35849066128),
    (3000, 400, 5, 20, 20): (14703096, 218121164),
    (65535, 100, 255, 8, 10): (80054331, 1437912392),
    (65536, 100, 256, 8, 10): (93228288, 1650794240),
}


def opts(m, **kw):
    o = _lib.default_opts()
    o.max_features = m
    for k, v in kw.items():
        setattr(o, k, v)
    return o


@pytest.mark.parametrize("size", sorted(ROWS))
def test_rows_are_estimated_without_list_tables(size):
    N, F, K, T, m = size
    assert _lib.fit_estimate(N, F, K, T, opts(m, search=_lib.CTA_SEARCH_ROWS)) == ROWS[size]
    # options under which no list is ever built
    for kw in ({"all_rows": 1}, {"subtree_max": 64}):
        assert _lib.fit_estimate(N, F, K, T, opts(m, **kw)) == ROWS[size]
    for mode in (_lib.CTA_MODE_HYBRID, _lib.CTA_MODE_PER_NODE):
        assert _lib.fit_estimate(N, F, K, T, opts(m, mode=mode))[0] == ROWS[size][0]


@pytest.mark.parametrize("size,lists", [((20000, 54, 7, 10, 7), False),         # too few trees and features
                                        ((65535, 100, 255, 8, 10), False),
                                        ((200000, 256, 20, 200, 16), True),     # enough of both
                                        ((20000, 4096, 5, 100, 64), True),
                                        ((3000, 400, 5, 20, 20), True),
                                        ((581012, 54, 7, 50, 7), True)])        # if its features have few values
def test_only_fits_that_may_use_lists_are_charged_their_tables(size, lists):
    N, F, K, T, m = size
    tables = 8 * N * F + N * (2 if N <= 65535 else 4) + 20 * F
    ds, ws = _lib.fit_estimate(N, F, K, T, opts(m))
    assert (ds - ROWS[size][0], ws) == (tables if lists else 0, ROWS[size][1])
    ds, ws = _lib.fit_estimate(N, F, K, T, opts(m, search=_lib.CTA_SEARCH_LISTS))
    assert (ds - ROWS[size][0], ws) == (tables, ROWS[size][1])


@pytest.mark.parametrize("size,trees_per_batch,lists", [((200000, 256, 20, 200, 16), 1, False),
                                                        ((200000, 256, 20, 200, 16), 4, True),
                                                        ((20000, 4096, 5, 100, 64), 1, True)])  # no large nodes
def test_few_trees_at_a_time_leave_large_nodes_to_rows(size, trees_per_batch, lists):
    rows = _lib.fit_estimate(*size[:4], opts(size[4], search=_lib.CTA_SEARCH_ROWS, trees_per_batch=trees_per_batch))
    auto = _lib.fit_estimate(*size[:4], opts(size[4], trees_per_batch=trees_per_batch))
    assert (auto[0] > rows[0]) == lists and auto[1] == rows[1]
