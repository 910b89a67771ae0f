"""Quantile binning on the device (pb_quantile_edges, pb_apply_bins) against the reference's
NumPy binning (data.py:44-111: np.quantile(method="linear") edges cast to float32,
searchsorted(side="left") clipped): bins bit-identical and edges bit-identical except for
the sign of a zero edge (-0.0 and +0.0 tie in a sort, so which one a quantile picks is the
sorting routine's choice; searchsorted treats them alike), including ties, a constant
column, a column holding NaN, NaN values against finite edges, a single row, and the row
gather the fit uses (era-major order); and against the reference's own bins and edges in the
golden fits."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def assert_edges_equal(got, want, msg=""):
    """Bitwise, except that -0.0 and +0.0 compare equal."""
    g = np.where(got == 0, np.float32(0), got)
    w = np.where(want == 0, np.float32(0), want)
    np.testing.assert_array_equal(g.view(np.uint32), w.view(np.uint32), err_msg=msg)


def _host_bins(X, nb):
    from packboost_amd.data import quantile_bin

    return quantile_bin(X, nb)


def _dev(X, nb, perm=None):
    import torch

    from packboost_amd.data import quantile_bin_device

    bins_fm, edges = quantile_bin_device(X, nb, torch.device("cuda"), perm=perm, chunk_features=3)
    n = X.shape[0]
    return bins_fm[:, :n].cpu().numpy().T, edges


def _data(seed, n, f):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, f)).astype(np.float32)
    X[:, 1] = np.round(X[:, 1] * 2) / 2          # heavy ties
    X[:, 2] = 3.5                                 # constant
    if f > 4:
        X[rng.integers(0, n, 5), 4] = np.nan      # NaN column -> NaN edges
    X[rng.integers(0, n, 7), 0] = np.nan if f <= 4 else X[0, 0]
    return X


@pytest.mark.parametrize("nb", [2, 5, 63, 128, 255])
def test_device_binning_matches_numpy(hip, nb):
    X = _data(nb, 3001, 7)
    print(f"[binning] nb={nb}", flush=True)
    hb, he = _host_bins(X, nb)
    db, de = _dev(X, nb)
    assert_edges_equal(de, he)
    np.testing.assert_array_equal(db, hb)
    perm = np.random.default_rng(1).permutation(X.shape[0])
    pb, _ = _dev(X, nb, perm=perm)
    np.testing.assert_array_equal(pb, hb[perm])


def test_device_binning_small_and_nan_values(hip):
    import torch

    from packboost_amd.data import apply_bins, apply_bins_device

    X1 = np.array([[1.5, -2.0, 0.0]], np.float32)
    hb, he = _host_bins(X1, 8)
    db, de = _dev(X1, 8)
    assert_edges_equal(de, he)
    np.testing.assert_array_equal(db, hb)
    X = _data(9, 2000, 4)  # NaN values in column 0, finite edges elsewhere
    hb, he = _host_bins(X, 16)
    db, de = _dev(X, 16)
    assert_edges_equal(de, he)
    np.testing.assert_array_equal(db, hb)
    Xn = np.random.default_rng(5).standard_normal((999, 4)).astype(np.float32) * 3
    Xn[::37, 1] = np.nan
    got = apply_bins_device(Xn, he, 16, torch.device("cuda"))[:, :999].cpu().numpy().T
    np.testing.assert_array_equal(got, apply_bins(Xn, he, 16))


def test_device_binning_matches_reference_golden(hip):
    from tests.test_fit_golden import CASES, load_case

    for name in CASES:
        d = load_case(name)
        nb = d["config"]["max_bins"]
        db, de = _dev(d["X"], nb)
        np.testing.assert_array_equal(db, d["bins"], err_msg=name)
        want = d["edges"].reshape(len(d["edge_lens"]), -1).astype(np.float32)  # [max_bins - 1, F]
        assert_edges_equal(de, want, name)


@pytest.mark.parametrize("n,f,nb", [(1, 1, 2), (127, 31, 3), (128, 32, 4), (129, 33, 17), (1000, 70, 129),
                                    (5001, 5, 255), (300_000, 40, 64), (399_999, 1, 5), (400_001, 1, 5),
                                    (800_003, 2, 64), (300_001, 7, 128), (300_001, 7, 129), (300_001, 8, 255)])
def test_bin_rows_shapes(hip, n, f, nb):
    """Tile, feature-group and search-depth edges, few features on either side of the counts that go
    through a feature-major copy, strided and feature-major inputs, with and without a row gather:
    bins equal NumPy's searchsorted (values on the edges, signed zeros, infinities and NaN included),
    padding rows 0."""
    import torch

    from packboost_amd.data import apply_bins_device

    rng = np.random.default_rng(n + f)
    edges = np.sort(np.round(rng.standard_normal((nb - 1, f)), 2).astype(np.float32), axis=0)
    edges[edges == 0] = -0.0
    X = np.round(rng.standard_normal((n, f)), 2).astype(np.float32) * 2
    X[rng.random((n, f)) < 0.05] = np.nan
    X[rng.random((n, f)) < 0.05] = np.inf
    X[rng.random((n, f)) < 0.05] = -np.inf
    X[rng.random((n, f)) < 0.05] = 0.0
    want = np.empty((n, f), np.uint8)
    for j in range(f):
        want[:, j] = np.minimum(np.searchsorted(edges[:, j], X[:, j], side="left"), nb - 1)
    perm = rng.permutation(n)
    wide = torch.zeros((n, f + 3), device="cuda")
    wide[:, 2:2 + f] = torch.from_numpy(X).cuda()
    inputs = (X, np.asfortranarray(X), wide[:, 2:2 + f], torch.from_numpy(X).cuda().t().contiguous().t())
    for x in inputs:
        for p in (None, perm):
            got = apply_bins_device(x, edges, nb, torch.device("cuda"), perm=p, chunk_features=9)
            assert got.shape == (f, (n + 15) // 16 * 16) and not bool(got[:, n:].any())
            np.testing.assert_array_equal(got[:, :n].cpu().numpy().T, want if p is None else want[p])


@pytest.mark.parametrize("n,nb", [(1, 5), (2, 255), (3, 2), (16384, 128), (16385, 255), (16385, 2), (40_003, 63),
                                  (530_001, 255)])
def test_column_quantiles(hip, n, nb):
    """The selection's edges equal NumPy's at its size limits (columns sorted in LDS up to 16384
    rows, 255 splitters up to 2^19 rows, 1023 above) on columns that strain it: sorted and reversed
    input, few distinct values, one heavy value, a constant, long-tailed and negative values,
    infinities, signed zeros, a NaN, and one value next to a crowd of equal ones. Where infinities
    leave NaN edges below finite ones, searchsorted has no answer of its own: there the row-major
    and the feature-major binning must agree."""
    import torch

    from packboost_amd.data import quantile_bin_device

    rng = np.random.default_rng(n + nb)
    z = rng.standard_normal(n).astype(np.float32)
    cols = [z, np.sort(z), np.sort(z)[::-1], np.round(z), np.where(rng.random(n) < 0.9, np.float32(0.25), z),
            np.full(n, -7.5), np.exp(6 * z), -np.exp(-8 * z), np.where(rng.random(n) < 0.01, np.inf, z),
            np.where(rng.random(n) < 0.4, -np.inf, z), np.where(rng.random(n) < 0.5, -0.0, 0.0),
            np.where(np.arange(n) == n // 2, np.nan, z), np.where(np.arange(n) == n - 1, 1.0, 2.0), z * 1e-41]
    X = np.stack([c.astype(np.float32) for c in cols], axis=1)
    with np.errstate(invalid="ignore"):
        want_b, want_e = _host_bins(X, nb)
        ascends = np.array([np.array_equal(np.sort(e), e, equal_nan=True) for e in want_e.T])
        got = []
        for x in (X, torch.from_numpy(np.asfortranarray(X)).cuda()):
            bins_fm, edges = quantile_bin_device(x, nb, torch.device("cuda"), chunk_features=9)
            one_nan = [np.where(np.isnan(e), np.float32(np.nan), e) for e in (edges, want_e)]  # inf - inf: any sign
            assert_edges_equal(*one_nan, f"n={n} nb={nb}")
            got.append(bins_fm[:, :n].cpu().numpy().T)
            np.testing.assert_array_equal(got[-1][:, ascends], want_b[:, ascends])
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("n", [2, 1003, 16384, 16386, 30_002, 530_002])
def test_zero_edges_keep_their_sign(hip, n):
    """Columns whose zeros all have one sign (a rectified column and its negative, and zeros alone):
    edges equal NumPy's bit for bit, signs of zeros included, sorted in LDS and selected."""
    import torch

    from packboost_amd.data import quantile_bin_device

    z = np.maximum(np.random.default_rng(n).standard_normal(n), 0).astype(np.float32)
    X = np.stack([z, -z, np.zeros_like(z), np.full_like(z, -0.0)], axis=1)
    want = _host_bins(X, 8)[1]
    assert np.signbit(want[want == 0]).any()
    for x in (X, np.asfortranarray(X)):
        edges = quantile_bin_device(x, 8, torch.device("cuda"))[1]
        np.testing.assert_array_equal(edges.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,f", [(50, 1), (50, 7), (1, 3)])
def test_overlapping_columns(hip, n, f):
    """One column seen as several, and windows over one series: their columns overlap in memory."""
    import torch

    from packboost_amd.data import apply_bins_device, quantile_bin_device

    dev = torch.device("cuda")
    series = torch.randn(n + f, generator=torch.Generator().manual_seed(n)).to(dev)
    for x in (series[:n, None].expand(n, f), series.as_strided((n, f), (1, 1)), series[None, :f].expand(n, f)):
        X = x.cpu().numpy().copy()
        want_b, want_e = _host_bins(X, 6)
        got, edges = quantile_bin_device(x, 6, dev)
        assert_edges_equal(edges, want_e, f"strides {x.stride()}")
        np.testing.assert_array_equal(got[:, :n].cpu().numpy().T, want_b)
        again = apply_bins_device(x, want_e, 6, dev)
        np.testing.assert_array_equal(again[:, :n].cpu().numpy().T, want_b)
