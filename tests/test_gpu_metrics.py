"""Round metrics on the device (pb_era_corr) against the reference's era correlation
(PackBoost._era_correlation_np, booster.py:909-929), computed here in float64 NumPy.

Bars: per-era and mean correlations within 1e-9 (both sides in double) on data with empty,
single-row and constant eras; the fit's train metric within 1e-5 of the NumPy metric of
predict() (the fit's running predictions and predict() sum trees in different orders); the
eval metric within 1e-9 of the NumPy metric of the oracle's tree-order float32 sum, the order
in which the eval predictions accumulate."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def era_corr_np(era, y, p):
    """The reference's metric (booster.py:909-929) in float64."""
    cors = []
    for e in np.unique(era):
        m = era == e
        yy, pp = y[m].astype(np.float64), p[m].astype(np.float64)
        if yy.size < 2:
            continue
        sy, sp = yy.std(), pp.std()
        if sy <= 1e-12 or sp <= 1e-12:
            continue
        c = float(((yy - yy.mean()) * (pp - pp.mean())).mean()) / (sy * sp)
        if np.isfinite(c):
            cors.append(c)
    return float(np.mean(cors)) if cors else float("nan")


def test_era_corr_kernel(hip):
    import torch

    rng = np.random.default_rng(0)
    sizes = [500, 0, 1, 300, 40, 1000, 2, 700]
    E = len(sizes)
    era = np.repeat(np.arange(E), sizes)
    N = era.size
    y = rng.standard_normal(N).astype(np.float32)
    p = (0.3 * y + rng.standard_normal(N)).astype(np.float32)
    y[era == 4] = 1.25  # constant target: skipped
    offs = np.zeros(E + 1, np.int32)
    offs[1:] = np.cumsum(sizes)
    dev = torch.device("cuda")
    yd, pd_ = torch.from_numpy(y).to(dev), torch.from_numpy(p).to(dev)
    od = torch.from_numpy(offs).to(dev)
    scratch = torch.empty(E + 1, dtype=torch.float64, device=dev)
    lib = hip.load()
    hip.check(lib.pb_era_corr(yd.data_ptr(), pd_.data_ptr(), od.data_ptr(), E, scratch.data_ptr(),
                              scratch.data_ptr() + 8 * E, hip.stream_ptr()), "pb_era_corr")
    got = scratch.cpu().numpy()
    for e in range(E):
        want = era_corr_np(np.zeros(sizes[e]), y[era == e], p[era == e])
        if np.isnan(want):
            assert np.isnan(got[e]), e
        else:
            assert abs(got[e] - want) <= 1e-9, (e, got[e], want)
    assert abs(got[E] - era_corr_np(era, y, p)) <= 1e-9
    # no era counts -> NaN
    hip.check(lib.pb_era_corr(yd.data_ptr(), yd.data_ptr(), od[2:4].data_ptr(), 1, scratch.data_ptr(),
                              scratch.data_ptr() + 8, hip.stream_ptr()), "pb_era_corr")
    assert np.isnan(scratch[1].item())


def test_fit_round_metrics(hip):
    from packboost_amd import PackBoost, PackBoostConfig
    from tests.test_fit_golden import load_case

    d = load_case("fit_dir_alpha")  # interleaved era labels
    rng = np.random.default_rng(1)
    X2 = rng.standard_normal((900, d["X"].shape[1])).astype(np.float32)
    y2 = (X2[:, 0] + 0.1 * rng.standard_normal(900)).astype(np.float32)
    era2 = rng.integers(0, 7, size=900) * 5
    print("[round metrics]", flush=True)
    model = PackBoost(PackBoostConfig(**d["config"])).fit(
        d["X"], d["y"], d["era"], num_rounds=d["rounds"], eval_sets=[("valid", X2, y2, era2)])
    m = model.round_metrics[-1]
    assert m["round"] == d["rounds"]
    assert abs(m["train_corr"] - era_corr_np(d["era"], d["y"], model.predict(d["X"]))) <= 1e-5
    # the eval predictions accumulate float32(w * leaf) tree by tree, the reference's eval and
    # CPU predict order (booster.py:604-655, 709-712): the metric is exact on that sum
    from oracle import oracle as om
    from packboost_amd.data import apply_bins

    bins2 = apply_bins(X2, model._binner.bin_edges, model.config.max_bins)
    p_eval = om.predict(model._rounds, model.config.pack_size, model._tree_weight, bins2)
    assert abs(m["valid_corr"] - era_corr_np(era2, y2, p_eval)) <= 1e-9
    # PackBoost.predict (the compiled forest's double sums, rounded once) within 1e-5 of it
    np.testing.assert_allclose(model.predict(X2), p_eval, rtol=0, atol=1e-5)
    assert all(np.isfinite(r["train_corr"]) for r in model.round_metrics)


@pytest.mark.parametrize("sizes", [
    [1], [4096], [4097], [20_000], [4095, 1, 0, 4096, 0, 50_000], [0, 0, 70_000, 2, 0, 1, 12_289, 0],
    [400_000] + [3] * 40 + [50_000], [9000] * 70], ids=str)
def test_era_corr_rows(hip, sizes):
    """pb_era_corr_rows (long eras over many workgroups: window edges, windows of several eras,
    empty, single-row and constant eras) against float64 NumPy and pb_era_corr, within 1e-9."""
    import torch

    from packboost_amd.booster import _corr_scratch, _era_corr_enqueue

    E, N = len(sizes), int(sum(sizes))
    rng = np.random.default_rng(N)
    era = np.repeat(np.arange(E), sizes)
    y = (3 + rng.standard_normal(N)).astype(np.float32)
    p = (0.3 * y + rng.standard_normal(N) - 7).astype(np.float32)
    if E > 4:
        p[era == 3] = -1.5  # constant: skipped
    dev = torch.device("cuda")
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)).to(dev)
    yd, pd_ = torch.from_numpy(y).to(dev), torch.from_numpy(p).to(dev)
    scratch = _corr_scratch(N, E, dev)
    out, old = torch.empty(1, dtype=torch.float64, device=dev), torch.empty(E + 1, dtype=torch.float64, device=dev)
    _era_corr_enqueue(yd, pd_, off, scratch, out)
    hip.check(hip.load().pb_era_corr(yd.data_ptr(), pd_.data_ptr(), off.data_ptr(), E, old.data_ptr(),
                                     old.data_ptr() + 8 * E, hip.stream_ptr()), "pb_era_corr")
    got, was = scratch[:E].cpu().numpy(), old.cpu().numpy()
    for e in range(E):
        want = era_corr_np(np.zeros(sizes[e]), y[era == e], p[era == e])
        np.testing.assert_allclose([got[e], was[e]], [want, want], rtol=0, atol=1e-9)
    np.testing.assert_allclose([out.item(), was[E]], [era_corr_np(era, y, p)] * 2, rtol=0, atol=1e-9)


@pytest.mark.parametrize("n", [2**31 - 1, 2**31 - 4095, 2**31 - 4096])
def test_era_corr_rows_to_the_last_row(hip, n):
    """The longest tables the era correlations take: one era whose last rows alone vary, so its
    correlation comes from the last windows of rows, and an era of those rows (row numbers up to
    2^31 - 1, which a step of 256 rows passes)."""
    import torch

    from packboost_amd.booster import _corr_scratch, _era_corr_enqueue

    dev = torch.device("cuda")
    if torch.cuda.mem_get_info(dev)[0] < 24 << 30:
        pytest.skip("needs 24 GiB of device memory")
    tail = 3000
    rng = np.random.default_rng(5)
    yt = rng.standard_normal(tail).astype(np.float32)
    pt = (yt + rng.standard_normal(tail)).astype(np.float32)
    y, p = torch.zeros(n, device=dev), torch.zeros(n, device=dev)
    y[n - tail:], p[n - tail:] = torch.from_numpy(yt), torch.from_numpy(pt)
    off = torch.tensor([0, n], dtype=torch.int32, device=dev)
    scratch = _corr_scratch(n, 1, dev).zero_()
    out = torch.empty(1, dtype=torch.float64, device=dev)
    _era_corr_enqueue(y, p, off, scratch, out)
    # the tail as an era of its own, by pb_era_corr's workgroup per era
    ends, each = torch.tensor([n - tail, n], dtype=torch.int32, device=dev), torch.empty(2, dtype=torch.float64, device=dev)
    hip.check(hip.load().pb_era_corr(y.data_ptr(), p.data_ptr(), ends.data_ptr(), 1, each.data_ptr(),
                                     each.data_ptr() + 8, hip.stream_ptr()), "pb_era_corr")
    np.testing.assert_allclose(each.cpu().numpy(), [era_corr_np(np.zeros(tail), yt, pt)] * 2, rtol=0, atol=1e-9)
    yd, pd_ = yt.astype(np.float64), pt.astype(np.float64)
    my, mp = yd.sum() / n, pd_.sum() / n  # of all rows; those before the tail are zero
    syy, spp, syp = ((a * b).sum() - n * ma * mb for a, b, ma, mb in
                     ((yd, yd, my, my), (pd_, pd_, mp, mp), (yd, pd_, my, mp)))
    np.testing.assert_allclose(out.item(), syp / np.sqrt(syy * spp), rtol=0, atol=1e-9)


@pytest.mark.parametrize("depth,B", [(0, 3), (1, 1), (6, 8), (9, 2), (10, 5)])
def test_fold_tree(hip, depth, B):
    """pb_fold_tree (records in LDS up to 1024 nodes, in memory above) against pb_predict_bins and
    B separate float32 adds: the same roundings, so equal bit for bit."""
    import torch

    from packboost_amd.booster import _to_column_major, _tree_records
    from tests.test_gpu_forest import _forest

    dev = torch.device("cuda")
    N, F = 3001, 40
    a = _forest(depth, 2, 1, depth, F, ragged=True, max_thr=30)[1]
    bins = _to_column_major(torch.randint(0, 32, (N, F), dtype=torch.uint8, device=dev), dev)
    lib, v = hip.load(), torch.empty(N, device=dev)
    t = {k: torch.from_numpy(np.ascontiguousarray(a[k]).astype(d)).to(dev) for k, d in (
        ("feature", np.int32), ("threshold", np.int32), ("left", np.int32), ("right", np.int32),
        ("value", np.float32), ("is_leaf", np.uint8))}
    hip.check(lib.pb_predict_bins(bins.data_ptr(), N, bins.shape[1], F, *(t[k].data_ptr() for k in t),
                                  len(a["value"]), v.data_ptr(), hip.stream_ptr()), "pb_predict_bins")
    want = torch.randn(N, device=dev)
    got = want.clone()
    term = torch.tensor(0.1, device=dev) * v
    for _ in range(B):
        want = want + term
    rec = torch.from_numpy(_tree_records(a)).to(dev)
    hip.check(lib.pb_fold_tree(bins.data_ptr(), N, bins.shape[1], F, rec.data_ptr(), len(a["value"]), B,
                               float(np.float32(0.1)), got.data_ptr(), hip.stream_ptr()), "pb_fold_tree")
    assert torch.equal(got, want)
