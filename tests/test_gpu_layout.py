"""Row-major bins to the kernels' column-major layout (pb_transpose_bins) against torch's own
transposition: tile edges and remainders, unaligned rows, a row gather, a row chunk of a larger
column stride, zeroed padding rows and the bin limit. Bytes, so every comparison is exact."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F", [(1, 1), (15, 16), (16, 17), (255, 127), (256, 128), (257, 129), (1000, 2376),
                                 (4099, 31), (4099, 32), ((1 << 20) - 5, 9), ((1 << 20) + 5, 6),
                                 ((1 << 20) + 5, 7), ((1 << 20) + 5, 15), ((1 << 20) + 5, 16)])
@pytest.mark.parametrize("gather", [False, True])
def test_transpose_bins(hip, n, F, gather):
    import torch

    from packboost_amd.engine import column_major_bins, padded_rows

    rng = np.random.default_rng(n * 7 + F)
    X = torch.from_numpy(rng.integers(0, 200, size=(n, F + 5), dtype=np.uint8)).cuda()[:, 3:3 + F]  # unaligned rows
    perm = rng.permutation(n) if gather else None
    want = (X if perm is None else X[torch.from_numpy(perm).cuda()]).t()
    for src in (X, X.contiguous(), X.view(torch.int8), X.t().contiguous().t(), X.cpu().numpy()):
        chunk = 512 if n < 10_000 else 1 << 18
        got = column_major_bins(src, perm, torch.device("cuda:0"), chunk_rows=chunk, limit=200)
        assert got.shape == (F, padded_rows(n))
        assert torch.equal(got[:, :n], want) and not bool(got[:, n:].any())
        if int(want.max()):
            with pytest.raises(ValueError, match="max_bins"):
                column_major_bins(src, perm, torch.device("cuda:0"), chunk_rows=chunk, limit=int(want.max()))


@pytest.mark.parametrize("limit", [1, 5, 127, 128, 129, 200, 255])
def test_bin_limit(hip, limit):
    """One code at the limit is refused wherever it sits, in row-major, feature-major and host tables
    (each checked on its own route); all below it pass."""
    import torch

    from packboost_amd.engine import column_major_bins

    dev = torch.device("cuda:0")
    n, F = 300, 150
    ok = torch.randint(0, limit, (n, F), dtype=torch.uint8, device=dev)
    ok[0, 0] = limit - 1
    layouts = (lambda x: x, lambda x: x.t().contiguous().t(), lambda x: x.cpu().numpy(),
               lambda x: np.asfortranarray(x.cpu().numpy()))
    for lay in layouts:
        column_major_bins(lay(ok), None, dev, chunk_rows=128, limit=limit)
    for r, f in ((0, 0), (299, 149), (255, 128), (256, 127), (37, 3)):
        for code in {limit, 255}:
            bad = ok.clone()
            bad[r, f] = code
            for lay in layouts:
                with pytest.raises(ValueError, match="max_bins"):
                    column_major_bins(lay(bad), None, dev, chunk_rows=128, limit=limit)
