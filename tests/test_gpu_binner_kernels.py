"""The binner's kernels at the edges of their tiles and groups, against torch
and the oracle's numpy binner."""

import numpy as np
import pytest
import torch

from yabt_amd import Binner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F,longest", [
    (1, 1, 255), (15, 60, 1), (255, 61, 255), (256, 4, 128), (257, 60, 127), (1000, 121, 255), (300, 500, 30),
    (70001, 2, 254), (600, 17, 0),
])
def test_transform_equals_searchsorted(n, F, longest):
    rng = np.random.default_rng(n + F)
    dev = torch.device("cuda", 0)
    X = rng.normal(size=(n, F)).astype(np.float32)
    X[rng.random((n, F)) < 0.1] = np.nan
    X[rng.random((n, F)) < 0.05] = np.inf
    X[rng.random((n, F)) < 0.05] = -np.inf
    b = Binner(256)
    b.edges_, b.medians_ = [], rng.normal(size=F).astype(np.float32)
    for f in range(F):     # 0 .. longest edges a feature, infinities among them, and values that equal an edge
        k = longest if f == 0 else int(rng.integers(0, longest + 1))
        e = np.sort(rng.choice(np.concatenate([rng.normal(size=600), X[np.isfinite(X)][:50]]), k)).astype(np.float32)
        if k > 3 and f % 2:
            e[0], e[-1] = -np.inf, np.inf
        b.edges_.append(torch.from_numpy(np.unique(e)))
    Xi = np.where(np.isnan(X), b.medians_, X).astype(np.float32)
    want = np.stack([np.searchsorted(b.edges_[f].numpy(), Xi[:, f]) for f in range(F)], axis=1).astype(np.uint8)
    Xd = torch.from_numpy(X).to(dev)
    assert np.array_equal(b.transform(Xd).cpu().numpy(), want)            # rows of F bytes, not aligned
    lay, imp = b.layouts(Xd)
    assert np.array_equal(lay.fm[:, :n].cpu().numpy(), want.T)
    assert np.array_equal(lay.rm[:n, :F].cpu().numpy(), want)
    assert int(lay.fm[:, n:].sum()) == 0 and int(lay.rm[:, F:].sum()) == 0
    assert np.array_equal(imp.cpu().numpy().view(np.uint32), Xi.view(np.uint32))
    wide = torch.zeros((n, F + 3), device=dev)                             # a column stride of 1, a longer row
    wide[:, :F] = Xd
    assert np.array_equal(b.transform(wide[:, :F]).cpu().numpy(), want)
