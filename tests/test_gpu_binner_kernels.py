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
    (2_100_003, 1, 200), (530_001, 4, 255), (9001, 13, 100), (270_001, 29, 64),   # tiles of 4096 rows down to 16
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


def _column(rng, kind, n):
    if kind == "normal":
        x = rng.normal(size=n)
    elif kind == "counts":           # ties of every size, one of them the median's
        x = np.floor(rng.exponential(3.0, size=n))
    elif kind == "zeros":            # zero IQR: the std fallback
        x = np.where(rng.random(n) < 0.9, 0.0, rng.normal(size=n))
    elif kind == "half":             # the median's two values lie in two far blocks of ties
        x = np.where(np.arange(n) % 2 == 0, -1.0, 3.0)
    elif kind == "narrow":           # keys that differ in their last bits only
        x = 1.0 + rng.integers(0, 50, size=n) * 2.0 ** -23
    else:                            # "constant"
        x = np.full(n, 2.5)
    return x.astype(np.float32)


KINDS = ["normal", "counts", "zeros", "half", "narrow", "constant"]


@pytest.mark.parametrize("n,missing", [(2, 0.0), (4095, 0.0), (4096, 0.3), (4097, 0.0), (8193, 0.01), (65537, 0.5),
                                       (200_001, 0.0), (200_002, 0.2), (900_001, 0.05)])
def test_fit_equals_numpy(n, missing):
    """Sort chunks' edges, the std fallback's buffers (whole, partial, with NaN
    gaps) and the medians' brackets, against the oracle's numpy binner."""
    from oracle import boost_oracle as BO
    rng = np.random.default_rng(n)
    X = np.stack([_column(rng, k, n) for k in KINDS], axis=1)
    X[rng.random(X.shape) < missing] = np.nan
    ref, b = BO.Binner(256).fit(X), Binner(256).fit(X)
    for f in range(X.shape[1]):
        want = ref.edges_[f].astype(np.float32)
        assert np.array_equal(b.edges_[f].numpy().view(np.uint32), want.view(np.uint32)), KINDS[f]
    assert np.array_equal(b.scales_.numpy().view(np.uint32), ref.scales_.view(np.uint32))
    assert np.array_equal(b.medians_.view(np.uint32), np.nanmedian(X, axis=0).astype(np.float32).view(np.uint32))


def _medians(X, rows):
    """yabt_bin_fit's medians of X from a caller's own sample."""
    import ctypes
    from yabt_amd import _lib
    (n, F), m = X.shape, len(rows)
    dev = torch.device("cuda", 0)
    Xd, rows = torch.from_numpy(X).to(dev), torch.from_numpy(rows).to(dev)
    lib = _lib.load()
    nb = int(lib.yabt_bin_fit_workspace_bytes(m, F))
    ws = torch.empty(nb, dtype=torch.uint8, device=dev)
    edges, ne = torch.empty((F, 255), device=dev), torch.empty(F, dtype=torch.int32, device=dev)
    sc, med = torch.empty(F, device=dev), torch.empty(F, device=dev)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    _lib.check(lib.yabt_bin_fit(p(Xd), F, n, F, p(rows), m, 256, p(ws), nb, p(edges), 255, p(ne), p(sc), p(med),
                                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "yabt_bin_fit")
    return med.cpu().numpy()


def test_medians_of_a_sample_that_is_not_random():
    """The C entry takes any rows as the sample: the medians are of all rows."""
    rng = np.random.default_rng(5)
    n, F, m = 30_000, 300, 5000
    X = rng.normal(size=(n, F)).astype(np.float32)
    X = np.sort(X, axis=0)
    X[:, 7] = np.nan
    med = _medians(X, np.arange(m))                                        # the smallest values
    want = np.zeros(F, np.float32)
    keep = np.arange(F) != 7
    want[keep] = np.median(X[:, keep], axis=0)
    assert np.array_equal(med.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,m", [(300_000, 2000), (300_001, 40), (50_000, 1), (40_000, 9000)])
def test_medians_where_few_features_have_a_bracket(n, m):
    """A sample so small that the rows around the median would not fit its
    lists (no bracket), beside columns of ties (a bracket) and one whose sample is
    all NaN (a bracket that misses), over two tiles of the select."""
    rng = np.random.default_rng(n)
    rows = rng.choice(n, m, replace=False)
    X = np.stack([_column(rng, KINDS[f % len(KINDS)], n) for f in range(20)], axis=1)
    X[rows, 17] = np.nan
    X[rng.random(n) < 0.3, 4] = np.nan
    med = _medians(X, rows)
    assert np.array_equal(med.view(np.uint32), np.nanmedian(X, axis=0).astype(np.float32).view(np.uint32))
