"""The reference-arithmetic grower's per-fit root table (yabt_ref_root_order)
against the bucketing of the root in each call (k_walk_sort): identical trees,
rows[] and leaf ids, bit for bit, and both the oracle's (its row-order fp32
chains, oracle/grow_oracle.c; yabt/_cgrow/grow.c:37-62).  Ragged tiles, a single
partial tile, runs of a bin that are longer than the chains' reads ahead (64, and
most of a tile), and features of few bins, whose groups of bins differ between the
two roots: the table knows the largest bin, the call only the declared count.
"""

import numpy as np
import pytest
import torch

from yabt_amd import grow_hip as G

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0) if torch.cuda.is_available() else None


def _bins(kind, n, F, rng):
    if kind == "uniform":
        return rng.integers(0, 256, size=(n, F)).astype(np.uint8)
    if kind == "few":
        # per feature a different span of bins: 28, 2, 1 (all zero: one run of
        # the whole tile, one group), 33 (bins 0..31 and a single row of bin 32
        # in one tile, which the groups must cover), 32, and 20 with 90% of
        # rows in bin 3 (runs of ~3700 per tile)
        spans = [28, 2, 1, 32, 32, 20]
        b = np.stack([rng.integers(0, spans[f % len(spans)], size=n) for f in range(F)], axis=1)
        sk = [f for f in range(F) if f % len(spans) == len(spans) - 1]
        b[:, sk] = np.where(rng.random((n, len(sk))) < 0.9, 3, b[:, sk])
        if F > 3:
            b[n // 2, 3] = 32     # the span-33 feature's largest bin in one row only
        return b.astype(np.uint8)
    # skewed: 90% of rows in bin 7, the rest spread (runs of ~3700 per tile)
    b = rng.integers(0, 256, size=(n, F)).astype(np.uint8)
    b[rng.random((n, F)) < 0.9] = 7
    return b


@pytest.mark.parametrize("kind,n,F,leaves", [
    ("uniform", 50_000, 12, 31),     # 13 tiles, the last one partial
    ("uniform", 100, 5, 8),          # one partial tile
    ("skewed", 30_000, 6, 24),       # runs above and below 64
    ("few", 60_000, 6, 31),          # spans of 1..33 bins: groups of 1 to 5 bins
])
def test_rank_table_root_equals_bucketed_root(kind, n, F, leaves):
    from oracle import oracle as O
    from tests.helpers import tree_arrays_equal
    rng = np.random.default_rng(11)
    bins = _bins(kind, n, F, rng)
    lay = G.make_layouts(torch.from_numpy(bins), DEV)
    gh = rng.normal(size=n).astype(np.float32), rng.uniform(0.05, 1.0, size=n).astype(np.float32)
    g, h = (torch.from_numpy(v).to(DEV) for v in gh)
    nbins = np.full(F, 256, np.int32)
    kw = dict(fmask=None, imat=None, ib=0.0, lam=1.0, gamma=0.0, mcw=1e-3, msl=5, lr=0.1,
              max_leaves=leaves, max_depth=64)
    print(f"reference root: {kind} n={n} F={F}", flush=True)
    a = G._grow_device_ref(lay, g, h, nbins, root_order=True, **kw)
    b = G._grow_device_ref(lay, g, h, nbins, root_order=False, **kw)
    torch.cuda.synchronize()
    assert a.n_nodes == b.n_nodes and a.n_nodes > 1
    for name in ("feature", "thr_bin", "left", "right", "depth"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
    assert torch.equal(a.value.view(torch.int32), b.value.view(torch.int32))
    assert torch.equal(a.rows, b.rows)
    assert torch.equal(a.leaf_of_row, b.leaf_of_row)
    want = O.grow(np.ascontiguousarray(bins.T), *gh, mode=O.MODE_FP32, nbins=nbins, msl=5, max_leaves=leaves)
    got = {k: getattr(a, k).cpu().numpy() for k in ("feature", "thr_bin", "left", "right", "value", "depth")}
    assert tree_arrays_equal(got, want) is None
    assert np.array_equal(a.rows.cpu().numpy(), want["rows"])


@pytest.mark.parametrize("kind,n,F", [("uniform", 70_001, 9), ("skewed", 20_000, 4), ("few", 50_003, 12)])
def test_reference_root_histogram_equals_oracle(kind, n, F):
    """yabt_ref_root_hist bit for bit against the oracle's row-order fp32
    build_hist (oracle/grow_oracle.c, grow.c:37-62)."""
    from oracle import oracle as O
    rng = np.random.default_rng(5)
    bins = _bins(kind, n, F, rng)
    g = rng.normal(size=n).astype(np.float32)
    h = rng.uniform(0.05, 1.0, size=n).astype(np.float32)
    lay = G.make_layouts(torch.from_numpy(bins), DEV)
    print(f"reference root histogram: {kind} n={n} F={F}", flush=True)
    got = G.ref_root_hist(lay, torch.from_numpy(g).to(DEV), torch.from_numpy(h).to(DEV)).cpu().numpy()
    want = O.hist_f32(np.ascontiguousarray(bins.T), g, h)
    assert got.shape == want.shape
    assert np.array_equal(got.view(np.uint32), want.astype(np.float32).view(np.uint32))
