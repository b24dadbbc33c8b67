"""Depth-batched growth where its chunks, places and early ends meet: against
split-by-split growth, bit for bit."""

import numpy as np
import pytest
import torch

from yabt_amd import grow_hip as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F,nb,depth,msl,const_h,outlier", [
    (1, 3, 8, 3, 0, False, False),              # one row
    (17, 1, 2, 4, 1, False, False),             # one split, then nothing left to split
    (4096, 16, 256, 5, 1, True, False),         # whole routing blocks, one tile of features
    (4097, 33, 3, 9, 0, False, False),          # children without rows' worth of splits at the last depths
    (50_000, 17, 40, 12, 2, True, True),        # 4096 places, the wide contract
    (30_000, 5, 256, 13, 1, False, False),      # more places than the LDS counters
    (600_001, 20, 64, 6, 20, False, True),      # several chunks per child
])
def test_depth_batched_equals_sequential(n, F, nb, depth, msl, const_h, outlier):
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(n + F)
    bins = torch.from_numpy(rng.integers(0, nb, size=(n, F)).astype(np.uint8)).to(dev)
    g = rng.normal(size=n).astype(np.float32)
    if outlier:
        g[n // 2] = 1e5
    h = np.full(n, 0.25, np.float32) if const_h else rng.uniform(0.1, 1.0, size=n).astype(np.float32)
    lay = G.make_layouts(bins, dev)
    gd, hd = torch.from_numpy(g).to(dev), torch.from_numpy(h).to(dev)
    kw = dict(max_leaves=2 ** depth, max_depth=depth, msl=msl, mcw=0.0)
    a = G.grow_device(lay, gd, hd, np.full(F, nb, np.int32), growth="levelwise", **kw)
    b = G.grow_device(lay, gd, hd, np.full(F, nb, np.int32), growth="sequential", **kw)
    assert a.n_nodes == b.n_nodes
    for k in ("feature", "thr_bin", "left", "right", "depth"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k
    assert torch.equal(a.value.view(torch.int32), b.value.view(torch.int32))
    assert torch.equal(a.leaf_of_row, b.leaf_of_row)


@pytest.mark.parametrize("n,F,depth,gamma,most", [
    (1000, 5, 15, 1e9, 0),          # the root does not split: 32768 places for one node
    (20_000, 20, 15, 20.0, 0),      # a few splits, the deepest far above the cap
    (3000, 3, 1, 0.0, 0),           # the cap itself ends it
    (50_000, 6, 10, 5.0, 0),
    (300_000, 4, 15, 0.0, 4097),    # more splits of one depth than the LDS counters, the pick's and the scan's blocks
])
def test_work_follows_the_splits_that_exist(n, F, depth, gamma, most):
    """Growth that ends far above its cap, and depths with so many splits that
    the launches go over them in strides: split-by-split growth's tree."""
    dev = torch.device("cuda", 0)
    rng = np.random.default_rng(n + depth)
    bins = torch.from_numpy(rng.integers(0, 256, size=(n, F)).astype(np.uint8)).to(dev)
    signal = bins.float().sum(1) / 64 if most else (bins[:, 0] > 99).float()     # the first: even splits
    g = signal + torch.from_numpy(rng.normal(size=n).astype(np.float32)).to(dev)
    h = torch.ones(n, device=dev)
    lay = G.make_layouts(bins, dev)
    kw = dict(max_leaves=2 ** depth, max_depth=depth, msl=1, mcw=0.0, gamma=gamma, lam=0.0 if most else 1.0)
    a = G.grow_device(lay, g, h, np.full(F, 256, np.int32), growth="levelwise", **kw)
    kw["max_leaves"] = min(kw["max_leaves"], 32767)      # which no tree here reaches
    b = G.grow_device(lay, g, h, np.full(F, 256, np.int32), growth="sequential", **kw)
    assert a.n_nodes == b.n_nodes < 2 * 32767 - 1
    for k in ("feature", "thr_bin", "left", "right", "depth"):
        assert torch.equal(getattr(a, k), getattr(b, k)), k
    assert torch.equal(a.value.view(torch.int32), b.value.view(torch.int32))
    assert torch.equal(a.leaf_of_row, b.leaf_of_row)
    if most:
        splits = torch.bincount(a.depth[a.feature >= 0], minlength=depth)
        assert int(splits[:depth - 1].max()) >= most


def test_depth_batched_reports_non_finite():
    dev = torch.device("cuda", 0)
    lay = G.make_layouts(torch.zeros((100, 2), dtype=torch.uint8, device=dev), dev)
    g = torch.zeros(100, device=dev)
    g[7] = float("inf")
    with pytest.raises(ValueError):
        G.grow_device(lay, g, torch.ones(100, device=dev), np.full(2, 4, np.int32), growth="levelwise", max_leaves=8,
                      max_depth=3)
