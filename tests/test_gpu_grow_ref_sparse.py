"""The sparse reference builder where its sorts take four features a block, and
the sums that one pass over a tile decides, against the fp32 oracle (cgrow's
arithmetic), bit for bit."""

import numpy as np
import pytest
import torch

from oracle import boost_oracle as BO
from oracle import oracle as O
from tests.helpers import skewed_bins, tree_arrays_equal
from yabt_amd import _lib
from yabt_amd import grow_hip as G

pytestmark = pytest.mark.gpu

KEYS = ("feature", "thr_bin", "left", "right", "value", "depth")


def _gradients(rng, n, kind):
    g, h = rng.normal(size=n), rng.uniform(0.1, 1.0, size=n)
    if kind == "binades":        # sums that wander over powers of two; addends whose low bits fall below them
        g = g * 2.0 ** rng.integers(-30, 3, size=n)
    elif kind == "integers":     # no step rounds
        g, h = np.rint(4 * g), np.ones(n)
    elif kind == "zeros":        # whole tiles of zeros, and -0.0
        g = np.where(np.arange(n) % 9000 < 4500, -0.0, g)
        h = np.where(np.arange(n) % 9000 < 4500, 0.0, h)
    elif kind == "tiny":         # denormals beside ordinary values
        g = np.where(rng.random(n) < 0.3, 1e-40, g)
    return g.astype(np.float32), h.astype(np.float32)


@pytest.mark.parametrize("n,F,share,kind", [
    (210_001, 403, 0.9, "normal"),      # quads: 101 of them, the last of three features, 26 tiles and more
    (220_000, 330, 0.995, "binades"),   # quads; tiles of about twenty listed rows
    (4097, 9, 0.9, "integers"),
    (40_000, 6, 0.5, "zeros"),          # half of each tile listed
    (30_000, 5, 0.02, "tiny"),          # nearly every row listed
    (20_000, 7, 1.0, "normal"),         # no row listed
])
def test_sparse_equals_fp32_oracle(n, F, share, kind):
    rng = np.random.default_rng(n + F)
    bins = skewed_bins(rng, n, F, share)
    bins[:, 0] = rng.integers(0, 256, size=n)    # one column to split on in any case
    g, h = _gradients(rng, n, kind)
    layout = BO.sparse_layout(bins)
    nbins = np.full(F, 256, np.int32)
    kw = dict(max_leaves=24, msl=20)
    dev = torch.device("cuda", 0)
    lay = G.make_layouts(torch.from_numpy(bins), dev)
    gd, hd = torch.from_numpy(g).to(dev), torch.from_numpy(h).to(dev)
    res = G.grow_device(lay, gd, hd, nbins, arithmetic="reference", default_bin=layout[3], **kw)
    got = {k: getattr(res, k).cpu().numpy() for k in KEYS}
    want = O.grow(np.ascontiguousarray(bins.T), g, h, mode=O.MODE_FP32, nbins=nbins, sparse=layout, **kw)
    assert tree_arrays_equal(got, want) is None
    assert np.array_equal(res.rows.cpu().numpy(), want["rows"])
    if F > 300:      # groups of features that start inside a quad
        lib = _lib.load()
        lo, full = (int(f(n, F, 24, 1)) for f in (lib.yabt_grow_ref_workspace_min_bytes, lib.yabt_grow_ref_workspace_bytes))
        part = G._grow_device_ref(lay, gd, hd, nbins, workspace_bytes=lo + (full - lo) * 7 // 8, lam=1.0, gamma=0.0,
                                  mcw=1e-3, lr=0.1, max_depth=64, fmask=None, imat=None, ib=0.5, default_bin=layout[3], **kw)
        assert tree_arrays_equal({k: getattr(part, k).cpu().numpy() for k in KEYS}, want) is None
