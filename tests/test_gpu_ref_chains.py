"""The dense reference builder's chains (k_tile_chain, k_walk_chain_dense):
the root's histogram bit for bit against the oracle's row-order fp32 sums
(oracle/grow_oracle.c, grow.c:37-62) at the edges of a tile, of its four-row
loads and of the bin groups, and trees through either kernel."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import boost_oracle as BO
from oracle import oracle as O
from tests.helpers import tree_arrays_equal
from yabt_amd import _lib
from yabt_amd import grow_hip as G

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0) if torch.cuda.is_available() else None


def _data(n, F, top, seed=3):
    rng = np.random.default_rng(seed)
    bins = rng.integers(0, top, size=(n, F)).astype(np.uint8)
    bins[rng.random((n, F)) < 0.3] = top - 1          # a long run at the last group's end
    return bins, rng.normal(size=n).astype(np.float32), rng.uniform(0.05, 1.0, size=n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 4095, 4096, 4097, 8193, 12_290])
@pytest.mark.parametrize("F,top", [(3, 256), (3, 9), (300, 40)])   # 8 groups of 32 bins, of 2 (three empty), one group
def test_root_histogram_at_tile_edges(n, F, top):
    bins, g, h = _data(n, F, top)
    lay = G.make_layouts(torch.from_numpy(bins), DEV)
    print(f"root chains: n={n} F={F} top={top}", flush=True)
    got = G.ref_root_hist(lay, torch.from_numpy(g).to(DEV), torch.from_numpy(h).to(DEV)).cpu().numpy()
    want = O.hist_f32(np.ascontiguousarray(bins.T), g, h).astype(np.float32)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,F,top,nb", [
    (9_001, 4, 256, 256),    # one block per bin group for every child
    (9_001, 4, 200, 16),     # rows in bins past the declared count: the last group's
    (5_003, 40, 64, 64),     # few groups, then (40 features x 16 jobs) k_walk_chain_dense
    (4_099, 600, 32, 32),    # k_walk_chain_dense from the root on
    (70_001, 4, 256, 256),   # children of four tiles and more: k_tile_chain in 8 bin groups, later rounds dense
    (70_003, 5, 200, 16),    # the same with rows past the declared count
    (50_003, 70, 64, 64),    # two or three groups, then one block a feature
    (36_001, 260, 40, 40),   # more features than CUs: dense, the root from the table too
])
def test_bucketed_root_and_children(n, F, top, nb):
    """The root bucketed in the call and the root of the per-fit table take
    different kernels or bin counts, and both trees are the oracle's, bit for
    bit."""
    bins, g, h = _data(n, F, top)
    lay = G.make_layouts(torch.from_numpy(bins), DEV)
    kw = dict(fmask=None, imat=None, ib=0.0, lam=1.0, gamma=0.0, mcw=1e-3, msl=5, lr=0.1, max_leaves=63, max_depth=64)
    nbins = np.full(F, nb, np.int32)
    gd, hd = torch.from_numpy(g).to(DEV), torch.from_numpy(h).to(DEV)
    print(f"chains: n={n} F={F} top={top} nbins={nb}", flush=True)
    a, b = (G._grow_device_ref(lay, gd, hd, nbins, root_order=r, **kw) for r in (True, False))
    torch.cuda.synchronize()
    assert a.n_nodes == b.n_nodes and a.n_nodes > 1
    for name in ("feature", "thr_bin", "left", "right", "depth", "rows", "leaf_of_row"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
    assert torch.equal(a.value.view(torch.int32), b.value.view(torch.int32))
    want = O.grow(np.ascontiguousarray(bins.T), g, h, mode=O.MODE_FP32, nbins=nbins, msl=5, max_leaves=63)
    got = {k: getattr(a, k).cpu().numpy() for k in ("feature", "thr_bin", "left", "right", "value", "depth")}
    assert tree_arrays_equal(got, want) is None
    assert np.array_equal(a.rows.cpu().numpy(), want["rows"])


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("n,offset", [(4099, 0), (8192, 1), (5003, 1)])   # the columns' length, or their start, is no multiple of 16
def test_columns_that_no_wide_load_fits(n, offset, sparse):
    """Feature-major columns without padding or alignment, and a root table
    that starts two bytes into its buffer: the oracle's tree."""
    F = 3
    bins, g, h = _data(n, F, 200)
    whole = G.make_layouts(torch.from_numpy(bins), DEV)
    buf = torch.empty(offset + F * n, dtype=torch.uint8, device=DEV)
    fm = buf[offset:].view(F, n)
    fm.copy_(torch.from_numpy(np.ascontiguousarray(bins.T)))
    lay = G.BinLayouts(fm, whole.rm, n, F)
    layout = BO.sparse_layout(bins) if sparse else None
    nbins = np.full(F, 256, np.int32)
    kw = dict(lam=1.0, gamma=0.0, mcw=1e-3, msl=5, lr=0.1, max_leaves=15, max_depth=64)
    want = O.grow(np.ascontiguousarray(bins.T), g, h, mode=O.MODE_FP32, nbins=nbins, sparse=layout, msl=5, max_leaves=15)
    tables = [False] if sparse else [False, True]
    if not sparse:
        lib = _lib.load()
        nb = int(lib.yabt_ref_root_order_bytes(n, F))
        tab = torch.empty(nb + 2, dtype=torch.uint8, device=DEV)
        _lib.check(lib.yabt_ref_root_order(ctypes.c_void_p(fm.data_ptr()), n, n, F, ctypes.c_void_p(tab.data_ptr() + 2), nb,
                                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "yabt_ref_root_order")
        lay._root_order = tab[2:]
    for table in tables:
        print(f"unpadded columns: n={n} offset={offset} sparse={sparse} table={table}", flush=True)
        res = G._grow_device_ref(lay, torch.from_numpy(g).to(DEV), torch.from_numpy(h).to(DEV), nbins, fmask=None, imat=None,
                                 ib=0.0, default_bin=layout[3] if sparse else None, root_order=table, **kw)
        got = {k: getattr(res, k).cpu().numpy() for k in ("feature", "thr_bin", "left", "right", "value", "depth")}
        assert tree_arrays_equal(got, want) is None
        assert np.array_equal(res.rows.cpu().numpy(), want["rows"])
