"""yabt_predict's kernels at the edges of their ranges, against the same fp32
operations in numpy (trees in order, inputs in order), bit for bit."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_forest(rng, T, leaves, F, K, odd=()):
    """Concatenated node arrays of T random trees; ``odd`` names trees whose
    nodes a grower here would not write."""
    feature, thr, left, right, value, off = [], [], [], [], [], [0]
    for t in range(T):
        fe, le, ri = [-1], [-1], [-1]
        open_ = [0]
        L = int(leaves[t % len(leaves)])
        while len(open_) < L:
            n = open_.pop(int(rng.integers(len(open_))))
            fe[n] = int(rng.integers(F))
            le[n], ri[n] = len(fe), len(fe) + 1
            open_ += [len(fe), len(fe) + 1]
            fe += [-1, -1]
            le += [-1, -1]
            ri += [-1, -1]
        if t in odd and L >= 4:
            kind = odd[t]
            if kind == "swapped":                  # right child first
                le[0], ri[0] = ri[0], le[0]
            elif kind == "child":                  # a child outside the tree: rows stay at the parent
                ri[0] = len(fe) + 3
            elif kind == "feature":                # a feature outside X: a leaf to the walk
                fe[le[0]] = F + 2
            elif kind == "cycle":                  # the walk ends after as many steps as nodes
                fe[1], le[1], ri[1] = int(rng.integers(F)), 0, 0
        N = len(fe)
        feature += fe
        left += le
        right += ri
        thr += list(rng.normal(size=N).astype(np.float32))
        value += list(rng.normal(size=N).astype(np.float32))
        off.append(off[-1] + N)
    A = dict(off=np.array(off, np.int64), feature=np.array(feature, np.int64), thr=np.array(thr, np.float32),
             left=np.array(left, np.int64), right=np.array(right, np.int64), value=np.array(value, np.float32))
    if K:
        M = off[-1]
        A["net_k"] = rng.integers(0, K + 1, size=T).astype(np.int32)
        A["net_k"][rng.random(T) < 0.6] = K
        A["net_feats"] = rng.integers(0, F, size=(T, K)).astype(np.int32)
        A["net_feats"][rng.random((T, K)) < 0.05] = F + 1          # reads 0
        A["lin"] = rng.normal(size=(M, K)).astype(np.float32)
        A["lo"] = (rng.normal(size=(M, K)) - 1).astype(np.float32)
        A["hi"] = (A["lo"] + rng.uniform(0, 3, size=(M, K))).astype(np.float32)
        A["lo"][rng.random(M) < 0.1] = np.inf                      # an empty node's envelope
        A["hi"][np.isinf(A["lo"])] = -np.inf
    return A


def numpy_predict(A, X, K, clamp, start):
    n, F = X.shape
    acc = start.copy()
    rows = np.arange(n)
    for t in range(len(A["off"]) - 1):
        o, nt = A["off"][t], A["off"][t + 1] - A["off"][t]
        node = np.zeros(n, np.int64)
        live = np.ones(n, bool)
        for _ in range(nt):
            f = A["feature"][o + node]
            live &= (f >= 0) & (f < F)
            if not live.any():
                break
            x = X[rows, np.clip(f, 0, F - 1)]
            nxt = np.where(x <= A["thr"][o + node], A["left"][o + node], A["right"][o + node])
            live &= (nxt >= 0) & (nxt < nt)
            node = np.where(live, nxt, node)
        g = o + node
        c = A["value"][g]
        if K and A["net_k"][t] > 0:
            net = np.zeros(n, np.float32)
            for j in range(A["net_k"][t]):
                fj = A["net_feats"][t, j]
                x = X[:, fj] if fj < F else np.zeros(n, np.float32)
                if clamp:
                    x = np.fmin(np.fmax(x, A["lo"][g, j]), A["hi"][g, j])
                net = net + A["lin"][g, j] * x
            c = c + net
        acc = acc + c
    return acc


@pytest.mark.parametrize("n,F,T,leaves,K,clamp,odd", [
    (1, 3, 1, [1], 0, True, {}),
    (7, 20, 1030, [2, 5], 8, True, {3: "swapped", 4: "cycle"}),       # a block per row, two rounds of outputs
    (2048, 8, 5, [31], 8, True, {}),
    (2049, 8, 33, [31, 1, 2], 8, True, {1: "child", 5: "feature"}),    # tiles of 64
    (2111, 65, 40, [63], 3, False, {}),                                # features past the ones held ahead
    (32767, 5, 20, [16], 8, True, {7: "cycle"}),
    (32768, 5, 20, [16], 0, True, {2: "swapped", 9: "child"}),         # tiles of 256, one per block
    (70001, 17, 37, [63, 255], 8, True, {11: "feature", 12: "swapped"}),   # two tiles a block, a ragged last one
    (66000, 9, 6, [700, 3], 8, True, {}),                              # trees larger than the LDS
    (4097, 500, 30, [31], 8, True, {2: "child"}),                      # rows too wide for the LDS
    (4097, 200, 1, [31], 8, False, {}),                                # too few trees to stage wide rows
    (4097, 200, 2, [31], 8, False, {}),
    (20_001, 12, 1, [31], 8, True, {}),                                # a row per thread: one tree,
    (140_001, 90, 1, [31], 0, True, {0: "swapped"}),
    (140_001, 16, 3, [31, 2], 0, True, {1: "cycle"}),                  # three on narrow rows,
    (131_073, 300, 5, [31, 1], 0, True, {3: "child", 2: "feature"}),   # a few on wide ones
    (2049, 20, 0, [1], 0, True, {}),                                   # no tree
    (2049, 20, 75, [31, 1, 63], 0, True, {4: "child", 33: "cycle", 64: "swapped"}),   # constant leaves: tiles of 64,
    (32_767, 40, 33, [9, 200], 0, True, {8: "feature"}),               # trees that would not leave places for the groups,
    (4097, 500, 40, [31, 1], 0, True, {5: "cycle"}),                   # rows too wide for the LDS
    (20_003, 60, 20, [300, 2], 0, True, {}),
    (4099, 30, 20, [300, 5], 8, True, {2: "swapped"}),
    (270_001, 110, 18, [63], 8, True, {}),                             # two rounds of blocks, 64 rows a tile
])
def test_predict_equals_numpy(n, F, T, leaves, K, clamp, odd):
    import torch
    from yabt_amd import _lib
    rng = np.random.default_rng(n + 31 * F + T)
    A = random_forest(rng, T, leaves, F, K, odd)
    X = rng.normal(size=(n, F + 3)).astype(np.float32)
    X[rng.random(X.shape) < 0.02] = np.nan
    X[rng.random(X.shape) < 0.01] = np.inf
    dev = torch.device("cuda", 0)
    D = {k: torch.from_numpy(v).to(dev) for k, v in A.items()}
    Xd = torch.from_numpy(X).to(dev)
    p = lambda t: ctypes.c_void_p(t.data_ptr() if t is not None else 0)
    for accumulate in (0, 1):
        start = rng.normal(size=n).astype(np.float32) if accumulate else np.full(n, 0.25, np.float32)
        out = torch.from_numpy(start.copy()).to(dev)
        lo, hi = (D["lo"], D["hi"]) if K and clamp else (None, None)
        _lib.check(_lib.load().yabt_predict(
            p(Xd), F + 3, n, F, T, p(D["off"]), int(A["off"][-1]), p(D["feature"]), p(D["thr"]), p(D["left"]),
            p(D["right"]), p(D["value"]), K, p(D.get("net_k")), p(D.get("net_feats")), p(D.get("lin")), p(lo), p(hi),
            ctypes.c_float(0.25), accumulate, p(out), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
            "yabt_predict")
        with np.errstate(invalid="ignore"):
            want = numpy_predict(A, X[:, :F], K, clamp, start)
        got = out.cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))
