"""Row selection at the sizes where its branches change: lists the registers hold
or not, the radix select's early stop, ties cut by doc id, tails of a compacted
span, against the oracle's exact top-k."""
import numpy as np
import pytest
import torch

import gpusparse as gs
import oracle.oracle as O
from helpers import random_csr, random_queries

pytestmark = pytest.mark.gpu


def rows_of(kind, L, rng):
    x = rng.normal(size=(3, L)).astype(np.float32)
    if kind == "ties":           # few distinct values: the cut falls inside a run of ties
        # + 0.0: no -0.0, which the selection's bit order puts below 0.0 and numpy's sort beside it
        x = np.round(x * 2).astype(np.float32) + np.float32(0.0)
    elif kind == "equal":        # no key bit differs
        x[:] = -2.5
    elif kind == "close":        # keys differ in their low bits only
        x = (1.0 + np.arange(3 * L).reshape(3, L) % 513 * 2.0 ** -23).astype(np.float32)
    elif kind == "wide":         # infinities, the lowest value, both signs
        x[:, ::7] = np.inf
        x[:, 1::7] = -np.inf
        x[:, 2::7] = np.finfo(np.float32).min
    return x


@pytest.mark.parametrize("kind", ["random", "ties", "equal", "close", "wide"])
@pytest.mark.parametrize("L", [1, 63, 512, 513, 1025, 8191, 8193, 16385, 70001])
def test_row_selection(device, kind, L):
    x = rows_of(kind, L, np.random.default_rng(L))
    xd = torch.from_numpy(x).to(device)
    for k in sorted({1, 2, 255, 256, 257, 512, 1000, 4096, 4097, 8192, L}):
        if k > min(L, gs.MAX_K):
            continue
        print(f"topk_rows {kind} L={L} k={k}", flush=True)
        v, i = gs.topk_rows(xd, k)
        ov, oi = O.compacted_topk(x, None, k)
        assert np.array_equal(i.cpu().numpy(), oi) and np.array_equal(v.cpu().numpy(), ov)


@pytest.mark.parametrize("L", [1, 255, 4095, 4096, 4097, 12289, 20000])
def test_compaction_spans(device, L):
    rng = np.random.default_rng(L)
    wide = rng.normal(size=(4, L + 3)).astype(np.float32)
    x = wide[:, 1:L + 1]  # rows at any alignment, ld > L
    tau = np.array([-np.inf, np.sort(x[1])[-max(1, L // 50)], 0.0, 50.0], np.float32)
    xd = torch.from_numpy(wide).to(device)[:, 1:L + 1]
    for k in sorted({1, min(10, L), min(1000, L)}):
        for max_cand in (k, 8192):
            print(f"compacted_topk L={L} k={k} max_cand={max_cand}", flush=True)
            v, i = gs.compacted_topk(xd, torch.from_numpy(tau).to(device), k, max_cand=max_cand)
            ov, oi = O.compacted_topk(x, tau, k)
            assert np.array_equal(i.cpu().numpy(), oi) and np.array_equal(v.cpu().numpy(), ov)


@pytest.mark.parametrize("L", [300, 4097, 9000])
def test_compaction_of_nan(device, L):
    """NaN scores reach no threshold: they are not among the candidates."""
    rng = np.random.default_rng(L)
    x = rng.normal(size=(3, L)).astype(np.float32)
    x[:, ::3] = np.nan
    x[1, 1::3] = np.copysign(np.float32(np.nan), np.float32(-1))
    x[2] = np.nan
    tau = np.array([0.0, -np.inf, -np.inf], np.float32)
    v, i = gs.compacted_topk(torch.from_numpy(x).to(device), torch.from_numpy(tau).to(device), 250)
    ov, oi = O.compacted_topk(x, tau, 250)
    assert np.array_equal(i.cpu().numpy(), oi) and np.array_equal(v.cpu().numpy(), ov)


@pytest.mark.parametrize("n_docs", [1, 255, 256, 257, 4095, 4097, 20001])
@pytest.mark.parametrize("kind", ["f32", "f16", "u8", "repeats", "negative", "few"])
def test_dense_rows(device, kind, n_docs):
    """The dense path's slices (256 docs), searches inside a tile, score bins and
    candidate lists: docs at their edges, lists with repeated docs, negative and
    zero scores (no positive bin holds k docs), more terms than lanes."""
    rng = np.random.default_rng(n_docs)
    dt = {"f16": np.float16, "u8": np.uint8}.get(kind, np.float32)
    csr = random_csr(rng, n_docs, 90, max_len=60, dtype=dt, dup_rate=0.3 if kind == "repeats" else 0.0)
    if kind == "negative":
        csr = csr._replace(data=(csr.data - 1.0).astype(np.float32))
    ix = gs.build_from_csr(csr, device)
    ref = O.build_index(csr.indptr, csr.indices, csr.data, csr.shape[0], csr.shape[1])
    ti, tw = random_queries(rng, 5, 90, max_len=80, dtype=np.uint8 if kind == "u8" else np.float32, invalid_rate=0.1,
                            pad_to=80)
    if kind == "few":
        ti[:, 1:] = -1
    for k in sorted({1, min(10, n_docs), min(700, n_docs)}):
        for tile_log2 in (8, 10, 14):
            print(f"dense {kind} n_docs={n_docs} k={k} tile_log2={tile_log2}", flush=True)
            s, i = gs.search(ix, (ti, tw), k, path="dense", tile_log2=tile_log2)
            es, ei = O.search(ref, ti, tw, k)
            assert np.array_equal(i.cpu().numpy(), ei) and np.array_equal(s.cpu().numpy(), es.astype(s.cpu().numpy().dtype))


def test_dense_rows_of_ties_and_small_workspaces(device):
    """More docs in the highest bins than candidate slots, and a workspace with room
    for the scores only: both select from the whole row."""
    n = 40000
    rng = np.random.default_rng(5)
    indptr = np.arange(n + 1, dtype=np.int64)
    csr = gs.CSR(indptr, np.zeros(n, np.int32), np.full(n, 0.5, np.float32), (n, 3))
    ix = gs.build_from_csr(csr, device)
    ti, tw = np.array([[0], [1]], np.int32), np.ones((2, 1), np.float32)
    for k in (1, 1000):
        s, i = gs.search(ix, (ti, tw), k, path="dense")
        assert np.array_equal(i.cpu().numpy(), np.tile(np.arange(k), (2, 1)))
        assert np.array_equal(s.cpu().numpy(), np.array([[0.5] * k, [0.0] * k], np.float32))
    csr = random_csr(rng, 3000, 50, max_len=20)
    ix = gs.build_from_csr(csr, device)
    ti, tw = random_queries(rng, 4, 50)
    es, ei = gs.search(ix, (ti, tw), 20, path="dense")
    per_row = 4096 * 8  # one row's scores at 4096-doc tiles
    s, i = gs.search(ix, (ti, tw), 20, path="dense", tile_log2=12, dense_budget=per_row)
    assert torch.equal(s, es) and torch.equal(i, ei)
    # through the C ABI with exactly those bytes
    from gpusparse import _lib
    from gpusparse.index import gs_index_struct
    gidx = gs_index_struct(ix, 12)
    qt, qw = torch.from_numpy(ti).to(device), torch.from_numpy(tw).to(device)
    ws = torch.empty(per_row, dtype=torch.uint8, device=device)
    s, i = torch.empty_like(es), torch.empty_like(ei)
    _lib.check(_lib.lib().gs_search_dense(_lib.C.byref(gidx), _lib.ptr(qt), _lib.ptr(qw), 4, qt.shape[1], 20, None, 4,
                                          _lib.ptr(s), _lib.ptr(i), _lib.ptr(ws), ws.numel(),
                                          _lib.stream_ptr(device)), "gs_search_dense")
    assert torch.equal(s, es) and torch.equal(i, ei)
