"""The block search (128 heavy terms as int8 products on 64-doc blocks, the other
terms added in an LDS tile) against the oracle: block, chunk and group edges,
signs, repeated terms, and its copy's levels and words."""
import sys
import threading

import numpy as np
import pytest
import torch

import gpusparse as gs
import oracle.oracle as O
from gpusparse import synth
from gpusparse.index import ensure_blocks
from gpusparse._lib import BLOCK_HEAVY as H
from helpers import random_csr, random_queries

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_batch(monkeypatch):
    """Batches of any size on the block search, which the library keeps for large ones."""
    module = sys.modules["gpusparse.search"]
    monkeypatch.setattr(module, "BLOCK_MIN_QUERIES", 1)
    monkeypatch.setattr(module, "BLOCK_MIN_PAIRS", 1)


def ref_of(csr):
    return O.build_index(csr.indptr, csr.indices, csr.data, csr.shape[0], csr.shape[1])


def check(ix, ref, ti, tw, k, what):
    assert gs.search_plan(ix, ti.shape[0], ti.shape[1], k)["blocks"], what
    print(f"blocks {what} B={ti.shape[0]} T={ti.shape[1]} k={k}", flush=True)
    s, i = gs.search(ix, (ti, tw), k, path="fused")
    es, _, ei = O.c_search(ref, ti, tw, k, threads=8)
    assert np.array_equal(i.cpu().numpy(), ei), what
    assert np.array_equal(s.cpu().numpy(), es), what


def head_tail_csr(rng, n_docs, vocab, dtype, sign=False):
    """Rows of a few of 300 frequent terms (more than the heavy ones) and of rare ones."""
    rows = []
    for _ in range(n_docs):
        a = rng.choice(min(300, vocab), size=int(rng.integers(0, 20)), replace=False)
        b = rng.choice(vocab, size=int(rng.integers(0, 12)), replace=False)
        rows.append(np.unique(np.concatenate([a, b])))
    indptr = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int64)
    idx = np.concatenate(rows).astype(np.int32) if rows else np.zeros(0, np.int32)
    w = rng.lognormal(-0.5, 0.8, size=idx.size)
    if sign:
        w *= rng.choice([-1.0, 1.0], size=idx.size, p=[0.3, 0.7])
    return gs.CSR(indptr, idx, w.astype(dtype), (n_docs, vocab))


@pytest.mark.parametrize("dtype", [np.float32, np.float16])
@pytest.mark.parametrize("sign", [False, True])
def test_block_copy(device, dtype, sign):
    """Levels and words decode to the weights within half a level; each block holds
    its postings once."""
    rng = np.random.default_rng(3)
    n, V = 1000, 2000
    csr = head_tail_csr(rng, n, V, dtype, sign)
    ix = gs.build_from_csr(csr, device)
    b = ensure_blocks(ix)
    assert b.levels == (127 if sign else 255)
    D = np.zeros((n, V))
    D[np.repeat(np.arange(n), np.diff(csr.indptr)), csr.indices] = csr.data.astype(np.float64)
    W = np.abs(D).max(axis=0)
    heavy = b.heavy.cpu().numpy()
    lengths = np.bincount(csr.indices, minlength=V)
    assert np.array_equal(np.sort(lengths[heavy])[::-1], np.sort(lengths)[::-1][:H])
    off = 128 if b.levels == 255 else 0
    # bytes of a block: [doc / 16][term / 64][term % 64 / 16][doc % 16][term % 16]
    lv = b.head.cpu().numpy().reshape(-1, 4, H // 64, 4, 16, 16).transpose(0, 1, 4, 2, 3, 5).reshape(-1, H)
    lv = lv.astype(np.float64) + off
    assert not lv[n:].any()
    assert np.abs(lv[:n] * W[heavy] / b.levels - D[:, heavy]).max() <= 0.5003 * W[heavy].max() / b.levels
    assert np.array_equal(lv[:n] != 0, np.rint(D[:, heavy] * (b.levels / W[heavy])) != 0)
    rank, words, count = b.rank.cpu().numpy(), b.tail.cpu().numpy().view(np.uint32), b.count.cpu().numpy()
    term_of = np.full(b.n_tail, -1)
    tail_terms = np.flatnonzero(rank >= H)
    term_of[rank[tail_terms] - H] = tail_terms
    got = np.zeros((n, V))
    held = np.zeros((n, V), dtype=int)
    for blk in range(count.size):
        w = words[csr.indptr[blk * 64]:][:count[blk]]
        doc, t = blk * 64 + (w >> 16 & 63), term_of[w & 0xFFFF]
        np.add.at(held, (doc, t), 1)
        got[doc, t] = (w.view(np.int32) >> 22) * W[t] / 511
    tail = np.setdiff1d(np.arange(V), heavy)
    assert np.array_equal(held[:, tail], (D != 0)[:, tail].astype(int)) and not held[:, heavy].any()
    assert (np.abs(got - D)[:, tail] <= 0.5003 * W[tail] / 511).all()


@pytest.mark.parametrize("n_docs", [1, 63, 64, 65, 1000, 33000])
@pytest.mark.parametrize("B", [1, 16, 65, 513])
def test_block_edges(device, n_docs, B):
    rng = np.random.default_rng(n_docs + B)
    csr = head_tail_csr(rng, min(n_docs, 2000), 1500, np.float32)
    if n_docs > 2000:  # repeat the rows: ties everywhere
        m = -(-n_docs // 2000)
        csr = gs.CSR(np.concatenate([[0], np.cumsum(np.tile(np.diff(csr.indptr), m))]).astype(np.int64),
                     np.tile(csr.indices, m), np.tile(csr.data, m), (2000 * m, 1500))
    ix = gs.build_from_csr(csr, device)
    ref = ref_of(csr)
    ti, tw = random_queries(rng, B, 1500, max_len=30, invalid_rate=0.05)
    ti[B // 2:, ::2] %= 300
    ti[0] = -1                                  # an empty query
    for k in sorted({1, min(100, csr.shape[0]), min(1000, csr.shape[0])}):
        check(ix, ref, ti, tw, k, f"n_docs={n_docs}")


@pytest.mark.parametrize("kind", ["f16", "sign", "repeated", "query_signs", "tiny", "few_terms", "dup_tail", "unsorted",
                                  "long_rows"])
def test_block_weights(device, kind):
    rng = np.random.default_rng(len(kind))
    n, V = 5000, 3000
    dt = np.float16 if kind == "f16" else np.float32
    csr = head_tail_csr(rng, n, 40 if kind == "few_terms" else V, dt, kind == "sign")
    if kind == "tiny":  # one heavy and some tail lists far below the others' weights
        csr.data[csr.indices % 7 == 3] *= np.float32(1e-33)
        csr.data[csr.indices % 7 == 4] *= np.float32(1e-6)
    if kind == "dup_tail":  # a rare term twice in its docs
        extra = np.zeros(n, dtype=int)
        extra[::500] = 2
        indptr = csr.indptr + np.concatenate([[0], np.cumsum(extra)])
        idx, w = np.empty(indptr[-1], np.int32), np.empty(indptr[-1], np.float32)
        for d in range(n):
            a, b = csr.indptr[d], csr.indptr[d + 1]
            row = np.concatenate([csr.indices[a:b], np.full(extra[d], V, np.int32)])
            idx[indptr[d]:indptr[d + 1]] = row
            w[indptr[d]:indptr[d + 1]] = np.concatenate([csr.data[a:b], np.arange(1, extra[d] + 1) * 0.37])
        csr = gs.CSR(indptr.astype(np.int64), idx, w, (n, V + 1))
    if kind == "unsorted":
        for d in range(n):
            p = rng.permutation(csr.indptr[d + 1] - csr.indptr[d]) + csr.indptr[d]
            csr.indices[csr.indptr[d]:csr.indptr[d + 1]] = csr.indices[p]
            csr.data[csr.indptr[d]:csr.indptr[d + 1]] = csr.data[p]
    if kind == "long_rows":  # blocks of more postings than the copy's build stages in LDS
        n = 200
        m = 200 + 60 * (np.arange(n) % 2)
        idx = np.concatenate([np.sort(rng.choice(V, size=x, replace=False)) for x in m]).astype(np.int32)
        csr = gs.CSR(np.concatenate([[0], np.cumsum(m)]).astype(np.int64), idx,
                     rng.lognormal(-0.5, 0.8, size=idx.size).astype(np.float32), (n, V))
    ix = gs.build_from_csr(csr, device)
    ref = ref_of(csr)
    ti, tw = random_queries(rng, 70, csr.shape[1], max_len=30)
    ti[:, :8] = rng.integers(0, min(300, csr.shape[1]), size=(70, 8))
    tw[:, :8] = rng.lognormal(-0.5, 0.8, size=(70, 8))
    if kind == "repeated":  # one heavy term up to 25 times, one of them large, and rare terms repeated
        ti[:, 5:] = ti[:, 5:6]
        tw[:, 6] = 3000.0
        ti[35:, 20:] = 1700
    if kind == "query_signs":
        tw *= rng.choice([-1.0, 1.0], size=tw.shape, p=[0.4, 0.6]).astype(np.float32)
    if kind == "dup_tail":
        ti[::3, 9] = V
        tw[::3, 9] = 2.0
    for k in (10, min(500, n)):
        check(ix, ref, ti, tw, k, kind)


def test_block_fallback_rows(device):
    """Rows the block search hands to the dense path: non-finite and huge query
    weights, no positive score, fewer positive docs than k, candidates past the cap."""
    rng = np.random.default_rng(8)
    csr = head_tail_csr(rng, 3000, 900, np.float32)
    ix = gs.build_from_csr(csr, device)
    ref = ref_of(csr)
    ti, tw = random_queries(rng, 60, 900, max_len=20)
    tw[1] = 0.0
    tw[2] *= -1.0
    tw[3, 0] = 1e30
    ti[4] = -1
    ti[4, 0] = int(np.argmin(np.where(np.bincount(csr.indices, minlength=900) > 0,
                                      np.bincount(csr.indices, minlength=900), 10 ** 9)))
    check(ix, ref, ti, tw, 800, "fallback rows")
    st = {}
    s, i = gs.search(ix, (ti, tw), 50, path="fused", cand_cap=100, timing=st)
    es, _, ei = O.c_search(ref, ti, tw, 50, threads=8)
    assert np.array_equal(i.cpu().numpy(), ei) and np.array_equal(s.cpu().numpy(), es) and st["dense_rows"] > 0


@pytest.mark.parametrize("cfg,n_docs,B,k", [("C2", 40000, 600, 1000), ("C3", 50001, 512, 1000), ("C4", 30000, 300, 1000),
                                            ("C5", 40000, 200, 100)])
def test_block_configs(device, cfg, n_docs, B, k):
    docs, queries = synth.generate(synth.scaled(synth.CONFIGS[cfg], n_docs=n_docs, n_queries=B))
    ix = gs.build_from_csr(docs, device)
    ref = ref_of(docs)
    ti, tw, _ = O.to_query_tensors(queries.indptr, queries.indices, queries.data)
    if cfg == "C5":
        tw = tw.astype(np.uint8)
        assert gs.search_plan(ix, B, ti.shape[1], k)["blocks"]
        s, i = gs.search(ix, (ti, tw), k, path="fused")
        es, ei = O.search(ref, ti, tw, k)
        assert np.array_equal(i.cpu().numpy(), ei) and np.array_equal(s.cpu().numpy(), es)
        return
    check(ix, ref, ti, tw, k, cfg)
    cand, resc = gs.search_counts(ix, B, ti.shape[1], k)
    assert (resc[cand >= k] >= k).all() and (cand >= resc).all()


def test_block_counts_and_plan(device):
    """search_counts reads the workspace as the search that last used it laid it out:
    `waves`, which names no launch shape, keeps the block search, and counts of
    another search are refused.  A plan that answers "blocks" makes none of the
    other scorer's copies."""
    rng = np.random.default_rng(21)
    csr = head_tail_csr(rng, 4000, 1500, np.float32)
    ix = gs.build_from_csr(csr, device)
    ti, tw = random_queries(rng, 40, 1500, max_len=20)
    ti[:, 0], tw[:, 0] = 7, 1.0
    B, T, k = 40, ti.shape[1], 50
    plan = gs.search_plan(ix, B, T, k)
    assert plan["blocks"] and "head" not in ix.aux() and \
        not any(isinstance(key, tuple) and key[0] == "packed" for key in ix.aux())
    gs.search(ix, (ti, tw), k, path="fused", waves=8)
    cand, resc = gs.search_counts(ix, B, T, k)
    gs.search(ix, (ti, tw), k, path="fused")
    cand2, resc2 = gs.search_counts(ix, B, T, k)
    assert np.array_equal(cand, cand2) and np.array_equal(resc, resc2)
    assert (cand >= resc).all() and (cand <= 4000).all() and (cand >= k).all()
    for args, opts in (((B, T, k + 1), {}), ((B, T, k), {"hybrid": True}), ((B, T, k), {"cand_cap": 4096})):
        with pytest.raises(ValueError, match="other arguments"):
            gs.search_counts(ix, *args, **opts)
    gs.search(ix, (ti, tw), k, path="fused", hybrid=True)
    cand, resc = gs.search_counts(ix, B, T, k, hybrid=True)
    assert (cand >= resc).all() and (cand <= 4000).all() and (cand >= k).all()
    with pytest.raises(ValueError, match="other arguments"):
        gs.search_counts(ix, B, T, k)


@pytest.mark.parametrize("k", [10, 100, 1000])
def test_block_ordered_collection(device, k):
    """Documents in the order of their scores, the best last, as a collection in date,
    length or topical order has them for some queries: the launches' thresholds come
    from blocks spread over the whole collection, so a query's candidates stay near
    k per launch (in id order nearly every doc was one)."""
    rng = np.random.default_rng(k)
    n, V, B = 60_000, 400, 512
    rows = np.arange(n, dtype=np.int64)
    idx = np.stack([np.zeros(n), rng.integers(1, V, size=n)], axis=1).astype(np.int32)
    w = np.stack([0.5 + rows / n, rng.uniform(0.01, 0.02, size=n)], axis=1).astype(np.float32)
    csr = gs.CSR(2 * np.arange(n + 1, dtype=np.int64), idx.ravel(), w.ravel(), (n, V))
    ix = gs.build_from_csr(csr, device)
    ti = np.stack([np.zeros(B), 1 + np.arange(B) % (V - 1)], axis=1).astype(np.int32)
    tw = np.stack([rng.uniform(0.5, 2.0, size=B), np.ones(B)], axis=1).astype(np.float32)
    check(ix, ref_of(csr), ti, tw, k, "ordered")
    st = {}
    gs.search(ix, (ti, tw), k, path="fused", timing=st)
    cand, _ = gs.search_counts(ix, B, 2, k)
    # about k in each of the at most 5 launches, the docs within the margin (W_0 / 255
    # of the scores: 0.8% of the docs) and a block's granularity of the samples
    assert st["dense_rows"] == 0 and cand.max() <= 5 * (2 * k + n * 0.008 + 256)


def one_term_csr(n, weight, vocab=50):
    """n docs that all hold term 0 with the given weights and one other term, weakly."""
    idx = np.stack([np.zeros(n), 1 + np.arange(n) % (vocab - 1)], axis=1).astype(np.int32)
    w = np.stack([np.broadcast_to(weight, n), np.full(n, 0.001)], axis=1).astype(np.float32)
    return gs.CSR(2 * np.arange(n + 1, dtype=np.int64), idx.ravel(), w.ravel(), (n, vocab))


@pytest.mark.parametrize("n,k", [(16_000, 100), (16_000, 1000), (70_000, 100)])
def test_block_list_overflow(device, n, k):
    """One block emits 64 docs x 512 queries, twice what a workgroup's list holds: the
    rest goes straight to the queries' candidates.  16000 tied docs fit a query's
    slots and its rescoring; of 70000 a query takes what fits its slots, emits no
    more, and its row is done elsewhere."""
    B = 512
    csr = one_term_csr(n, 1.0)
    ix = gs.build_from_csr(csr, device)
    ti = np.zeros((B, 1), np.int32)
    tw = np.linspace(0.5, 2.0, B, dtype=np.float32)[:, None]
    check(ix, ref_of(csr), ti, tw, k, f"list overflow n={n}")
    st = {}
    gs.search(ix, (ti, tw), k, path="fused", timing=st)
    if n == 16_000:
        cand, resc = gs.search_counts(ix, B, 1, k)
        assert st["dense_rows"] == 0 and (cand == n).all() and (resc == n).all()
    else:
        assert st["dense_rows"] == B


def test_block_large_k_slots(device):
    """The most results of the fused path on a collection of several launches: the
    queries' slots hold what all of them emit (65536 did not)."""
    rng = np.random.default_rng(5)
    n, B, k = 6_000_000, 512, 8192
    csr = one_term_csr(n, rng.lognormal(-0.5, 0.8, size=n))
    ix = gs.build_from_csr(csr, device)
    ti = np.zeros((B, 1), np.int32)
    tw = np.linspace(0.5, 2.0, B, dtype=np.float32)[:, None]
    st = {}
    s, i = gs.search(ix, (ti, tw), k, path="fused", timing=st)
    assert gs.search_plan(ix, B, 1, k)["blocks"] and st["dense_rows"] == 0
    cand, _ = gs.search_counts(ix, B, 1, k)
    assert (cand >= k).all() and cand.max() > 65536
    w = csr.data[0::2].astype(np.float64)
    for q in (0, 255, 511):
        exact = w * float(tw[q, 0])
        best = np.lexsort((np.arange(n), -exact))[:k]
        assert np.array_equal(i[q].cpu().numpy(), best)
        assert np.array_equal(s[q].cpu().numpy(), exact[best].astype(np.float32))


def outlier_csr(rng, n, vocab, per_row, times):
    """n docs of per_row distinct terms of `vocab`, and in each list one weight `times`
    the largest other."""
    idx = np.sort(np.argpartition(rng.random((n, vocab), dtype=np.float32), per_row, axis=1)[:, :per_row], axis=1)
    w = rng.uniform(0.5, 1.0, size=(n, per_row)).astype(np.float32)
    flat, first = idx.ravel(), np.unique(idx.ravel(), return_index=True)[1]
    assert first.size == vocab and flat.size == n * per_row
    w.ravel()[first] = times
    return gs.CSR(per_row * np.arange(n + 1, dtype=np.int64), flat.astype(np.int32), w.ravel(), (n, vocab))


@pytest.mark.parametrize("B", [20, 300])
def test_block_margin_too_wide(device, B):
    """Lists with one weight far above the rest: the block copy's levels, relative to a
    list's largest weight, leave more docs within the margin than are rescored.  Such
    rows are searched once more as a batch of their own (300 queries: by the hybrid
    scorer, whose margin settles them; 20: as dense rows), not one by one densely."""
    rng = np.random.default_rng(B)
    n, V, k = 60_000, 160, 500
    csr = outlier_csr(rng, n, V, 24, 200.0)
    ix = gs.build_from_csr(csr, device)
    ti, tw = random_queries(rng, B, V, max_len=10)
    ti[:, 0], tw[:, 0] = rng.integers(0, V, size=B), 1.0
    st = {}
    check(ix, ref_of(csr), ti, tw, k, "outliers")
    s, i = gs.search(ix, (ti, tw), k, path="fused", timing=st)
    assert st["retried_rows"] > B // 2
    assert st["dense_rows"] < st["retried_rows"] // 4 if B == 300 else st["dense_rows"] >= st["retried_rows"]
    # the counts are the block search's own, not those of the rows searched again
    cand, resc = gs.search_counts(ix, B, ti.shape[1], k)
    assert (cand >= k).sum() >= st["retried_rows"] and (resc == 0).sum() >= st["retried_rows"]


def test_block_retry_without_room(device, monkeypatch):
    """Rows to search again that the GPU has no workspace for: dense rows."""
    rng = np.random.default_rng(300)
    n, V, k, B = 60_000, 160, 500, 300
    csr = outlier_csr(rng, n, V, 24, 200.0)
    ix = gs.build_from_csr(csr, device)
    ti, tw = random_queries(rng, B, V, max_len=10)
    ti[:, 0], tw[:, 0] = rng.integers(0, V, size=B), 1.0
    module = sys.modules["gpusparse.search"]
    workspace = module._workspace

    def small(index, nbytes, stream_key=0, plan=None):
        if plan[0] == "scorer":
            raise torch.cuda.OutOfMemoryError("no room")
        return workspace(index, nbytes, stream_key, plan)

    monkeypatch.setattr(module, "_workspace", small)
    st = {}
    check(ix, ref_of(csr), ti, tw, k, "no room")
    gs.search(ix, (ti, tw), k, path="fused", timing=st)
    assert st["retried_rows"] > B // 2 and st["dense_rows"] >= st["retried_rows"]


def test_block_copy_threads(device, monkeypatch):
    """Threads that search a new index at once, each on a stream of its own: the block copy
    is made once, and no thread reads it before it is whole."""
    rng = np.random.default_rng(31)
    csr = head_tail_csr(rng, 20_000, 3000, np.float16)
    ref = ref_of(csr)
    batches = [random_queries(rng, 30 + 40 * i, 3000, max_len=20) for i in range(4)]
    module = sys.modules["gpusparse.index"]
    builds, blocks = [], module.Blocks
    monkeypatch.setattr(module, "Blocks", lambda *a: builds.append(1) or blocks(*a))
    for trial in range(3):
        ix = gs.build_from_csr(csr, device)
        if trial:
            ix.aux().pop("fwd")  # the doc-major copy made with the blocks, not the uploaded CSR
        torch.cuda.synchronize()
        got, start = [None] * 4, threading.Barrier(4)

        def work(i):
            with torch.cuda.stream(torch.cuda.Stream(device)):
                start.wait(60)
                got[i] = [x.cpu().numpy() for x in gs.search(ix, batches[i], 100, path="fused")]

        builds.clear()
        threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(builds) == 1 and ix.aux()["blocks"] is not None
        for (ti, tw), out in zip(batches, got):
            es, _, ei = O.c_search(ref, ti, tw, 100, threads=8)
            assert np.array_equal(out[1], ei) and np.array_equal(out[0], es)


def test_block_streams(device):
    """Batches of different sizes in flight on two streams, each with a workspace of its own."""
    rng = np.random.default_rng(32)
    csr = head_tail_csr(rng, 30_000, 3000, np.float32)
    ix, ref = gs.build_from_csr(csr, device), ref_of(csr)
    streams = [torch.cuda.Stream(device) for _ in range(2)]
    jobs = [(*random_queries(rng, B, 3000, max_len=T), k) for B, T, k in
            ((512, 30, 100), (17, 8, 1000), (300, 60, 10), (1, 30, 500), (600, 20, 50), (64, 5, 1))]
    want = [O.c_search(ref, ti, tw, k, threads=8) for ti, tw, k in jobs]
    assert gs.search_plan(ix, 17, 8, 1000)["blocks"]
    for r in range(3):
        pending = []
        for i, (ti, tw, k) in enumerate(jobs):
            with torch.cuda.stream(streams[(i + r) % 2]):
                pending.append(gs.search_async(ix, (ti, tw), k, path="fused"))
        for p, (es, _, ei) in zip(pending, want):
            s, i = p.result()
            assert np.array_equal(i.cpu().numpy(), ei) and np.array_equal(s.cpu().numpy(), es)


@pytest.mark.parametrize("vocab", [57_345, 65_663, 65_664])
def test_block_vocabulary(device, vocab):
    """The most tail lists the copy's 16-bit ranks hold, all of them non-empty, and one more,
    which the block search leaves to the hybrid one."""
    rng = np.random.default_rng(vocab)
    n, B = 1500, 512
    per = -(-vocab // n)
    rows = [np.unique(np.concatenate([np.arange(d * per, min((d + 1) * per, vocab)),
                                      rng.integers(0, 400, size=20), rng.integers(0, vocab, size=20)]))
            for d in range(n)]
    indptr = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int64)
    idx = np.concatenate(rows).astype(np.int32)
    csr = gs.CSR(indptr, idx, rng.lognormal(-0.5, 0.8, size=idx.size).astype(np.float32), (n, vocab))
    ix, ref = gs.build_from_csr(csr, device), ref_of(csr)
    ti, tw = random_queries(rng, B, vocab, max_len=30)
    ti[:, ::3] = rng.integers(vocab - 300, vocab, size=ti[:, ::3].shape)
    tw[:, ::3] = 1.0
    if vocab == 65_664:
        assert not gs.search_plan(ix, B, ti.shape[1], 20)["blocks"]
        s, i = gs.search(ix, (ti, tw), 20, path="fused")
        es, _, ei = O.c_search(ref, ti, tw, 20, threads=8)
        assert np.array_equal(i.cpu().numpy(), ei) and np.array_equal(s.cpu().numpy(), es)
        return
    assert ensure_blocks(ix).n_tail == vocab - H
    check(ix, ref, ti, tw, 20, f"vocab={vocab}")
