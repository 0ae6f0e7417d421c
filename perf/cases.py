"""The retrieval work that this library is timed on, as cases with inputs of their own.

Collections and queries follow the laws of the repository's synthetic
configurations (gpusparse.synth): a SPLADE-like collection has about 120 terms a
document (lognormal row lengths), Zipf term ids over 30522 terms without
repeats inside a row and lognormal(-0.5, 0.8) weights clipped to 3; queries have
about 30 terms of the same laws, padded with -1 to the widest of the batch.
They are drawn here with torch on the GPU, from the seed alone.

A case is a dict of plain values:

  call     "search"    gpusparse.search(index, (terms, weights), k)
           "fused"     triton_fused_score, the reference's name for it
           "chunked"   triton_chunked_score_fused with the chunk bounds in hand
           "stream"    search_async over batches of 200 queries, two in flight, as
                       engine.retrieve drives it, without its Python rankings
           "build"     build_index from a host CSR
           "topk"      compacted_topk of dense fp32 score rows
  n_docs, zipf, weights ("f32", "f16", "u8")        the collection
  batch, q_mean, q_min, q_max, q_head, k            the queries and the answer
  rows, cols, k, keep                               the score rows of "topk"
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-sparse_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

VOCAB = 30522
W_MU, W_SIGMA, W_MAX = -0.5, 0.8, 3.0
DOC_MEAN, DOC_SIGMA, DOC_MIN, DOC_MAX = 120.0, 0.5, 16, 512
ROWS_PER_CHUNK = 1 << 15          # generated rows whose (row, term) keys fit int32 (32768 * 30522 < 2^31)
DOC_CHUNK = 131072                # the reference's chunk width (triton_chunked_score_fused)
BATCH = 200                       # queries per batch of a retrieval loop (retrieve's default)
W_BYTES = {"f32": 4, "f16": 2, "u8": 1}
TORCH_W = {"f32": torch.float32, "f16": torch.float16, "u8": torch.uint8}


def _search(name, call, n_docs, weights, batch, k, zipf=1.1, q_mean=30.0, q_min=4, q_max=107, q_head=0):
    case = {"call": call, "n_docs": n_docs, "zipf": zipf, "weights": weights, "batch": batch, "q_mean": q_mean,
            "q_min": q_min, "q_max": q_max, "q_head": q_head, "k": k}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one interactive query on a small collection: launches and latency
        _search("one_query_100k", "search", 100_000, "f32", 1, 10),
        # an offline batch on the same collection (configuration C1)
        _search("batch_100k", "search", 100_000, "f32", 256, 10),
        # one query, first page of results, on a collection of ordinary size with a ragged tail
        _search("one_query_1m", "fused", 1_000_003, "f16", 1, 100),
        # a serving batch on the large collection: few queries, latency matters
        _search("serving_8m", "search", 8_800_000, "f16", 16, 1000),
        # the headline: the large collection, offline batches (configuration C3)
        _search("batch_8m", "search", 8_800_000, "f16", 512, 1000),
        # ordinary collection, wide batches, fp32 weights (configuration C2)
        _search("batch_1m", "search", 1_000_000, "f32", 1024, 1000),
        # head-heavy terms and long queries (configuration C4's laws)
        _search("head_heavy_1m", "search", 1_000_000, "f32", 512, 1000, zipf=1.3, q_mean=80.0, q_min=16, q_max=256,
                q_head=8),
        # quantized impacts (configuration C5's laws), a ragged batch through the chunked entry point
        _search("impacts_3m", "chunked", 3_000_017, "u8", 200, 1000),
        # a retrieval loop with batches in flight: three batches, the last one short
        _search("stream_300k", "stream", 300_007, "f32", 437, 100),
        # indexing: host CSR to a GPU index
        {"name": "build_1m", "call": "build", "n_docs": 1_000_000, "zipf": 1.1, "weights": "f32"},
        {"name": "build_30k", "call": "build", "n_docs": 30_011, "zipf": 1.1, "weights": "f16"},
        # selection over dense score rows of one chunk's width, 2% of them above the threshold
        {"name": "topk_rows", "call": "topk", "rows": 64, "cols": DOC_CHUNK, "k": 1000, "keep": 0.02},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search"] * 4 + ["fused", "chunked", "stream", "build", "topk"])
    if kind == "topk":
        rows = _log_uniform(rng, 1, 512)
        cols = _log_uniform(rng, 4096, 1 << 20)
        while rows * cols > 64 << 20:
            rows = (rows + 1) // 2
        return {"call": kind, "rows": rows, "cols": cols, "k": _log_uniform(rng, 10, 1000),
                "keep": rng.choice([0.0, 0.005, 0.02])}
    n_docs = _log_uniform(rng, 20_000, 4_000_000)
    weights = rng.choice(["f32", "f16", "u8"])
    if kind == "build":
        return {"call": kind, "n_docs": min(n_docs, 1_500_000), "zipf": rng.choice([1.1, 1.3]), "weights": weights}
    if kind == "stream":
        return _search(None, kind, min(n_docs, 1_000_000), rng.choice(["f32", "f16"]), rng.randint(1, 600),
                       rng.choice([10, 100]))
    long_q = rng.random() < 0.25
    batch = _log_uniform(rng, 1, 1024)
    if long_q:
        batch = min(batch, 512)
    return _search(None, kind, n_docs, weights, batch, _log_uniform(rng, 10, 1000),
                   zipf=1.3 if long_q else 1.1, q_mean=80.0 if long_q else 30.0, q_min=16 if long_q else 4,
                   q_max=256 if long_q else 107, q_head=8 if long_q else 0)


# ---------------------------------------------------------------------- inputs


def _zipf_p(s):
    p = np.arange(1, VOCAB + 1, dtype=np.float64) ** -s
    return p / p.sum()


# draws with repeats that leave about `mean` distinct terms a row, per mean
def _oversample(mean, zipf):
    p = _zipf_p(zipf)
    lo, hi = 1.0, 8.0
    for _ in range(30):
        mid = 0.5 * (lo + hi)
        if (1.0 - (1.0 - p) ** (mid * mean)).sum() < mean:
            lo = mid
        else:
            hi = mid
    return hi


def _rows(gen, n, mean, sigma, lo, hi, zipf, weights, dev, head=0):
    """(row lengths int64 [n], term ids int32, weights) on the GPU; terms ascending
    and distinct inside a row.  `head`: that many draws more of the 50 first terms."""
    cdf = torch.from_numpy(np.cumsum(_zipf_p(zipf))).to(dev)
    over = _oversample(mean, zipf)
    z = torch.randn(n, generator=gen, device=dev, dtype=torch.float64)
    want = torch.exp(math.log(mean) - sigma * sigma / 2 + sigma * z).round().clamp(lo, hi)
    draws = (want * over).ceil().to(torch.int64)
    lens, terms, vals = [], [], []
    for r0 in range(0, n, ROWS_PER_CHUNK):
        d = draws[r0:r0 + ROWS_PER_CHUNK]
        m = d.numel()
        rid = torch.repeat_interleave(torch.arange(m, device=dev, dtype=torch.int32), d)
        u = torch.rand(rid.numel(), generator=gen, device=dev, dtype=torch.float64)
        t = torch.searchsorted(cdf, u, out_int32=True).clamp_(max=VOCAB - 1)
        key = rid * VOCAB + t
        if head:
            hr = torch.arange(m, device=dev, dtype=torch.int32).repeat_interleave(head)
            key = torch.cat([key, hr * VOCAB + torch.randint(0, 50, (hr.numel(),), generator=gen, device=dev,
                                                             dtype=torch.int32)])
        key = torch.sort(key).values
        key = key[torch.cat([torch.ones(1, dtype=torch.bool, device=dev), key[1:] != key[:-1]])]
        row = torch.div(key, VOCAB, rounding_mode="floor")
        if hi <= 256:  # queries: never more than `hi` terms
            start = torch.searchsorted(row, torch.arange(m, device=dev, dtype=torch.int32))
            key = key[torch.arange(key.numel(), device=dev) - start[row.long()] < hi]
            row = torch.div(key, VOCAB, rounding_mode="floor")
        w = torch.exp(W_MU + W_SIGMA * torch.randn(key.numel(), generator=gen, device=dev)).clamp_(max=W_MAX)
        if weights == "u8":
            w = (w * (255.0 / W_MAX)).round().clamp_(1, 255)
        lens.append(torch.bincount(row, minlength=m))
        terms.append(key - row * VOCAB)
        vals.append(w.to(TORCH_W[weights]))
    return torch.cat(lens), terms, vals


def _docs(case, seed, dev):
    if case["call"] == "build":
        # One structure per case, its rows in an order and with weights of the
        # seed's own: every seed's index has the same number of posting slots.
        lens, terms, _ = _rows(torch.Generator(device=dev).manual_seed(7), case["n_docs"], DOC_MEAN, DOC_SIGMA,
                               DOC_MIN, DOC_MAX, case["zipf"], "f32", dev)
        gen = torch.Generator(device=dev).manual_seed(2 * int(seed) + 1)
        perm = torch.randperm(case["n_docs"], generator=gen, device=dev)
        start = torch.cumsum(lens, 0) - lens
        new = lens[perm]
        at = torch.arange(int(new.sum()), device=dev)
        at += torch.repeat_interleave(start[perm] - (torch.cumsum(new, 0) - new), new)
        w = torch.exp(W_MU + W_SIGMA * torch.randn(at.numel(), generator=gen, device=dev)).clamp_(max=W_MAX)
        if case["weights"] == "u8":
            w = (w * (255.0 / W_MAX)).round().clamp_(1, 255)
        return new, [torch.cat(terms)[at]], [w.to(TORCH_W[case["weights"]])]
    gen = torch.Generator(device=dev).manual_seed(2 * int(seed) + 1)
    return _rows(gen, case["n_docs"], DOC_MEAN, DOC_SIGMA, DOC_MIN, DOC_MAX, case["zipf"], case["weights"], dev)


def _doc_csr(case, seed, dev):
    from gpusparse import CSR
    lens, terms, vals = _docs(case, seed, dev)
    indptr = np.zeros(case["n_docs"] + 1, dtype=np.int64)
    np.cumsum(lens.cpu().numpy(), out=indptr[1:])
    indices = torch.empty(int(indptr[-1]), dtype=torch.int32)
    data = torch.empty(int(indptr[-1]), dtype=TORCH_W[case["weights"]])
    at = 0
    for t, v in zip(terms, vals):
        indices[at:at + t.numel()] = t.cpu()
        data[at:at + t.numel()] = v.cpu()
        at += t.numel()
    return CSR(indptr, indices.numpy(), data.numpy(), (case["n_docs"], VOCAB))


def _queries(case, seed, dev):
    """(term ids int32 [B, T] padded with -1, weights [B, T] padded with 0)."""
    gen = torch.Generator(device=dev).manual_seed(2 * int(seed) + 2)
    w = "u8" if case["weights"] == "u8" else "f32"
    lens, terms, vals = _rows(gen, case["batch"], case["q_mean"], 0.5, case["q_min"], case["q_max"], case["zipf"], w,
                              dev, case["q_head"])
    T = int(lens.max())
    mask = torch.arange(T, device=dev)[None, :] < lens[:, None]
    qt = torch.full(mask.shape, -1, dtype=torch.int32, device=dev)
    qw = torch.zeros(mask.shape, dtype=TORCH_W[w], device=dev)
    qt[mask] = torch.cat(terms)
    qw[mask] = torch.cat(vals)
    return qt, qw


def _score_rows(case, seed, dev):
    """Dense fp32 score rows and the thresholds that a share `keep` of each row reaches."""
    gen = torch.Generator(device=dev).manual_seed(2 * int(seed) + 1)
    x = torch.randn(case["rows"], case["cols"], generator=gen, device=dev).exp_()
    if not case["keep"]:
        return x, None
    at = max(1, int(case["cols"] * case["keep"]))
    return x, torch.topk(x, at, dim=1).values[:, -1].contiguous()


def prepare(case, seed):
    import gpusparse as gs
    dev = torch.device("cuda:0")
    call = case["call"]
    if call == "topk":
        x, tau = _score_rows(case, seed, dev)
        return {"case": case, "scores": x, "tau": tau}
    csr = _doc_csr(case, seed, dev)
    if call == "build":
        return {"case": case, "csr": csr, "device": dev}
    index = gs.build_from_csr(csr, dev)
    qt, qw = _queries(case, seed, dev)
    state = {"case": case, "index": index, "qt": qt, "qw": qw}
    if call == "chunked":
        state["bounds"] = gs.build_chunk_boundaries(index, DOC_CHUNK)
    return state


def run(state):
    import gpusparse as gs
    case = state["case"]
    call = case["call"]
    if call == "topk":
        return gs.compacted_topk(state["scores"], state["tau"], case["k"])
    if call == "build":
        ix = gs.build_index(state["csr"], state["device"], weight_dtype=TORCH_W[case["weights"]])
        return {"doc_ids": ix.doc_ids, "scores": ix.scores, "offsets": ix.offsets, "lengths": ix.lengths,
                "padded_lengths": ix.padded_lengths, "max_scores": ix.max_scores}
    index, qt, qw, k = state["index"], state["qt"], state["qw"], case["k"]
    if call == "search":
        return gs.search(index, (qt, qw), k)
    if call == "fused":
        return gs.triton_fused_score(index, qt, qw, top_k=k)
    if call == "chunked":
        return gs.triton_chunked_score_fused(index, qt, qw, top_k=k, doc_chunk=DOC_CHUNK,
                                             chunk_bounds=state["bounds"])
    pending, done = [], []
    for b in range(0, case["batch"], BATCH):
        if len(pending) == 2:
            done.append(pending.pop(0).result())
        pending.append(gs.search_async(index, (qt[b:b + BATCH], qw[b:b + BATCH]), k, path="fused"))
    done += [p.result() for p in pending]
    return {"scores": [s for s, _ in done], "ids": [i for _, i in done]}


# ---------------------------------------------------------------------- what a pass needs


def _held(mean, sigma, zipf, head=0):
    """Share of the rows that hold each term (row lengths at their mean)."""
    p = _zipf_p(zipf)
    absent = (1.0 - p) ** (mean * _oversample(mean, zipf))
    if head:
        absent[:50] *= (1.0 - 1.0 / 50) ** head
    return 1.0 - absent


def work(case):
    if case["call"] == "topk":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n + 12 * case["rows"] * case["k"], "flops": n}
    held = _held(DOC_MEAN, DOC_SIGMA, case["zipf"]) * case["n_docs"]
    slot = 4 + W_BYTES[case["weights"]]
    if case["call"] == "build":
        # the CSR read and the term-major postings written
        return {"bytes": float(2 * slot * held.sum() + 8 * case["n_docs"]), "flops": float(held.sum())}
    # every posting of a term of the batch read once; a multiply and an add per
    # (query, posting)
    q = _held(case["q_mean"], 0.5, case["zipf"], case["q_head"])
    B = case["batch"]
    live = 1.0 - (1.0 - q) ** B
    return {"bytes": float(slot * (held * live).sum() + 8 * B * q.sum() + 12 * B * case["k"]),
            "flops": float(2.0 * B * (held * q).sum())}


def tolerance(case):
    # Scores are the fp64 sums rounded once to fp32 (uint8: exact integer sums),
    # ties ordered by doc id; the index and the selected rows are moved data.
    return "exact"


# ---------------------------------------------------------------------- 64-bit results


def _exact_scores(case, seed, dev):
    """fp64 [B, k] best scores of each query, best first: the sums over the
    query's terms, collected per run of documents and merged."""
    lens, terms, vals = _docs(case, seed, dev)
    qt, qw = (x.cpu() for x in _queries(case, seed, dev))
    B, k = case["batch"], min(case["k"], case["n_docs"])
    queries = [[(int(t), float(w)) for t, w in zip(qt[b], qw[b]) if t >= 0] for b in range(B)]
    best = torch.zeros(B, 0, dtype=torch.float64, device=dev)
    per = max(1, min(32, (4 << 30) // (8 * B * ROWS_PER_CHUNK)))  # generated chunks a run takes
    for c0 in range(0, len(terms), per):
        r0 = c0 * ROWS_PER_CHUNK
        ln = lens[r0:r0 + per * ROWS_PER_CHUNK]
        m = ln.numel()
        t = torch.cat(terms[c0:c0 + per])
        doc = torch.repeat_interleave(torch.arange(m, device=dev), ln)
        t, order = torch.sort(t, stable=True)
        doc = doc[order]
        w = torch.cat(vals[c0:c0 + per])[order].double()
        ends = torch.searchsorted(t, torch.arange(VOCAB + 1, device=dev, dtype=torch.int32)).tolist()
        acc = torch.zeros(B, m, dtype=torch.float64, device=dev)
        for b, terms_b in enumerate(queries):
            row = acc[b]
            for tt, q in terms_b:
                lo, hi = ends[tt], ends[tt + 1]
                if hi > lo:
                    row.index_add_(0, doc[lo:hi], w[lo:hi], alpha=q)
        best = torch.topk(torch.cat([best, torch.topk(acc, min(k, m), dim=1).values], dim=1),
                          min(k, best.shape[1] + min(k, m)), dim=1).values
        del acc, doc, w, t, order
    return best


def exact(case, seed):
    dev = torch.device("cuda:0")
    if case["call"] == "build":
        return None  # moved data, no computed numbers
    if case["call"] == "topk":
        x, tau = _score_rows(case, seed, dev)
        x = x.double()
        if tau is not None:  # rows with fewer than k scores reaching their threshold end in -inf
            x = x.masked_fill(x < tau[:, None], -math.inf)
        return torch.topk(x, case["k"], dim=1).values, None
    s = _exact_scores(case, seed, dev)
    if case["call"] == "stream":
        parts = list(torch.split(s, BATCH))
        return {"scores": parts, "ids": [None] * len(parts)}
    return s, None
