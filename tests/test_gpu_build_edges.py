"""Index build at the edges of the term scan's runs (16 waves of 64-term steps) and
of the per-list passes' parts (one wave per 8192 docs, at most 16)."""
import numpy as np
import pytest
import torch

import gpusparse as gs
import oracle.oracle as O
from helpers import random_csr

pytestmark = pytest.mark.gpu

FIELDS = ("doc_ids", "scores", "offsets", "lengths", "padded_lengths", "max_scores")


def assert_built(csr, device):
    ix = gs.build_from_csr(csr, device)
    ref = O.build_index(csr.indptr, csr.indices, csr.data, csr.shape[0], csr.shape[1])
    for f in FIELDS:
        assert np.array_equal(getattr(ix, f).cpu().numpy(), ref[f]), f
    return ix


@pytest.mark.parametrize("vocab", [1, 63, 64, 65, 1023, 1024, 1025, 8193, 16385, 70001])
def test_term_scan_edges(device, vocab):
    print(f"term scan vocab={vocab}", flush=True)
    assert_built(random_csr(np.random.default_rng(vocab), 300, vocab, max_len=40), device)


@pytest.mark.parametrize("n_docs", [8191, 8192, 16383, 16385, 131071, 131073])
def test_list_parts(device, n_docs):
    print(f"list parts n_docs={n_docs}", flush=True)
    d = np.arange(n_docs)
    held = np.stack([d % 2 == 0, d >= 0, d % 97 == 5, d == n_docs - 1, np.zeros(n_docs, bool)], axis=1)
    idx = np.nonzero(held)[1].astype(np.int32)
    rng = np.random.default_rng(1)
    w = rng.normal(size=idx.size).astype(np.float32)  # negative maxima included
    csr = gs.CSR(np.concatenate([[0], np.cumsum(held.sum(axis=1))]).astype(np.int64), idx, w, held.shape)
    ix = assert_built(csr, device)
    assert gs.check_lists(ix) == (0, 4) and not ix.aux()["dup"].any()
    max_abs = np.array([np.abs(w[idx == t]).max() if (idx == t).any() else 0.0 for t in range(5)], np.float32)
    assert np.array_equal(ix.aux()["max_abs"].cpu().numpy(), max_abs)
    # a swap and a repeat anywhere in the long list are found, whichever part holds them
    for at in (1, 4095, n_docs // 2, n_docs - 1):
        docs = ix.doc_ids.clone()
        o = int(ix.offsets[1])
        docs[o + at] = docs[o + at - 1]
        bad = gs.GPUInvertedIndex(docs, ix.scores, ix.offsets, ix.lengths, ix.padded_lengths, ix.max_scores, n_docs, 5,
                                  ix.device)
        assert gs.check_lists(bad) == (0, 4) and bad.aux()["dup"].tolist() == [0, 1, 0, 0, 0]
        docs[o + at - 1], docs[o + at] = int(ix.doc_ids[o + at]), int(ix.doc_ids[o + at - 1])
        assert gs.check_lists(bad)[0] == 1
