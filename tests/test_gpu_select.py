"""Row selection at the sizes where its branches change: lists the registers hold
or not, the radix select's early stop, ties cut by doc id, tails of a compacted
span, against the oracle's exact top-k."""
import numpy as np
import pytest
import torch

import gpusparse as gs
import oracle.oracle as O

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
