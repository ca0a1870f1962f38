"""GPU parity of the greedy segment scan at the edges of its vectors: rows that start off a
16-byte boundary, vocabularies around a segment and a vector, maxima at every cut, ties, NaN."""
import numpy as np
import pytest
import torch

import gollmgo_amd.verify as gv
from helpers import say

pytestmark = pytest.mark.gpu


def argmax_first(row):
    """First index of the maximum by a sequential `>` scan from element 0 (NaN never wins)."""
    if np.isnan(row[0]):
        return 0
    return int(np.nanargmax(row))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1, 7, 9, 4095, 4096, 4097, 4099, 8193, 12287])
def test_argmax_of_rows_at_any_alignment(gpu, dt, V):
    say(f"greedy rows {dt} V={V}")
    B, K = 3, 2
    rng = np.random.default_rng(V)
    x = rng.integers(-4, 4, (B, K + 1, V)).astype(np.float32)  # many ties
    cuts = [0, V - 1, V // 2, min(V - 1, 4095), min(V - 1, 4096), max(0, V - 9)]
    for i in range(B * (K + 1)):
        x[i // (K + 1), i % (K + 1), cuts[i % len(cuts)]] = 9.0
    x[0, 0, min(V - 1, 3)] = np.nan
    x[1, 0, :] = -np.inf
    logits = torch.from_numpy(x).to(dt).cuda()
    rows = logits.float().cpu().numpy()
    best = np.array([[argmax_first(rows[b, j]) for j in range(K + 1)] for b in range(B)])
    drafts = best[:, :K].astype(np.int32)
    drafts[2, 1] = -1  # rejected
    acc, tok = gv.accept_greedy(logits, torch.from_numpy(drafts).cuda(), torch.full((B,), K, dtype=torch.int32, device="cuda"))
    assert acc.tolist() == [K, K, 1]
    assert tok.tolist() == [best[0, K], best[1, K], best[2, 1]]


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,V", [(342, 7), (341, 4097), (342, 4097), (342, 2051)])
def test_argmax_of_many_rows(gpu, dt, B, V):
    """More segments than a wave per SIMD (whole segments per wave), and around that number."""
    say(f"greedy many rows {dt} B={B} V={V}")
    K = 2
    x = np.random.default_rng(V + B).integers(-4, 4, (B, K + 1, V)).astype(np.float32)
    x[5, 0, :] = -np.inf
    x[6, 1, 0] = np.nan
    best = np.array([[argmax_first(row) for row in rows] for rows in x])
    drafts = best[:, :K].astype(np.int32)
    acc, tok = gv.accept_greedy(torch.from_numpy(x).to(dt).cuda(), torch.from_numpy(drafts).cuda(),
                                torch.full((B,), K, dtype=torch.int32, device="cuda"))
    assert acc.tolist() == [K] * B
    assert tok.tolist() == best[:, K].tolist()
