"""GPU parity of the small top-k draw at the lengths where its list changes path, bit for bit
against the oracle: lists ranked by all pairs (up to 1024 elements), longer ones (ties in the
threshold bin), ones past the list's capacity (the literal rule), k around the largest."""
import numpy as np
import pytest
import torch

from helpers import say
from test_gpu_sample import TD, case, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top_k,top_p", [(1, 0.0), (2, 0.3), (64, 0.95), (1000, 0.9), (1024, 0.0), (1024, 0.999), (1025, 0.9)])
@pytest.mark.parametrize("dt,V", [("bf16", 20011), ("f32", 8192)])
def test_lengths(gpu, dt, V, top_k, top_p):
    lg, host, drafts, n, u = case(6, 2, V, dt, seed=top_k + V, accept_all=1.0)
    check(lg, host, drafts, n, u, 0.9, top_k, top_p, f"topk dt={dt} V={V} k={top_k} p={top_p}")


@pytest.mark.parametrize("ties", [500, 1500, 4500])
@pytest.mark.parametrize("top_p", [0.0, 0.9])
def test_crowded_threshold(gpu, ties, top_p):
    """`ties` equal logits around the k-th: the list holds them all, ties kept by index."""
    say(f"topk ties={ties} p={top_p}")
    B, K, V, top_k = 4, 1, 16000, 300
    lg, host, drafts, n, u = case(B, K, V, "f32", seed=ties, accept_all=1.0)
    host = host.copy()
    rng = np.random.default_rng(ties)
    for b in range(B):
        at = rng.permutation(V)
        host[b, :, at[:ties]] = 9.0
        host[b, :, at[ties:ties + 200]] = 9.0 + rng.random((200, 1)).astype(np.float32)
    n[:] = 0
    check(torch.from_numpy(host).to(TD["f32"]), host, drafts, n, u, 0.9, top_k, top_p, f"ties={ties} p={top_p}")


def test_special_rows(gpu):
    """-inf below the k-th element, NaN, +inf, one sure token, +0 and -0 as ties."""
    B, K, V = 5, 0, 6000
    host = np.random.default_rng(2).normal(0, 2, (B, 1, V)).astype(np.float32)
    host[0, 0, 30:] = -np.inf
    host[1, 0, 77] = np.nan
    host[2, 0, 78] = np.inf
    host[3, 0, 79] = 80.0
    host[4] = np.where(np.arange(V) % 2, 0.0, -0.0)
    host[4, 0, :10] = 1.0
    drafts, n = np.zeros((B, 0), np.int32), np.zeros(B, np.int32)
    for top_k, top_p in [(40, 0.9), (40, 0.0), (3, 0.5)]:
        for u in (0.0, 0.37, 0.999999):
            check(torch.from_numpy(host), host, drafts, n, np.full(B, u), 0.8, top_k, top_p, f"special k={top_k} p={top_p} u={u}")


@pytest.mark.parametrize("top_k,top_p", [(400, 0.0), (401, 0.0), (401, 0.9), (768, 0.9), (769, 0.9), (768, 0.0)])
@pytest.mark.parametrize("dt,V", [("bf16", 20011), ("f32", 900)])
def test_k_around_the_largest_list(gpu, dt, V, top_k, top_p):
    lg, host, drafts, n, u = case(6, 1, V, dt, seed=top_k + V, accept_all=1.0)
    check(lg, host, drafts, n, u, 0.9, top_k, top_p, f"topk limit dt={dt} V={V} k={top_k} p={top_p}")
