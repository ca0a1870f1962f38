"""GPU parity of the nucleus draw at the sizes where its ranking changes path, bit for bit
against the oracle: the cut inside a group of equal logits ranked by pairs (up to 1024), by the
radix descent, or past the gathered list (the literal rule)."""
import numpy as np
import pytest
import torch

from helpers import say
from test_gpu_sample import TD, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ties", [1, 2, 511, 513, 1023, 1024, 1025, 4000, 4096, 4097])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_cut_in_ties(gpu, ties, dt):
    say(f"topp ties={ties} dt={dt}")
    B, V = 6, 17011
    rng = np.random.default_rng(ties)
    host = rng.normal(-9, 1, (B, 1, V)).astype(np.float32)
    for b in range(B):
        at = rng.permutation(V)
        host[b, 0, at[:ties]] = 1.0
        host[b, 0, at[ties:ties + 3]] = 1.0 + b  # the mass above the group grows with b (b = 0: three more ties)
    lg = torch.from_numpy(host).to(TD[dt])
    host = lg.float().numpy()
    drafts, n = np.zeros((B, 0), np.int32), np.zeros(B, np.int32)
    for top_p in (0.3, 0.77, 0.999):
        check(lg, host, drafts, n, rng.random(B), 0.9, 0, top_p, f"ties={ties} p={top_p}")


@pytest.mark.parametrize("V", [1, 2, 63, 8191, 8193, 1 << 18])
def test_vocabularies(gpu, V):
    B = 4
    host = np.random.default_rng(V).normal(0, 2.5, (B, 1, V)).astype(np.float32)
    drafts, n = np.zeros((B, 0), np.int32), np.zeros(B, np.int32)
    for top_p in (1e-6, 0.5, 0.95):
        check(torch.from_numpy(host), host, drafts, n, np.linspace(0.05, 0.97, B), 0.8, 0, top_p, f"V={V} p={top_p}")
