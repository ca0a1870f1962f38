"""GPU parity of the nucleus draw at the sizes where its ranking changes path, bit for bit
against the oracle: the cut inside a group of equal logits ranked by pairs (up to 1024), by the
radix descent, or past the gathered list (the literal rule)."""
import numpy as np
import pytest
import torch

import gollmgo_amd.verify as gv
from helpers import say
from oracle import oracle as ora
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


@pytest.mark.parametrize("top_p", [1e-3, 0.5, 0.9, 0.999999, float(np.nextafter(np.float32(1), np.float32(0)))])
@pytest.mark.parametrize("T", [0.8, 40.0, 3e-6, 2e-8])
def test_rejection_bins_of_the_boundary(gpu, T, top_p):
    """The histogram's bins: few (small top_p), all (top_p next to 1), all because the bin
    numbers are past the grid's exact range (small T); rows flat, steep, in levels, with one
    segment's maximum far above or below the others."""
    say(f"rejection bins T={T} top_p={top_p}")
    B, K, V = 6, 3, 40009
    rng = np.random.default_rng(int(T * 100) + int(top_p * 1000))
    host = rng.normal(0, 2, (B, K + 1, V)).astype(np.float32)
    host[1, :, 8192:16384] += 11.0
    host[2, :, 8192:16384] -= 30.0
    host[3] *= 0.05
    host[4] = np.round(host[4] * 2) / 2
    host[5, :, ::5000] += 25.0
    if T < 1e-4:
        host = (3.0 + host * T).astype(np.float32)  # neighbouring floats, some bins apart
    drafts = np.argsort(-host[:, :K], axis=-1, kind="stable")[:, :, :200]
    drafts = np.take_along_axis(drafts, rng.integers(0, 200, (B, K, 1)) // rng.integers(1, 200, (B, K, 1)), -1)[..., 0]
    drafts = np.ascontiguousarray(drafts.astype(np.int32))
    n = np.full(B, K, np.int32)
    u = (rng.random((B, K + 1)) * 0.05).astype(np.float32)
    acc, tok = gv.accept_rejection(torch.from_numpy(host).cuda(), torch.from_numpy(drafts).cuda(),
                                   torch.from_numpy(n).cuda(), torch.from_numpy(u).cuda(), T, top_p)
    torch.cuda.synchronize()
    ea, et = ora.accept_rejection(host, drafts, n, u, T, top_p, None)
    assert np.array_equal(acc.cpu().numpy(), ea) and np.array_equal(tok.cpu().numpy(), et), (acc, ea, tok, et)
