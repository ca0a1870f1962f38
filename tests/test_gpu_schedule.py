"""GPU parity of the automatic attention schedule at the edges of its cutting rules: few
items cut into many pieces, items just below and above the shortest piece, one key, mixed
lengths, and more sequences than the plan ranks; against the CPU oracle."""
import numpy as np
import pytest

from helpers import TOL, say
from test_gpu_kv import run_attention_case

pytestmark = pytest.mark.gpu

# (pool, R, Hq, H, contexts): cached keys before the verify rows.
CASES = [
    ("fp8", 5, 4, 1, [3001]),                       # one item, pieces of 12 64-token chunks
    ("fp8", 1, 1, 1, [0]),                          # a single key
    ("bf16", 5, 8, 2, [16 * 32 - 5, 16 * 32 - 4]),  # a full shortest piece, and one key more
    ("fp8", 2, 8, 2, [12 * 64 - 2, 12 * 64 - 1]),
    ("int8", 9, 4, 1, [9000, 40]),                  # three row tiles; many pieces next to one
    ("f16", 3, 8, 8, [700, 16, 2500, 1]),
    ("bf16", 1, 2, 1, [40000]),                     # 79 pieces of one item
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_few_items(gpu, case):
    dt, R, Hq, H, ctx = CASES[case]
    say(f"schedule few items {CASES[case]}")
    err = run_attention_case(dt, len(ctx), R, Hq, H, 128, 16, ctx, src="bf16", q_dt="bf16", seed=40 + case)
    assert err <= TOL[dt]


@pytest.mark.parametrize("long_ctx", [600, 17000])
def test_more_sequences_than_the_plan_ranks(gpu, long_ctx):
    """1100 sequences: one workgroup per item, or stream-K where the longest table row holds
    more than 16384 keys."""
    say(f"schedule 1100 sequences, longest {long_ctx}")
    ctx = [int(x) for x in np.random.default_rng(5).integers(0, 60, 1100)]
    ctx[700] = long_ctx
    err = run_attention_case("bf16", 1100, 1, 1, 1, 128, 16, ctx, src="bf16", q_dt="bf16", seed=9)
    assert err <= TOL["bf16"]
