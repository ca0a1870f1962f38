"""GPU parity of the per-row attention kernel over its variants: V by 16-byte runs or by element
(block size, pool type), every partition of a row in one workgroup or merged by a launch of its
own, one to five 64-dim groups, rows that are no multiple of 16 bytes; against the oracle."""
import pytest

from helpers import TOL, say
from test_gpu_kv import run_attention_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "fp8", "int8"])
@pytest.mark.parametrize("D,bs", [(64, 32), (64, 8), (40, 16), (96, 64), (100, 4), (128, 12), (256, 16), (300, 8)])
def test_variants(gpu, dt, D, bs):
    # Partitions of 64 keys: up to eight per row meet in one workgroup, more in the merge launch.
    for ctx, part in (([0, 70, 500], 64), ([3, 700], 64), ([900, 33], 256), ([90, 10], 0)):
        say(f"per-row dt={dt} D={D} bs={bs} ctx={ctx} partition={part}")
        err = run_attention_case(dt, len(ctx), 2, 4, 2, D, bs, ctx, partition=part, seed=D + bs)
        assert err <= TOL[dt]


def test_ragged_rows(gpu):
    say("per-row ragged")
    err = run_attention_case("f32", 3, 4, 4, 2, 64, 16, [100, 7, 300], row_counts=[4, 1, 2], seed=1)
    assert err <= TOL["f32"]
