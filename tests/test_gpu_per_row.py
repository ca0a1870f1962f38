"""GPU parity of the per-row attention kernel over its variants: V by 16-byte runs or by element
(block size, pool type), every partition of a row in one workgroup or merged by a launch of its
own, one to five 64-dim groups, rows that are no multiple of 16 bytes; against the oracle."""
import pytest
import torch

from gollmgo_amd._lib import lib
from gollmgo_amd.verify import device_bytes
from helpers import TOL, say
from test_gpu_kv import make_cache, run_attention_case

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


@pytest.mark.parametrize("bs", [16, 8])
def test_fp8_codes(gpu, bs):
    """All 256 E4M3 codes, as the V of a sequence's only key, come back exactly (NaN as NaN)."""
    say(f"per-row fp8 codes bs={bs}")
    H, D = 4, 64
    kv = make_cache("fp8", H, D, bs, 1)
    kv.set_head_scales(0, [1.0] * H, [1.0] * H)
    kv.append(0, torch.zeros(1, H, D, device="cuda"), torch.zeros(1, H, D, device="cuda"),
              torch.zeros(1, dtype=torch.int32, device="cuda"))
    codes = torch.arange(256, dtype=torch.uint8)
    v = device_bytes(lib().gg_kv_v_layer_ptr(kv.handle, 0), (2 * H - 1) * bs * D)
    torch.as_strided(v, (H, D), (2 * bs * D, bs)).copy_(codes.view(H, D))
    out = torch.zeros(1, 1, H, D, device="cuda")
    kv.attention(0, torch.ones_like(out), out, torch.ones(1, dtype=torch.int32, device="cuda"),
                 torch.zeros(1, 1, dtype=torch.int32, device="cuda"), 1.0, partition_tokens=64)
    torch.cuda.synchronize()
    assert torch.equal(out.cpu().flatten().nan_to_num(999.0), codes.view(torch.float8_e4m3fn).float().nan_to_num(999.0))
    kv.close()
