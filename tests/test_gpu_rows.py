"""GPU parity of the MFMA attention for head_dim 64 and for more than 64 query rows per kv head
(row groups), against the float64 oracle and against the per-row kernel it took over from
(an explicit partition still runs that one): no less exact, for every pool and query type."""
import math

import pytest
import torch

from gollmgo_amd.workloads import CONFIGS, VerifyConfig
from helpers import TOL, say
from test_gpu_kv import _fused_vs_separate, make_cache, run_attention_case

pytestmark = pytest.mark.gpu

# (B, R, Hq, H, D, contexts): row tiles 1 to 4 at head_dim 64, then groups of rows.
SHAPES = [
    (2, 1, 2, 2, 64, [0, 130]),
    (3, 5, 24, 4, 64, [40, 700, 1500]),        # 30 rows: two tiles
    (2, 3, 32, 2, 64, [33, 5000]),             # 48 rows: three
    (2, 16, 8, 2, 64, [17, 900]),              # 64 rows: four
    (2, 9, 32, 4, 64, [300, 64]),              # 72 rows: two groups of three tiles
    (2, 5, 32, 2, 128, [600, 90]),             # 80 rows: three groups of two tiles
    (1, 65, 4, 1, 128, [2000]),                # 260 rows: nine groups
]


@pytest.mark.parametrize("dt", ["bf16", "f16", "fp8", "int8"])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_no_less_exact_than_the_per_row_kernel(gpu, dt, shape):
    B, R, Hq, H, D, ctx = SHAPES[shape]
    for q_dt in ("bf16", "f16", "f32"):
        say(f"rows dt={dt} q={q_dt} shape={SHAPES[shape]}")
        err = run_attention_case(dt, B, R, Hq, H, D, 16, ctx, src="bf16", q_dt=q_dt, seed=60 + shape)
        ref = run_attention_case(dt, B, R, Hq, H, D, 16, ctx, src="bf16", q_dt=q_dt, seed=60 + shape, partition=64)
        print(f"  rel err {err:.2e}, per-row kernel {ref:.2e}")
        assert err <= TOL[dt]
        # The largest of a few thousand fp32-level errors each; 2e-6 is 16 units of 2^-23.
        assert err <= max(2 * ref, 2e-6), (err, ref)


@pytest.mark.parametrize("dt", ["bf16", "f16", "fp8", "int8"])
def test_mean_error_of_the_per_row_kernel(gpu, monkeypatch, dt):
    """The error's 2-norm over all shapes and query types, which averages over the roundings of some
    hundred thousand outputs: no larger than the per-row kernel's."""
    import test_gpu_kv

    sums = {}

    def norms(got, ref):
        return float(((got.astype("f8") - ref) ** 2).sum() / (ref.astype("f8") ** 2).sum())

    monkeypatch.setattr(test_gpu_kv, "rel_err_per_vector", norms)
    for q_dt in ("bf16", "f16", "f32"):
        say(f"rows mean error dt={dt} q={q_dt}")
        for part in (0, 64):
            sums[part] = sum(run_attention_case(dt, B, R, Hq, H, D, 16, ctx, src="bf16", q_dt=q_dt, seed=90 + i, partition=part)
                             for i, (B, R, Hq, H, D, ctx) in enumerate(SHAPES)) ** 0.5
        print(f"  {sums[0]:.2e}, per-row kernel {sums[64]:.2e}")
        assert sums[0] <= 1.02 * sums[64], (q_dt, sums)  # (two estimates of a rounding error)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("q_sd", [1e-6, 1e6])
def test_queries_far_from_one(gpu, dt, q_sd):
    """Queries are scaled into the f16 operand range by a power of two and back."""
    say(f"rows q_sd={q_sd} dt={dt}")
    for q_dt in ("bf16", "f32"):
        B, R, Hq, H, D, ctx = SHAPES[1]
        err = run_attention_case(dt, B, R, Hq, H, D, 16, ctx, src="bf16", q_dt=q_dt, seed=3, q_sd=q_sd,
                                 kv_sd=3.0 / max(q_sd, 1.0), v_sd=1.0)
        assert err <= TOL[dt]


@pytest.mark.parametrize("dt", ["bf16", "fp8"])
def test_ragged_rows(gpu, dt):
    """Row groups that a short sequence has no rows for write nothing."""
    say(f"rows ragged dt={dt}")
    err = run_attention_case(dt, 3, 6, 64, 4, 128, 16, [300, 1000, 17], row_counts=[6, 1, 3], src="bf16", q_dt="bf16",
                             seed=7)
    assert err <= TOL[dt]


@pytest.mark.parametrize("dt", ["bf16", "f16", "fp8", "int8"])
@pytest.mark.parametrize("Hq,H,D,R,B,ctx", [
    (32, 8, 64, 6, 5, (100, 2500)),    # rows patched from LDS (past the first chunks)
    (32, 8, 64, 6, 5, (0, 40)),        # rows in the first chunks
    (16, 2, 64, 8, 40, (200, 900)),    # four row tiles
    (32, 2, 128, 6, 6, (100, 1500)),   # three row groups of an item append the same rows
])
def test_append_attention_equals_append_then_attention(gpu, monkeypatch, dt, Hq, H, D, R, B, ctx):
    say(f"rows fused append dt={dt} Hq={Hq} H={H} D={D} R={R} ctx={ctx}")
    monkeypatch.setitem(CONFIGS, 99, VerifyConfig("rows", B, R - 1, Hq, H, D, 16, ("uniform", *ctx), dt, "bf16", 1000,
                                                  "f32", "greedy", seed=D + R))
    # (Ragged row counts leave unwritten positions behind the context here, and an int8 block
    # re-quantises whatever bytes they hold.)
    _fused_vs_separate(99, dt, B, ("uniform", *ctx), dt != "int8")
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dt", ["f16", "bf16", "fp8"])
@pytest.mark.parametrize("R", [8, 9, 12, 16])
@pytest.mark.parametrize("Hq,H,D", [(4, 4, 64), (8, 4, 64), (16, 4, 64), (8, 1, 128)])
def test_append_attention_around_the_staged_rows(gpu, monkeypatch, dt, R, Hq, H, D):
    """Draft rows at the number a piece stages in LDS and above it (appended before the piece's
    loads there), for one to four row tiles: rows that start at block offsets 0, 4 and 13, in and
    past the first chunks, all rows or ragged counts; pool bytes and outputs bit for bit."""
    ctx = (40, 320, 324, 333, 896, 900, 909)
    say(f"rows fused append around the staged rows dt={dt} R={R} Hq={Hq} H={H} D={D}")
    monkeypatch.setitem(CONFIGS, 99, VerifyConfig("rows", len(ctx), R - 1, Hq, H, D, 16, ("list", *ctx), dt, "bf16", 1000,
                                                  "f32", "greedy", seed=D + R))
    for rc in (False, True):
        _fused_vs_separate(99, dt, len(ctx), ("list", *ctx), rc)
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dt", ["bf16", "f16", "fp8", "int8"])
@pytest.mark.parametrize("shape", [0, 1, 3, 5, 6, 7])
def test_any_finite_scale(gpu, dt, shape):
    """Softmax scales at and below zero, and so small that the score multiplier underflows:
    masked keys stay masked, a negative scale turns the order of the scores round."""
    B, R, Hq, H, D, ctx = (SHAPES + [(2, 5, 16, 2, 128, [40, 700])])[shape]  # (the last: 40 rows at head_dim 128)
    for scale in (0.0, -0.0, -0.125, 1e-44, -1e-44):
        for q_dt in ("bf16", "f16", "f32"):
            say(f"rows dt={dt} q={q_dt} scale={scale} shape={shape}")
            err = run_attention_case(dt, B, R, Hq, H, D, 16, ctx, src="bf16", q_dt=q_dt, seed=70 + shape, scale=scale)
            assert err <= TOL[dt]


@pytest.mark.parametrize("dt", ["f16", "fp8", "int8"])
@pytest.mark.parametrize("Hq,H,D,R", [(16, 4, 64, 9), (32, 2, 128, 5), (16, 4, 128, 5)])
def test_append_attention_at_a_negative_scale(gpu, monkeypatch, dt, Hq, H, D, R):
    """A planned call at such a scale appends its rows and leaves the plan as it was."""
    ctx = (40, 333, 900)
    say(f"rows fused append at a negative scale dt={dt} Hq={Hq} H={H} D={D} R={R}")
    monkeypatch.setitem(CONFIGS, 99, VerifyConfig("rows", len(ctx), R - 1, Hq, H, D, 16, ("list", *ctx), dt, "bf16", 1000,
                                                  "f32", "greedy", seed=D + R))
    _fused_vs_separate(99, dt, len(ctx), ("list", *ctx), False, scale=-0.125)


@pytest.mark.parametrize("dt", ["bf16", "f16", "fp8", "int8"])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_values_that_are_not_finite(gpu, dt, shape):
    """NaN and infinities in the K and V of draft rows, in the context's V and in a query row reach
    the rows that the per-row kernel lets them reach, and no other; the append inside the call too."""
    B, R, Hq, H, D, ctx = SHAPES[shape]
    bs, inf, nan = 16, float("inf"), float("nan")
    gen = torch.Generator(device="cuda").manual_seed(80 + shape)
    keys = [c + R for c in ctx]
    nbs = [(n + bs - 1) // bs for n in keys]
    bt = torch.zeros(B, max(nbs), dtype=torch.int32)
    slots, first = [], 1
    for b in range(B):
        bt[b, :nbs[b]] = torch.arange(first, first + nbs[b])
        slots += [first * bs + t for t in range(keys[b])]
        first += nbs[b]
    draft = [sum(keys[:b]) + ctx[b] + j for b in range(B) for j in range(R)]
    slots, draft = torch.tensor(slots, dtype=torch.int32).cuda(), torch.tensor(draft).cuda()
    bt, kt = bt.cuda(), torch.tensor(keys, dtype=torch.int32).cuda()
    src = torch.float16 if dt == "f16" else torch.bfloat16
    for case in ("v nan", "v inf", "v both", "k nan", "context v", "q inf"):
        if dt == "int8" and case != "q inf":
            continue  # (a byte holds neither)
        if dt == "fp8" and case not in ("v nan", "k nan", "q inf"):
            continue  # (infinities saturate)
        for q_dt in (torch.bfloat16, torch.float32):
            say(f"rows not finite dt={dt} shape={shape} {case} q={q_dt}")
            kx, vx = (torch.randn(len(slots), H, D, device="cuda", generator=gen).to(src) for _ in range(2))
            q = torch.randn(B, R, Hq, D, device="cuda", generator=gen).to(q_dt)
            last = draft[R - 1::R]  # (each sequence's last row)
            if case in ("v nan", "v both"):
                vx[last, :, 3] = nan
            if case in ("v inf", "v both"):
                vx[draft[R // 2::R], 0, 5:7] = inf
                vx[last, -1, 5] = -inf
            if case == "k nan":
                kx[last, -1, 7] = nan
            if case == "context v":
                vx[draft[0::R] // 2, 0, 9] = inf
            if case == "q inf":
                q, kx = q * 1e5, kx * 1e-5
                q[:, R // 2, Hq // 2, 1] = inf
            outs = []
            for mode in ("per-row", "separate", "fused"):
                kv = make_cache(dt, H, D, bs, first)
                if dt == "fp8":
                    kv.set_head_scales(0, [1e-7 if case == "q inf" else 0.01] * H, [0.01] * H)
                context = torch.ones(len(slots), dtype=torch.bool, device="cuda")
                context[draft] = False
                for rows in (context, ~context)[:1 if mode == "fused" else 2]:
                    if rows.any():
                        kv.append(0, kx[rows].contiguous(), vx[rows].contiguous(), slots[rows].contiguous())
                out = torch.zeros(B, R, Hq, D, device="cuda")
                if mode == "per-row":
                    kv.attention(0, q, out, kt, bt, D ** -0.5, partition_tokens=64)
                else:
                    ws = kv.attention_workspace(B, R, Hq, bt.shape[1], 0)
                    kv.attention_plan(kt, R, Hq, bt.shape[1], ws)
                    if mode == "fused":
                        new = [x[draft].contiguous() for x in (kx, vx)]
                        kv.append_attention(0, *new, q, out, kt, bt, D ** -0.5, ws)
                    else:
                        kv.attention(0, q, out, kt, bt, D ** -0.5, workspace=ws, planned=True)
                torch.cuda.synchronize()
                outs.append(out.cpu())
                kv.close()
            ref = outs[0]
            assert case == "v nan" or ref.isfinite().any(), case
            for got in outs[1:]:
                for f in (torch.isnan, torch.isposinf, torch.isneginf):
                    assert torch.equal(f(got), f(ref)), (case, f)
                fin = ref.isfinite()
                # (Outputs below 5, each side within 2e-6 of its largest.)
                assert (got[fin] - ref[fin]).abs().max() <= 2e-5, case
