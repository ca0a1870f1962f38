"""GPU parity of the append by block runs (large calls; INT8 at every size), bit for bit against
the oracle mirror: prompts that start inside a block, head_dims below the largest, runs of
skipped rows longer than the kernel's slot window, rows in no order."""
import numpy as np
import pytest
import torch

from helpers import PoolMirror, append_rows, say
from test_gpu_kv import make_cache

pytestmark = pytest.mark.gpu


def check(dt, src, H, D, calls, nb, seed):
    rng = np.random.default_rng(seed)
    kv = make_cache(dt, H, D, 16, nb)
    mirror = PoolMirror(kv)
    if dt == "fp8":
        sc = rng.uniform(0.005, 0.05, H).astype(np.float32)
        kv.set_head_scales(0, sc, sc)
        mirror.set_head_scales(sc, sc)
    # Every byte written first, so that the whole pools compare.
    calls = [np.arange(nb * 16)] + calls
    for i, slots in enumerate(calls):
        slots = np.asarray(slots, np.int32)
        k = rng.normal(0, 1 + i, (len(slots), H, D)).astype(np.float32)
        v = rng.normal(0, 1 + i, (len(slots), H, D)).astype(np.float32)
        append_rows(kv, mirror, k, v, slots, src)
        mirror.compare_with_device()
    kv.close()


def prompt(order, first, n):
    p = first + np.arange(n)
    return order[p // 16] * 16 + p % 16


@pytest.mark.parametrize("dt", ["fp8", "bf16", "f16", "int8"])
@pytest.mark.parametrize("src,D,first", [("bf16", 128, 0), ("f32", 64, 5), ("f16", 96, 15), ("bf16", 8, 1)])
def test_prompt(gpu, dt, src, D, first):
    say(f"append runs prompt dt={dt} src={src} D={D} first={first}")
    order = np.random.default_rng(D).permutation(90)
    check(dt, src, 2, D, [prompt(order, first, 1100), prompt(order, first + 1100, 17)], 90, D + first)


@pytest.mark.parametrize("dt", ["fp8", "int8"])
@pytest.mark.parametrize("n", [40, 1200])
def test_skipped_rows_around_runs(gpu, dt, n):
    """Skipped rows inside a run, before one and after one, in streaks that fill the slot
    window (a run's other rows, or the row before it, then lie outside it)."""
    say(f"append runs skipped rows dt={dt} n={n}")
    order = np.random.default_rng(n).permutation(90)
    slots = list(prompt(order, 3, n))
    for at, streak in ((n - 3, 70), (20, 90), (9, 1), (0, 33)):
        slots[at:at] = [-1] * streak
    check(dt, "bf16", 2, 64, [slots], 90, n)


@pytest.mark.parametrize("dt", ["fp8", "f16"])
def test_rows_in_no_order(gpu, dt):
    say(f"append runs shuffled dt={dt}")
    slots = np.random.default_rng(4).permutation(90 * 16)[:1300]
    check(dt, "bf16", 2, 128, [slots], 90, 8)


@pytest.mark.parametrize("dt", ["fp8", "bf16", "int8"])
@pytest.mark.parametrize("gaps", [(0, 1), (0, 1, 2), (1, 2, 3), (2,), (15, 31, 32, 47), (0, 0, 63, 64, 255, 256, 257)])
def test_skipped_rows_inside_runs(gpu, dt, gaps):
    """Gaps around the number of skipped rows that ends a run, at every place of a block, and runs
    as long as they get."""
    say(f"append runs gaps dt={dt} gaps={gaps}")
    rng = np.random.default_rng(len(gaps))
    order = rng.permutation(90)
    slots = []
    for slot in prompt(order, 7, 1100):
        slots += [slot] + [-1] * rng.choice(gaps)
    check(dt, "bf16", 8, 64, [slots], 90, 5)


@pytest.mark.parametrize("dt", ["fp8", "bf16", "f16", "int8"])
@pytest.mark.parametrize("src,H,D", [("bf16", 8, 128), ("f32", 9, 64), ("f16", 8, 96), ("bf16", 12, 8)])
def test_runs_of_any_length(gpu, dt, src, H, D):
    """Enough rows and heads for block runs in every pool: a prompt, verify rows of many sequences
    (one to sixteen rows that start anywhere in a block and may cross into the next), rows in no
    order, and short runs next to long ones, with skipped rows between."""
    say(f"append runs any length dt={dt} src={src} H={H} D={D}")
    rng = np.random.default_rng(H * D)
    order = rng.permutation(180)

    def sequences(lengths):
        slots, blk = [], 0
        for n in lengths:
            first = rng.integers(0, 16)
            if blk * 16 + first + n > 180 * 16:
                break
            slots += list(prompt(order, blk * 16 + first, n))
            blk += (first + n + 15) // 16
        return slots

    one = [prompt(order, 16 * i + 3, 1)[0] for i in range(180)]
    mixed = []
    for slot in sequences(rng.choice([1, 2, 3, 5, 9, 16, 17, 40], 200)):
        mixed += [slot] + [-1] * int(rng.choice([0, 0, 0, 0, 1, 5]))
    calls = [prompt(order, 5, 1200), sequences([5] * 180), one, mixed]
    if dt != "int8":  # (a block's scale follows its runs one after the other)
        calls.append(rng.permutation(180 * 16)[:1300])
    # (Calls below the limit are filled up with skipped rows.)
    check(dt, src, H, D, [list(c) + [-1] * max(0, 1100 - len(c)) for c in calls], 180, D)


@pytest.mark.parametrize("dt", ["fp8", "bf16", "int8"])
@pytest.mark.parametrize("first", [0, 8092])
def test_skipped_rows_cost_no_more_than_written_ones(gpu, dt, first):
    """A hundred rows of a prompt padded to 8192, before or after the skipped ones, against 8192
    rows (walked row by row, the skipped ones took ninety times as long as these)."""
    H, D, n = 8, 128, 8192
    say(f"append runs padded dt={dt} first={first}")
    kv = make_cache(dt, H, D, 16, n // 16)
    if dt == "fp8":
        kv.set_head_scales(0, [0.01] * H, [0.01] * H)
    k = torch.randn(n, H, D, device="cuda", dtype=torch.bfloat16)
    full = torch.arange(n, dtype=torch.int32, device="cuda")
    padded = torch.full_like(full, -1)
    padded[first:first + 100] = full[:100]
    times = []
    for slots in (full, padded):
        kv.append(0, k, k, slots)
        best = float("inf")
        for _ in range(5):  # (the best of five: a host that stalls once does not count)
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(20):
                kv.append(0, k, k, slots)
            end.record()
            torch.cuda.synchronize()
            best = min(best, start.elapsed_time(end) / 20 * 1e3)
        times.append(best)
    kv.close()
    print(f"  full {times[0]:.1f} us, padded {times[1]:.1f} us")
    assert times[1] < 4 * times[0]  # (launches and host noise included)
