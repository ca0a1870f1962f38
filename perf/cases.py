"""Performance cases of the speculative-decoding verify path.

Each case is one call (or one short sequence of calls) that a serving loop makes on every
decode step, through the entry points of gollmgo_amd.verify:

  attention   the attention plan of a step, then per layer the draft rows' KV append and the
              paged multi-query attention (attention_plan, append_attention)
  greedy      greedy acceptance over full-vocabulary logits (accept_greedy)
  sample      the same with the bonus token sampled (accept_greedy_sample)
  rejection   rejection-sampling acceptance (accept_rejection)
  prompt      the KV rows of a prompt (or a chunk of one) written to the pool (append)
  step        a whole small step: draft lookup, plan, layers, greedy acceptance

listed() names the standing cases, draw() samples the same ranges. The context lengths and
draft counts of a case follow from the case alone, so its work is a fixed number; block
placement and all values come from the seed.
"""
import math

import numpy as np
import torch

import gollmgo_amd.verify as gv
from gollmgo_amd._lib import DType, lib
from gollmgo_amd.workloads import VerifyConfig, make_histories

POOLS = {"f32": DType.F32, "f16": DType.F16, "bf16": DType.BF16, "fp8": DType.FP8_E4M3, "int8": DType.INT8}
POOL_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1, "int8": 1}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BLOCK = 16


def attention(pool, seqs, drafts, q_heads, kv_heads, dim, lo, hi, layers, io="bf16", shared=0.0, ragged=False):
    return {"kind": "attention", "pool": pool, "io": io, "seqs": seqs, "drafts": drafts, "q_heads": q_heads,
            "kv_heads": kv_heads, "dim": dim, "ctx_lo": lo, "ctx_hi": hi, "layers": layers, "shared": shared,
            "ragged": ragged}


def accept(kind, dtype, seqs, drafts, vocab, temperature=0.0, top_k=0, top_p=1.0, probs=False, ragged=False):
    return {"kind": kind, "dtype": dtype, "seqs": seqs, "drafts": drafts, "vocab": vocab,
            "temperature": temperature, "top_k": top_k, "top_p": top_p, "probs": probs, "ragged": ragged}


def prompt(pool, rows, kv_heads, dim, layers, first=0):
    return {"kind": "prompt", "pool": pool, "rows": rows, "kv_heads": kv_heads, "dim": dim, "layers": layers,
            "first": first}


def step(pool, seqs, drafts, q_heads, kv_heads, dim, lo, hi, layers, vocab, dtype, history, io):
    c = attention(pool, seqs, drafts, q_heads, kv_heads, dim, lo, hi, layers, io)
    c.update(kind="step", vocab=vocab, dtype=dtype, history=history)
    return c


def listed():
    named = {
        # The whole step of the smallest configuration (4 sequences, fp32 pool, head_dim 64):
        # nothing but launches and latency.
        "step-tiny-f32": step("f32", 4, 4, 8, 2, 64, 64, 256, 1, 32000, "f32", 256, "f32"),
        # One user chatting: a single sequence, a layer after another.
        "attn-single-fp8": attention("fp8", 1, 4, 32, 8, 128, 3001, 3001, 16, ragged=True),
        # The 3B-shaped bf16 configuration: 32 sequences, one row tile per kv head.
        "attn-3b-bf16": attention("bf16", 32, 4, 24, 8, 128, 512, 4096, 2),
        # The 8B-shaped fp8 configuration, the framework's headline: 64 sequences, a fifth of
        # the prefix blocks shared by pairs of sequences.
        "attn-8b-fp8": attention("fp8", 64, 5, 32, 8, 128, 1024, 8192, 2, shared=0.2),
        # Long documents: 8 sequences of 16k to 32k keys in an int8 pool.
        "attn-long-int8": attention("int8", 8, 8, 32, 8, 128, 16384, 32768, 1),
        # A small model with head_dim 64 in an f16 pool, drafts of uneven length.
        "attn-dim64-f16": attention("f16", 16, 4, 32, 8, 64, 512, 4096, 2, io="f16", ragged=True),
        # Many query heads on few kv heads: 80 query rows share each K/V head.
        "attn-wide-bf16": attention("bf16", 16, 4, 32, 2, 128, 512, 4096, 2),
        # Greedy acceptance of the 3B configuration's logits.
        "greedy-bf16": accept("greedy", "bf16", 32, 4, 128256),
        # Greedy drafts with the bonus token sampled at the engine's temperature, top-k, top-p.
        "sample-bf16": accept("sample", "bf16", 32, 4, 128256, 0.8, 50, 0.95, ragged=True),
        # Rejection sampling against a draft model's distributions (8B configuration).
        "reject-probs-f32": accept("rejection", "f32", 64, 5, 128256, 0.8, probs=True),
        # Rejection sampling of n-gram drafts with a nucleus (mixed configuration).
        "reject-topp-f32": accept("rejection", "f32", 128, 5, 128256, 0.8, top_p=0.95),
        # A prompt's KV written by one prefill chunk, quantised on the way.
        "prompt-fp8": prompt("fp8", 8192, 8, 128, 4),
    }
    return [dict(c, name=n) for n, c in named.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention"] * 5 + ["greedy", "sample", "rejection", "rejection", "prompt", "step"])
    pool = rng.choice(["bf16", "bf16", "f16", "fp8", "fp8", "int8"])
    if kind == "attention":
        q_heads, kv_heads = rng.choice([(32, 8), (32, 8), (24, 8), (8, 8), (16, 8), (8, 2), (32, 2), (64, 8)])
        dim = rng.choice([128, 128, 64])
        drafts = rng.randint(0, 8)
        wide = dim != 128 or q_heads // kv_heads * (drafts + 1) > 64
        seqs = _log_int(rng, 1, 24 if wide else 128)
        # No more keys than the largest listed case of the kind reads.
        most = (75e6 if wide else 550e6) / (2 * kv_heads * dim * POOL_BYTES[pool] * seqs)
        hi = _log_int(rng, 128, max(160, min(32768 if not wide else 8192, most)))
        lo = max(1, int(hi * rng.choice([1.0, 0.5, 0.125])))
        return attention(pool, seqs, drafts, q_heads, kv_heads, dim, lo, hi, rng.randint(1, 2),
                         io=rng.choice(["bf16", "bf16", "f16"]), shared=rng.choice([0.0, 0.0, 0.2]),
                         ragged=rng.random() < 0.5)
    if kind == "prompt":
        kv_heads = rng.choice([2, 8])
        return prompt(pool, _log_int(rng, 16, 8192), kv_heads, rng.choice([64, 128, 128]), rng.randint(1, 4),
                      rng.choice([0, 0, rng.randint(1, 15)]))
    if kind == "step":
        f32 = rng.random() < 0.4
        q_heads, kv_heads, dim = rng.choice([(8, 2, 64), (24, 8, 128), (32, 8, 128)])
        hi = _log_int(rng, 64, 1024)
        return step("f32" if f32 else pool, _log_int(rng, 1, 16), rng.randint(1, 6), q_heads, kv_heads, dim,
                    max(1, hi // 4), hi, rng.randint(1, 4), rng.choice([32000, 50001, 128256]),
                    "f32" if f32 else "bf16", _log_int(rng, 256, 8192), "f32" if f32 else "bf16")
    dtype = rng.choice(["bf16", "f32", "f16"])
    vocab = rng.choice([32000, 50001, 128256, 128256, 160000])
    drafts = rng.randint(1, 8)
    seqs = _log_int(rng, 1, min(128, int(98.5e6 / ((drafts + 1) * vocab))))
    ragged = rng.random() < 0.5
    if kind == "greedy":
        return accept(kind, dtype, seqs, drafts, vocab, ragged=ragged)
    if kind == "sample":
        return accept(kind, dtype, seqs, drafts, vocab, rng.choice([0.6, 0.8, 1.0]), rng.choice([0, 40, 50]),
                      rng.choice([0.9, 0.95, 1.0]), ragged=ragged)
    probs = rng.random() < 0.5
    return accept(kind, dtype, max(1, seqs // 2) if probs else seqs, drafts, vocab, rng.choice([0.6, 0.8, 1.0]),
                  top_p=rng.choice([0.9, 0.95, 1.0]), probs=probs, ragged=ragged)


# ---- what follows from the case alone

def _contexts(c):
    r = np.random.default_rng([c["seqs"], c["ctx_lo"], c["ctx_hi"]])
    return r.integers(c["ctx_lo"], c["ctx_hi"] + 1, c["seqs"]).astype(np.int64)


def _row_counts(c):
    """Verify rows per sequence: 1 + its drafts (the drafter may find fewer than asked for)."""
    R = c["drafts"] + 1
    if not c["ragged"]:
        return np.full(c["seqs"], R, np.int64)
    r = np.random.default_rng([c["seqs"], R, 17])
    n = r.integers(1, R + 1, c["seqs"])
    return np.where(r.random(c["seqs"]) < 0.6, R, n).astype(np.int64)


def _shared_blocks(c, ctx):
    """Blocks at the front of sequence 2i + 1 that are sequence 2i's."""
    n = np.zeros(c["seqs"], np.int64)
    if c["shared"]:
        for i in range(0, c["seqs"] - 1, 2):
            n[i + 1] = int(c["shared"] * min(ctx[i], ctx[i + 1])) // BLOCK
    return n


def _layout(c, seed):
    """(ctx, rows, keys, block tables, pool blocks): blocks in random order over the pool."""
    ctx, rows = _contexts(c), _row_counts(c)
    keys = ctx + rows
    need = (keys + BLOCK - 1) // BLOCK
    shared = _shared_blocks(c, ctx)
    total = int((need - shared).sum())
    order = np.random.default_rng([seed, 1]).permutation(total).astype(np.int32)
    tables = np.zeros((c["seqs"], int(need.max())), np.int32)
    at = 0
    for b in range(c["seqs"]):
        s = int(shared[b])
        if s:
            tables[b, :s] = tables[b - 1, :s]
        n = int(need[b]) - s
        tables[b, s:s + n] = order[at:at + n]
        at += n
    return ctx, rows, keys, tables, total


# ---- values

def _gen(seed, *more):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(np.random.SeedSequence([seed, *more]).generate_state(1, np.uint64)[0] >> 1))
    return g


def _src(c):
    return torch.float32 if c.get("io") == "f32" else torch.bfloat16


def _rows(c, seed, layer, n, what):
    """K and V of n tokens of one layer, as the model's projections give them."""
    g = _gen(seed, layer, what)
    shape = (n, c["kv_heads"], c["dim"])
    return (torch.randn(shape, device="cuda", dtype=_src(c), generator=g),
            torch.randn(shape, device="cuda", dtype=_src(c), generator=g))


def _head_scales(x):
    return [float(v) for v in (x.float().abs().amax(dim=(0, 2)) / 448.0).clamp_min(1e-8).cpu()]


class _PoolBytes:
    """Device memory of a KVCache as torch sees it. A tensor made from this object keeps it,
    and with it the cache whose memory it names."""

    def __init__(self, kv, ptr, nbytes):
        self.kv = kv
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 3,
                                         "strides": None}


def _pool_view(kv, layer):
    """A layer's K and V tiles, as bytes."""
    return torch.as_tensor(_PoolBytes(kv, lib().gg_kv_k_layer_ptr(kv.handle, layer), 2 * kv.layer_bytes), device="cuda")


def _block_scales(kv, layer):
    """An int8 layer's fp16 block scales of K and of V, as bytes."""
    n = kv.num_blocks * kv.num_kv_heads * 2
    return [torch.as_tensor(_PoolBytes(kv, ptr(kv.handle, layer), n), device="cuda")
            for ptr in (lib().gg_kv_k_scale_ptr, lib().gg_kv_v_scale_ptr)]


def _filled_pool(c, seed, blocks):
    """A pool with every slot written, as after the prompts of all its sequences."""
    kv = gv.KVCache(c["layers"], blocks, BLOCK, c["kv_heads"], c["dim"], POOLS[c["pool"]])
    slots = torch.arange(blocks * BLOCK, dtype=torch.int32, device="cuda")
    for layer in range(c["layers"]):
        k, v = _rows(c, seed, layer, blocks * BLOCK, 0)
        if c["pool"] == "fp8":
            kv.set_head_scales(layer, _head_scales(k), _head_scales(v))
        kv.append(layer, k, v, slots)
    return kv


def _queries(c, seed):
    g = _gen(seed, 2)
    shape = (c["seqs"], c["drafts"] + 1, c["q_heads"], c["dim"])
    return [torch.randn(shape, device="cuda", dtype=TORCH[c["io"]], generator=g) for _ in range(c["layers"])]


def _prepare_attention(c, seed):
    _, rows, keys, tables, blocks = _layout(c, seed)
    kv = _filled_pool(c, seed, blocks)
    B, R = c["seqs"], c["drafts"] + 1
    q = _queries(c, seed)
    new = [_rows(c, seed, layer, B * R, 3) for layer in range(c["layers"])]
    s = {"kv": kv, "q": q, "out": [torch.zeros_like(x) for x in q], "new": new, "layers": c["layers"], "R": R,
         "Hq": c["q_heads"], "keys": torch.from_numpy(keys.astype(np.int32)).cuda(),
         "tables": torch.from_numpy(tables).cuda(),
         "rows": torch.from_numpy(rows.astype(np.int32)).cuda() if c["ragged"] else None,
         "scale": 1.0 / math.sqrt(c["dim"]), "pool": [_pool_view(kv, layer) for layer in range(c["layers"])]}
    s["ws"] = kv.attention_workspace(B, R, c["q_heads"], tables.shape[1])
    return s


def _logits(c, seed):
    """Next-token logits: a broad floor, and in every row a few candidates above it, from a
    near tie to a sure token."""
    g = _gen(seed, 4)
    B, R, V = c["seqs"], c["drafts"] + 1, c["vocab"]
    x = torch.randn(B, R, V, device="cuda", generator=g) * 2.0
    at = torch.randint(0, V, (B, R, 32), device="cuda", generator=g)
    height = torch.rand(B, R, 1, device="cuda", generator=g) * 12.0 + 4.0
    x.scatter_add_(2, at, torch.rand(B, R, 32, device="cuda", generator=g) * height)
    return x.to(TORCH[c["dtype"]])


def _prepare_accept(c, seed):
    B, K, V = c["seqs"], c["drafts"], c["vocab"]
    logits = _logits(c, seed)
    g = _gen(seed, 5)
    s = {"logits": logits, "n": torch.from_numpy((_row_counts(c) - 1).astype(np.int32)).cuda()}
    probs = torch.softmax(logits[:, :K].float() * 1.5, dim=-1).contiguous() if c.get("probs") else None
    mode = logits[:, :K].float().argmax(dim=-1).to(torch.int32)
    other = torch.randint(0, V, (B, K), device="cuda", dtype=torch.int32, generator=g)
    hit = 0.95 if c["kind"] == "sample" else 0.8
    s["drafts"] = torch.where(torch.rand(B, K, device="cuda", generator=g) < hit, mode, other).contiguous()
    s["probs"] = probs
    s["out"] = (torch.zeros(B, dtype=torch.int32, device="cuda"), torch.zeros(B, dtype=torch.int32, device="cuda"))
    if c["kind"] == "rejection":
        s["u"] = torch.rand(B, K + 1, device="cuda", generator=g)
        s["ws"] = gv.rejection_workspace(B, K, V)
    elif c["kind"] == "sample":
        s["u"] = torch.rand(B, device="cuda", dtype=torch.float64, generator=g)
        s["ws"] = gv.sample_workspace(B, K, V)
    else:
        s["ws"] = gv.greedy_workspace(B, K, V)
    return s


def _prompt_slots(c, seed):
    """Slots of a prompt chunk that starts at offset `first` of its first block."""
    blocks = (c["first"] + c["rows"] + BLOCK - 1) // BLOCK
    order = np.random.default_rng([seed, 6]).permutation(blocks)
    p = c["first"] + np.arange(c["rows"])
    return (order[p // BLOCK] * BLOCK + p % BLOCK).astype(np.int32), blocks


def _prepare_prompt(c, seed):
    slots, blocks = _prompt_slots(c, seed)
    kv = _filled_pool(c, seed, blocks)
    s = {"kv": kv, "slots": torch.from_numpy(slots).cuda(),
         "new": [_rows(c, seed, layer, c["rows"], 3) for layer in range(c["layers"])],
         "pool": [_pool_view(kv, layer) for layer in range(c["layers"])]}
    s["scales"] = [x for layer in range(c["layers"]) for x in _block_scales(kv, layer)] if c["pool"] == "int8" else []
    return s


def _prepare_step(c, seed):
    s = _prepare_attention(c, seed)
    s["accept"] = _prepare_accept(c, seed)
    cfg = VerifyConfig("", c["seqs"], c["drafts"], c["q_heads"], c["kv_heads"], c["dim"], BLOCK, (), c["pool"],
                       c["io"], c["vocab"], c["dtype"], "greedy", repeat_rate=0.3)
    s["history"] = torch.from_numpy(make_histories(cfg, c["history"], seed % (1 << 31))).cuda()
    s["history_len"] = torch.full((c["seqs"],), c["history"], dtype=torch.int32, device="cuda")
    s["next"] = (torch.zeros(c["seqs"], c["drafts"], dtype=torch.int32, device="cuda"),
                 torch.zeros(c["seqs"], dtype=torch.int32, device="cuda"))
    s["K"] = c["drafts"]
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attention":
        s = _prepare_attention(case, seed)
    elif kind == "prompt":
        s = _prepare_prompt(case, seed)
    elif kind == "step":
        s = _prepare_step(case, seed)
    else:
        s = _prepare_accept(case, seed)
    s["kind"] = kind
    s["options"] = (case.get("temperature", 0.0), case.get("top_k", 0), case.get("top_p", 1.0))
    return s


# ---- one pass

def _run_attention(s):
    kv = s["kv"]
    kv.attention_plan(s["keys"], s["R"], s["Hq"], s["tables"].shape[1], s["ws"], row_counts=s["rows"])
    for layer in range(s["layers"]):
        k, v = s["new"][layer]
        kv.append_attention(layer, k, v, s["q"][layer], s["out"][layer], s["keys"], s["tables"], s["scale"],
                            s["ws"], row_counts=s["rows"])
    return {"out": s["out"], "pool": s["pool"]}


def run(s):
    kind = s["kind"]
    if kind == "attention":
        return _run_attention(s)
    if kind == "prompt":
        for layer, (k, v) in enumerate(s["new"]):
            s["kv"].append(layer, k, v, s["slots"])
        return {"pool": s["pool"], "scales": s["scales"]}
    if kind == "step":
        gv.ngram_draft(s["history"], s["history_len"], 3, s["K"], out=s["next"])
        got = _run_attention(s)
        a = s["accept"]
        gv.accept_greedy(a["logits"], a["drafts"], a["n"], workspace=a["ws"], out=a["out"])
        return dict(got, accepted=a["out"][0], token=a["out"][1], next=s["next"][0], next_n=s["next"][1])
    temperature, top_k, top_p = s["options"]
    if kind == "greedy":
        acc, tok = gv.accept_greedy(s["logits"], s["drafts"], s["n"], workspace=s["ws"], out=s["out"])
    elif kind == "sample":
        acc, tok = gv.accept_greedy_sample(s["logits"], s["drafts"], s["n"], s["u"], temperature, top_k, top_p,
                                           workspace=s["ws"], out=s["out"])
    else:
        acc, tok = gv.accept_rejection(s["logits"], s["drafts"], s["n"], s["u"], temperature, top_p,
                                       draft_probs=s["probs"], workspace=s["ws"], out=s["out"])
    return {"accepted": acc, "token": tok}


# ---- what a pass cannot do without

def _attention_work(c):
    ctx, rows = _contexts(c), _row_counts(c)
    keys = ctx + rows
    unique = int((keys - _shared_blocks(c, ctx) * BLOCK).sum())
    eb, io = POOL_BYTES[c["pool"]], 4 if c["io"] == "f32" else 2
    src = 4 if _src(c) == torch.float32 else 2
    n = int(rows.sum())
    per_layer = (unique * 2 * c["kv_heads"] * c["dim"] * eb + 2 * n * c["q_heads"] * c["dim"] * io
                 + n * 2 * c["kv_heads"] * c["dim"] * (src + eb))
    if c["pool"] == "int8":
        per_layer += unique // BLOCK * 2 * c["kv_heads"] * 2
    flops = int((4 * keys * rows).sum()) * c["q_heads"] * c["dim"]
    return {"bytes": c["layers"] * per_layer, "flops": c["layers"] * flops}


def _accept_work(c):
    rows = int(_row_counts(c).sum())
    eb = 4 if c["dtype"] == "f32" else 2
    b = rows * c["vocab"] * eb
    if c.get("probs"):
        b += (rows - c["seqs"]) * c["vocab"] * 4
    return {"bytes": b, "flops": rows * c["vocab"] * (1 if c["kind"] in ("greedy", "step") else 8)}


def work(case):
    kind = case["kind"]
    if kind == "attention":
        return _attention_work(case)
    if kind == "prompt":
        per = 2 * case["kv_heads"] * case["dim"]
        n = case["layers"] * case["rows"] * per
        return {"bytes": n * (2 + POOL_BYTES[case["pool"]]), "flops": 2 * n}
    if kind == "step":
        a, b = _attention_work(case), _accept_work(case)
        h = case["seqs"] * case["history"] * 4
        return {"bytes": a["bytes"] + b["bytes"] + h, "flops": a["flops"] + b["flops"]}
    return _accept_work(case)


def tolerance(case):
    # Decisions, tokens and pool bytes are whole numbers and stay the same. Attention: the
    # rounding of the output type (bf16 2^-9, f16 2^-12) and, in f32, sums in another order.
    if case["kind"] not in ("attention", "step"):
        return "exact"
    return {"rel": {"bf16": 4e-3, "f16": 1e-3, "f32": 5e-6}[case["io"]]}


# ---- the same in 64 bits, with torch alone

def _int8(x, scale):
    inv = torch.where(scale > 0, 1.0 / scale, torch.zeros_like(scale))
    return torch.round(x * inv).clamp(-127, 127)


def _exact_pool(c, x, new, rows, keys, tables):
    """[blocks, BLOCK, H, D] float64 values of one layer's K (or V) pool after the append of
    the verify rows `new` [B, R, H, D], from the fill x [blocks * BLOCK, H, D]."""
    H, D = c["kv_heads"], c["dim"]
    x = x.float().view(-1, BLOCK, H, D)
    pool = c["pool"]
    if pool == "int8":
        scale = (x.abs().amax(dim=(1, 3), keepdim=True) / 127.0).half().float()  # [blocks, 1, H, 1]
        q = _int8(x, scale)
    elif pool == "fp8":
        sc = torch.tensor(_head_scales(x.view(-1, H, D)), dtype=torch.float32, device=x.device).view(1, 1, H, 1)
        enc = lambda t: (t * (1.0 / sc)).clamp(-448, 448).to(torch.float8_e4m3fn).float()  # noqa: E731
        q = enc(x)
    else:
        enc = lambda t: t.to(TORCH[pool]).float()  # noqa: E731
        q = enc(x)
    for b in range(c["seqs"]):
        n, first = int(rows[b]), int(keys[b] - rows[b])
        j = 0
        while j < n:
            off = (first + j) % BLOCK
            m = min(n - j, BLOCK - off)
            blk = int(tables[b, (first + j) // BLOCK])
            r = new[b, j:j + m].float()  # [m, H, D]
            if pool == "int8":
                old = scale[blk] if off else torch.zeros_like(scale[blk])  # [1, H, 1]
                now = torch.maximum(old, (r.abs().amax(dim=(0, 2)).view(1, H, 1) / 127.0).half().float())
                grown = _int8(q[blk, :off] * old, now)
                q[blk, :off] = torch.where(now != old, grown, q[blk, :off])
                q[blk, off:off + m] = _int8(r, now)
                scale[blk] = now
            else:
                q[blk, off:off + m] = enc(r.unsqueeze(0))[0]
            j += m
    if pool == "int8":
        return q.double() * scale.double()
    return q.double() * sc.double() if pool == "fp8" else q.double()


def _exact_attention(c, seed):
    _, rows, keys, tables, blocks = _layout(c, seed)
    B, R, H, D = c["seqs"], c["drafts"] + 1, c["kv_heads"], c["dim"]
    G = c["q_heads"] // H
    outs = []
    for layer, q in enumerate(_queries(c, seed)):
        kx, vx = _rows(c, seed, layer, blocks * BLOCK, 0)
        kn, vn = (t.view(B, R, H, D) for t in _rows(c, seed, layer, B * R, 3))
        kp, vp = _exact_pool(c, kx, kn, rows, keys, tables), _exact_pool(c, vx, vn, rows, keys, tables)
        out = torch.zeros(B, R, c["q_heads"], D, dtype=torch.float64, device="cuda")
        for b in range(B):
            n, L = int(rows[b]), int(keys[b])
            t = torch.from_numpy(tables[b, :(L + BLOCK - 1) // BLOCK].astype(np.int64)).cuda()
            k = kp[t].reshape(-1, H, D)[:L].permute(1, 2, 0).contiguous()  # [H, D, L]
            v = vp[t].reshape(-1, H, D)[:L].permute(1, 0, 2).contiguous()  # [H, L, D]
            qb = q[b, :n].double().view(n, H, G, D).permute(1, 0, 2, 3).reshape(H, n * G, D)
            s = torch.matmul(qb, k).view(H, n, G, L) / math.sqrt(D)
            pos = torch.arange(L, device="cuda").view(1, 1, 1, L)
            last = (L - n + torch.arange(n, device="cuda")).view(1, n, 1, 1)
            p = torch.softmax(s.masked_fill(pos > last, -math.inf), dim=-1)
            o = torch.matmul(p.reshape(H, n * G, L), v).view(H, n, G, D)
            out[b, :n] = o.permute(1, 0, 2, 3).reshape(n, c["q_heads"], D)
        outs.append(out)
    return outs


def exact(case, seed):
    if case["kind"] not in ("attention", "step"):
        return None
    return {"out": _exact_attention(case, seed), "pool": None}
