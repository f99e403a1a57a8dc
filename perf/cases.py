"""The work that a program hands to this package, as cases that can be timed and compared.

A case is one pass through the public entry points: an attention call of a decode step (the stream-ordered
``torch.ops.fa_amd`` operators, or the blocking ``lib.paged_attention_*.run`` of the reference's own
programs), an append to the KV pools, or an append followed by the attention that reads it.  The fields:

  kind     "attention", "append", or "step" (append one token per sequence, then attend)
  api      "op": torch.ops.fa_amd.*, asynchronous;  "run": lib.*.run, which waits and returns kernel times
  entry    "loop" (single pass) or "reduce" (context split over partitions, then merged)
  q        type of queries and outputs: "fp16" or "bf16";  kv: "16" (the same type), "e5m2" or "e4m3"
  S, H, Hk, D, B   sequences, query heads, kv heads, head size, tokens per block
  rows     pool layout: "head" [blocks, kv_heads, block, D] or "token" [blocks, block, kv_heads, D]
  lens     how context lengths spread over lo .. hi: "uniform", "lognormal" (median lo, cut at hi) or "full" (all hi)
  QL       query tokens per sequence (1 = decode; more = verifying drafted tokens)
  sinks, alibi, softcap, window   what is added to or done with the scores (softcap 0, window -1: not)
  scales   of an FP8 pool: "tensor", "head" or "block"
  tokens, slots    of an append: how many rows; "prefill" (consecutive slots per sequence) or "decode" (anywhere)
"""
import math
import statistics

import torch

from flash_attention_factory_amd import torch_ops  # noqa: F401  (registers torch.ops.fa_amd)
from flash_attention_factory_amd.lib import (kv_cache_write, paged_attention_fp8_loop, paged_attention_fp8_reduce,
                                             paged_attention_loop, paged_attention_reduce)

_RUN = {("loop", False): paged_attention_loop, ("reduce", False): paged_attention_reduce,
        ("loop", True): paged_attention_fp8_loop, ("reduce", True): paged_attention_fp8_reduce}
_Q = {"fp16": torch.float16, "bf16": torch.bfloat16}
_FP8 = {"e5m2": torch.float8_e5m2, "e4m3": torch.float8_e4m3fn}
_DEFAULTS = dict(kind="attention", api="op", entry="loop", q="fp16", kv="16", S=1, H=8, Hk=8, D=128, B=16, rows="head",
                 lens="uniform", lo=1, hi=1024, QL=1, sinks=False, alibi=False, softcap=0.0, window=-1, scales="tensor",
                 tokens=0, slots="decode")


def _case(**fields):
    return {**_DEFAULTS, **fields}


def listed():
    return [
        # the smallest step: a few short sequences of a small model, append and attend
        _case(name="step_few_short", kind="step", S=4, H=8, Hk=8, D=64, lo=1, hi=256),
        # a handful of users with a few thousand tokens each, grouped-query heads
        _case(name="loop_few_users", q="bf16", S=3, H=32, Hk=8, lo=900, hi=4096),
        # a decode batch of a 7B-shaped model with 16-bit and with byte pools
        _case(name="loop_fp16_batch", S=32, H=32, Hk=32, lo=512, hi=2048),
        _case(name="loop_e5m2_batch", kv="e5m2", S=32, H=32, Hk=32, lo=512, hi=2048),
        # the reference's own measuring loop: 64 equal rows, blocks of 64, sinks, its blocking call ...
        _case(name="run_fp16_equal_rows", api="run", S=64, H=64, Hk=8, D=64, B=64, rows="token", lens="full", hi=1500, sinks=True),
        # ... and its byte pools, through the split entry
        _case(name="reduce_e5m2_equal_rows", entry="reduce", kv="e5m2", S=64, H=40, Hk=8, D=64, B=64, rows="token", lens="full",
              hi=1500, sinks=True),
        # one user with a long document: latency
        _case(name="reduce_one_long", entry="reduce", q="bf16", S=1, H=32, Hk=8, lens="full", hi=30011),
        # a few long documents
        _case(name="reduce_fp16_long", entry="reduce", S=8, H=32, Hk=8, lo=8192, hi=32768),
        # a large serving mix, byte pools: the largest call
        _case(name="reduce_e5m2_mix", entry="reduce", q="bf16", kv="e5m2", S=128, H=64, Hk=8, lens="lognormal", lo=4096, hi=32768),
        # four drafted tokens per sequence verified at once, byte pools with a scale per head
        _case(name="reduce_verify_tokens", entry="reduce", q="bf16", kv="e4m3", S=48, H=64, Hk=8, lo=257, hi=6000, QL=4, scales="head"),
        # a layer with capped scores, a local window, distance penalties and sinks
        _case(name="loop_window_cap", q="bf16", S=24, H=32, Hk=16, B=32, lo=300, hi=5000, sinks=True, alibi=True, softcap=30.0,
              window=1023),
        # the append of a prefill
        _case(name="append_prefill", kind="append", kv="e5m2", Hk=8, tokens=32768, slots="prefill"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_MOST_BYTES = 1.5e9  # what a drawn call may have to move: below the largest listed one


def draw(rng):
    while True:
        kind = rng.choices(["attention", "append", "step"], [0.72, 0.14, 0.14])[0]
        entry = rng.choice(["loop", "reduce"])
        kv = rng.choices(["16", "e5m2", "e4m3"], [0.5, 0.3, 0.2])[0]
        group = rng.choice([1, 1, 2, 4, 4, 5, 7, 8])
        heads = rng.choice([2, 4, 5, 8, 8, 16, 32])
        c = _case(kind=kind, entry=entry, kv=kv, q=rng.choice(["fp16", "bf16"]), S=_log_int(rng, 1, 300), H=group * heads, Hk=heads,
                  D=rng.choice([128, 128, 64]), B=rng.choice([16, 16, 32, 64]), rows=rng.choice(["head", "head", "token"]),
                  lens=rng.choice(["uniform", "uniform", "lognormal", "full"]), sinks=rng.random() < 0.25)
        c["hi"] = _log_int(rng, 64, 8192 if entry == "loop" else 32768)
        c["lo"] = max(1, int(c["hi"] * rng.uniform(0.05, 0.6)))
        if kind == "append":
            c.update(tokens=_log_int(rng, 1, 32768), slots=rng.choice(["prefill", "decode"]))
        elif kind == "attention":
            c["api"] = rng.choice(["op", "op", "op", "run"])
            extra = rng.random()
            if extra < 0.15:
                c.update(QL=rng.randint(2, 8))
            elif extra < 0.3:
                c.update(softcap=rng.choice([0.0, 30.0]), window=rng.choice([-1, 511, 1023]), alibi=rng.random() < 0.5)
        if kv != "16":
            c["scales"] = rng.choice(["tensor", "tensor", "head", "block"])
        if work(c)["bytes"] <= _MOST_BYTES:
            return c


def _lengths(case):
    """The batch's context lengths in ascending order.  They are the distribution's own quantiles, so that
    every seed deals the same work (in another order, to other blocks)."""
    n, lo, hi = case["S"], case["lo"], case["hi"]
    least = max(case["QL"], 1)
    if case["lens"] == "full":
        return [max(least, hi)] * n
    at = [(k + 0.5) / n for k in range(n)]
    if case["lens"] == "uniform":
        got = [lo + u * (hi - lo) for u in at]
    else:
        normal = statistics.NormalDist()
        got = [lo * math.exp(0.75 * normal.inv_cdf(u)) for u in at]
    return [max(least, min(hi, int(round(x)))) for x in got]


def _partition(case):
    return 512 if case["D"] == 128 else 256  # what the library takes by default


def prepare(case, seed):
    dev = torch.device("cuda")
    c = case
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    host = torch.Generator()
    host.manual_seed(seed)
    q_type, fp8 = _Q[c["q"]], c["kv"] != "16"
    S, H, Hk, D, B, QL = c["S"], c["H"], c["Hk"], c["D"], c["B"], c["QL"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device=dev, dtype=torch.float16).to(q_type)

    lens = torch.tensor(_lengths(c), dtype=torch.int64)[torch.randperm(S, generator=host)]
    if c["kind"] == "append":  # a pool with twice the room that the tokens need
        need = 2 * -(-c["tokens"] // B)
    else:
        need = int(((lens + B - 1) // B).sum())
    blocks = need + need // 8 + 1
    shape = (blocks, Hk, B, D) if c["rows"] == "head" else (blocks, B, Hk, D)
    k_scales = v_scales = None
    if c["scales"] != "tensor":  # about what the largest value of a head or block asks for
        of = (Hk,) if c["scales"] == "head" else (blocks, Hk)
        k_scales, v_scales = (0.5 + torch.rand(of, generator=g, device=dev) for _ in range(2))
    pools = []
    for _ in range(2):
        pool = normal(*shape)
        pools.append(pool.to(_FP8[c["kv"]]) if fp8 else pool)
    # the views that the entry points take: [blocks, block_size, kv_heads, head_size]
    keys, values = (p.permute(0, 2, 1, 3) if c["rows"] == "head" else p for p in pools)
    s = dict(case=c, fp8=fp8, pools=[p.view(torch.uint8) if fp8 else p for p in pools], keys=keys, values=values, k_scales=k_scales,
             v_scales=v_scales, fp8_scale=1.0)
    perm = torch.randperm(blocks, generator=host)
    if c["kind"] == "append":
        n = c["tokens"]
        if c["slots"] == "prefill":
            t = torch.arange(n)
            slots = perm[t // B] * B + t % B
        else:
            slots = torch.randperm(blocks * B, generator=host)[:n]
        s.update(new_keys=normal(n, Hk, D), new_values=normal(n, Hk, D), slots=slots.to(dev))
        return s
    per_seq = (lens + B - 1) // B
    tables = torch.zeros((S, int(per_seq.max())), dtype=torch.int32)
    tables[torch.arange(tables.size(1))[None, :] < per_seq[:, None]] = perm[:need].to(torch.int32)
    if c["kind"] == "step":  # the newest token of every sequence
        last = lens - 1
        slots = tables[torch.arange(S), last // B].to(torch.int64) * B + last % B
        s.update(new_keys=normal(S, Hk, D), new_values=normal(S, Hk, D), slots=slots.to(dev))
    q_shape = (S, H, D) if QL == 1 else (S, QL, H, D)
    s.update(query=normal(*q_shape), out=torch.zeros(q_shape, dtype=q_type, device=dev), tables=tables.to(dev),
             lens=lens.to(torch.int32).to(dev), longest=int(lens.max()), scale=1.0 / math.sqrt(D),
             sinks=normal(H) if c["sinks"] else None,
             slopes=torch.exp2(-8.0 * torch.arange(1, H + 1, device=dev) / H).float() if c["alibi"] else None)
    if c["entry"] == "reduce":
        parts = -(-s["longest"] // _partition(c))
        s.update(exp_sums=torch.zeros((S * QL, H, parts), device=dev), max_logits=torch.zeros((S * QL, H, parts), device=dev),
                 tmp_out=torch.zeros((S * QL, H, parts, D), device=dev))
    return s


def _append(s):
    torch.ops.fa_amd.kv_cache_write(s["new_keys"], s["new_values"], s["keys"], s["values"], s["slots"], s["fp8_scale"],
                                    s["k_scales"], s["v_scales"])


def _attend_op(s):
    c = s["case"]
    head = (s["query"], s["keys"], s["values"], s["tables"], s["lens"], s["scale"])
    more = dict(sinks=s["sinks"], alibi_slopes=s["slopes"], softcap=c["softcap"], window_left=c["window"])
    if s["fp8"]:
        head += (s["fp8_scale"],)
        more.update(k_scales=s["k_scales"], v_scales=s["v_scales"])
    ops = torch.ops.fa_amd
    if c["entry"] == "loop":
        (ops.paged_attention_fp8_loop if s["fp8"] else ops.paged_attention_loop)(s["out"], *head, **more)
    else:
        (ops.paged_attention_fp8_reduce if s["fp8"] else ops.paged_attention_reduce)(
            s["out"], s["exp_sums"], s["max_logits"], s["tmp_out"], *head, max_context_len=s["longest"], **more)


def _attend_run(s):
    c = s["case"]
    split = c["entry"] == "reduce"
    head = (s["max_logits"], s["exp_sums"], s["tmp_out"]) if split else (None, None, None)
    head += (s["out"], None, s["query"], s["keys"], s["values"], s["tables"], s["lens"], c["H"] // c["Hk"], s["scale"])
    more = dict(apply_alibi=c["alibi"], apply_softcap=c["softcap"] > 0, window_left=c["window"] if c["window"] >= 0 else None)
    if s["fp8"]:
        head += (s["fp8_scale"],)
        more.update(k_scales=s["k_scales"], v_scales=s["v_scales"])
    _RUN[c["entry"], s["fp8"]].run(*head, c["B"], s["longest"], s["slopes"], s["sinks"], c["softcap"], **more)


def run(state):
    kind = state["case"]["kind"]
    if kind != "attention":
        _append(state)
    if kind == "append":
        return state["pools"]
    (_attend_run if state["case"]["api"] == "run" else _attend_op)(state)
    return [state["out"], *state["pools"]] if kind == "step" else state["out"]


def work(case):
    c = case
    kv_bytes = 2 if c["kv"] == "16" else 1
    row = 2 * c["Hk"] * c["D"]  # elements of one token's K and V rows
    if c["kind"] == "append":
        return {"bytes": c["tokens"] * (row * (2 + kv_bytes) + 8), "flops": 0}
    read = scores = entries = 0
    for n in _lengths(c):
        seen = n if c["window"] < 0 else min(n, c["window"] + c["QL"])  # keys that some query token sees
        read += seen
        scores += c["QL"] * min(n, c["window"] + 1 if c["window"] >= 0 else n) - c["QL"] * (c["QL"] - 1) // 2
        entries += -(-seen // c["B"])
    total = read * row * kv_bytes + 2 * c["S"] * c["QL"] * c["H"] * c["D"] * 2 + entries * 4 + c["S"] * 4
    if c["scales"] == "block":
        total += entries * c["Hk"] * 8
    if c["kind"] == "step":
        total += c["S"] * (row * (2 + kv_bytes) + 8)
    return {"bytes": total, "flops": max(scores, 0) * 4 * c["H"] * c["D"]}


def tolerance(case):
    """Appends place and round single values: their bytes are the bytes.  Attention rounds the probabilities and
    the output to the query type: against the same attention in 64 bits the results differ by 2.5e-4 to 2.9e-4
    (fp16) and 2.0e-3 to 2.4e-3 (bf16) over the ranges above; four to five times that is stated."""
    if case["kind"] == "append":
        return "exact"
    return {"rel": 1.2e-3 if case["q"] == "fp16" else 1e-2}
