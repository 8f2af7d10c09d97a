"""The work a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values; its ``kind`` names the entry point:

* ``attn``        one attention step through
                  ``fused_real_pruning_flat_segmented_attention``
* ``pack``        the slab fill through ``pack_flat_segments_kv`` (one launch
                  per kept prior scale)
* ``produce``     the QKV epilogue through ``qkv_produce``
* ``generation``  every scale of one layer through ``SegmentedLayerCache.step``
* ``layer``       every scale of one whole attention layer (projections,
                  producer, cache step) through the enabled model's forward

A step attends with the ``scale``-th token map of the 13-scale schedule
(``SIDES_1M``; ``aspect`` = height / width, 1 for the square schedule, others
give odd lengths) over the prior scales that its heads keep: ``policy``
"budget" keeps each (head, scale) so that ``budget`` of the prior rows remain
on average, "skewed" draws very different retained lengths per head.
``dtypes``: "bf16" / "fp16" (q, k, v and output), "fp16qk" (fp16 q/k, bf16 v:
what the model's layer runs in its TF32 mode), "model" (fp32 q/k as cosine
attention gives them, bf16 v and output: the model under bf16 autocast) and
"fp32" (the model without autocast).  ``planned``: the call carries the work
plan of its tables, as the segmented cache does; without it the call is the
reference operator's own.  ``k_rows`` "split": K held as split rows (what the
producer writes), "plain": fp32 rows.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

from heatkv_amd import (  # noqa: E402
    SIDES_1M,
    attention_item_shape,
    build_slab_schedule,
    fused_real_pruning_flat_segmented_attention,
    pack_flat_segments_kv,
)
from heatkv_amd import harness  # noqa: E402
from heatkv_amd.produce import precompute_rope2d_freqs_grid, qkv_produce, rope2d_freqs_table  # noqa: E402
from heatkv_amd.segmented_cache import SegmentedLayerCache  # noqa: E402

D = 128
FORCED = 3  # scales every head keeps
DEVICE = "cuda"


# ---------------------------------------------------------------- cases

def listed():
    step = dict(kind="attn", aspect=1.0, policy="budget", budget=0.1, k_rows="plain", lse=False)
    return [
        # An early scale of the 2B model (a CFG pair, 16 heads, 16 tokens): the
        # latency of one launch.
        dict(step, name="scale2_2b_bf16", batch=2, heads=16, scale=2, dtypes="bf16", planned=True),
        # A middle scale (32 x 32 tokens) called as the reference calls its
        # operator: no work plan.
        dict(step, name="scale9_2b_bf16_dropin", batch=2, heads=16, scale=9, dtypes="bf16", planned=False),
        # The last step of a 1024 x 1024 image, 2B model: the headline.
        dict(step, name="final_2b_bf16", batch=2, heads=16, scale=12, dtypes="bf16", planned=True),
        # The last step of the 8B class, four images at once.
        dict(step, name="final_8b_bf16", batch=8, heads=32, scale=12, dtypes="bf16", planned=True),
        # A wide image (odd token counts), heads of very different retained
        # lengths, fp16, with the log-sum-exp.
        dict(step, name="wide_skewed_fp16", batch=3, heads=12, scale=11, aspect=0.57, policy="skewed",
             dtypes="fp16", planned=True, lse=True),
        # The last 2B step at the model's own precision: what its layer runs
        # under bf16 autocast.
        dict(step, name="final_2b_model", batch=2, heads=16, scale=12, dtypes="model", planned=True, k_rows="split"),
        # A middle step at that precision from a program that only swapped the
        # operator: fp32 K rows, no plan.
        dict(step, name="scale10_2b_model_dropin", batch=2, heads=16, scale=10, dtypes="model", planned=False),
        # A late step of the model without autocast: everything fp32.
        dict(step, name="scale11_2b_fp32", batch=2, heads=16, scale=11, dtypes="fp32", planned=True),
        # The QKV epilogue of the last 2B step, with the append of a prior
        # scale's share of heads.
        dict(kind="produce", name="produce_2b_final", batch=2, heads=16, length=4096, dtypes="model", append=True),
        # Compaction at its largest: the 8B class keeping every prior row.
        dict(kind="pack", name="slab_fill_8b", batch=8, heads=32, scale=12, aspect=1.0, policy="budget", budget=1.0,
             dtypes="bf16"),
        # A whole 13-scale generation of one layer's cache: attention, dense
        # prefix, appends; dense and pruned, small and large launches.
        dict(kind="generation", name="generation_2b_bf16", batch=2, heads=16, scales=13, budget=0.1, dtypes="bf16"),
        # The same of one whole attention layer under bf16 autocast.
        dict(kind="layer", name="layer_2b", batch=2, heads=16, scales=13, budget=0.1),
    ]


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["attn"] * 6 + ["produce", "pack", "generation", "layer"])
    batch, heads = rng.choice([1, 2, 2, 3, 4, 8]), rng.choice([5, 12, 16, 16, 20, 32])
    budget = round(math.exp(rng.uniform(math.log(0.05), 0.0)), 3)
    if kind in ("attn", "pack"):
        c = dict(kind=kind, batch=batch, heads=heads, scale=rng.choice([1, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12]),
                 aspect=round(math.exp(rng.uniform(-0.8, 0.8)), 3), policy=rng.choice(["budget", "budget", "skewed"]),
                 budget=budget)
        if kind == "pack":
            return dict(c, scale=max(c["scale"], 5), dtypes=rng.choice(["bf16", "model", "fp16"]))
        c["dtypes"] = rng.choice(["bf16", "bf16", "fp16", "fp16qk", "model", "model", "fp32"])
        if c["dtypes"] in ("model", "fp32"):
            c["batch"], c["heads"] = min(batch, 4), min(heads, 16)
        c["planned"] = rng.random() < 0.7
        c["k_rows"] = rng.choice(["split", "plain"]) if c["dtypes"] == "model" else "plain"
        c["lse"] = rng.random() < 0.25
        return c
    if kind == "produce":
        return dict(kind=kind, batch=batch, heads=heads,
                    length=int(round(math.exp(rng.uniform(math.log(16), math.log(4096))))),
                    dtypes=rng.choice(["model", "bf16", "fp16qk", "fp32"]), append=rng.random() < 0.5)
    c = dict(kind=kind, batch=rng.choice([1, 2, 2, 4]), heads=rng.choice([8, 16]), scales=rng.choice([7, 10, 12, 13]),
             budget=round(rng.uniform(0.08, 0.5), 3))
    if kind == "generation":
        c["dtypes"] = rng.choice(["bf16", "fp16", "model"])
    return c


# ---------------------------------------------------------------- shapes and policies

def _sides(count, aspect):
    """(height, width) of the first ``count`` token maps."""
    r = math.sqrt(aspect)
    return [(max(1, round(s * r)), max(1, round(s / r))) for s in SIDES_1M[:count]]


def _ranges(case):
    out, at = {}, 0
    for i, (h, w) in enumerate(_sides(case["scale"] + 1, case["aspect"])):
        out[i] = (at, at + h * w)
        at += h * w
    return out


def _keep(case, gen):
    """bool [H, prior scales]: which prior scales each head keeps."""
    t, ranges = case["scale"], _ranges(case)
    sizes = [ranges[s][1] - ranges[s][0] for s in range(t)]
    prefix, forced = sum(sizes), sum(sizes[:FORCED])
    if case["policy"] == "skewed":
        u = torch.rand((case["heads"],), generator=gen, dtype=torch.float64)
        keep = torch.zeros((case["heads"], t), dtype=torch.bool)
        for h in range(case["heads"]):
            want = int(math.exp(float(u[h]) * math.log(prefix + 1))) - 1
            for s in sorted(range(t), key=lambda i: -sizes[i]):
                if sizes[s] <= want:
                    keep[h, s] = True
                    want -= sizes[s]
        return keep
    p = 1.0 if prefix <= forced else min(1.0, max(0.0, (case["budget"] * prefix - forced) / (prefix - forced)))
    keep = torch.rand((case["heads"], t), generator=gen, dtype=torch.float64) < p
    keep[:, :FORCED] = True
    return keep


def _policy_seed(case):
    """Which heads keep which scales belongs to the case, as a model's orders do."""
    return 1 + 16 * case["heads"] + (case["scales"] - 1 if "scales" in case else case["scale"])


def _schedule(case):
    keep = _keep(case, torch.Generator().manual_seed(_policy_seed(case)))
    dropped = {s: {h for h in range(keep.shape[0]) if not keep[h, s]} for s in range(keep.shape[1])}
    sched = build_slab_schedule(lambda t: {s: dropped[s] for s in range(min(t, keep.shape[1]))},
                                num_heads=case["heads"], scale_ranges=_ranges(case), num_scales=case["scale"] + 1)
    return keep, sched


def _types(name):
    """q/k dtype, v dtype, output dtype."""
    return {"bf16": (torch.bfloat16,) * 3, "fp16": (torch.float16,) * 3,
            "fp16qk": (torch.float16, torch.bfloat16, torch.bfloat16),
            "model": (torch.float32, torch.bfloat16, torch.bfloat16), "fp32": (torch.float32,) * 3}[name]


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)


def _head_scale(heads):
    """Learned scales of cosine attention, as the model's layers carry them."""
    return torch.linspace(math.log(4.0), math.log(100.0), heads, device=DEVICE).exp()


def _cosine(case):
    """Whether q and k are cosine attention's (unit k, q times its head's scale)."""
    return case["dtypes"] in ("model", "fp32", "fp16qk")


def _qkv(case, gen, batch, heads, length):
    qk, vt, _ = _types(case["dtypes"])
    q, k, v = (_randn(gen, batch, heads, length, D) for _ in range(3))
    if _cosine(case):
        q = torch.nn.functional.normalize(q, dim=-1) * _head_scale(heads).view(1, heads, 1, 1)
        k = torch.nn.functional.normalize(k, dim=-1)
    return q.to(qk), k.to(qk), v.to(vt)


def _softmax_scale(case):
    return 1.0 if _cosine(case) else 1.0 / math.sqrt(D)


def _split_rows(x):
    """fp32 rows as split rows (128 bf16 high parts, 128 low parts; same bytes), typed fp32."""
    hi = x.to(torch.bfloat16)
    lo = (x - hi.float()).to(torch.bfloat16)
    return torch.cat((hi, lo), dim=-1).view(torch.float32)


# ---------------------------------------------------------------- prepare

def _attn_inputs(case, seed):
    keep, sched = _schedule(case)
    gen, ranges = _gen(seed), _ranges(case)
    length = ranges[case["scale"]][1] - ranges[case["scale"]][0]
    q, k, v = _qkv(case, gen, case["batch"], case["heads"], length)
    qk, vt, _ = _types(case["dtypes"])
    sk, sv = (_randn(gen, case["batch"], sched.capacity, D) for _ in range(2))
    if _cosine(case):
        sk = torch.nn.functional.normalize(sk, dim=-1)
    return sched, q, k, v, sk.to(qk), sv.to(vt)


def _prepare_attn(case, seed):
    sched, q, k, v, sk, sv = _attn_inputs(case, seed)
    split = case["k_rows"] == "split"
    if split:
        k, sk = _split_rows(k), _split_rows(sk)
    st, en, ct = sched.device_tables(case["scale"], q.device)
    plan = None
    if case["planned"]:
        plan = sched.device_work_plan(
            case["scale"], q.device, case["batch"], int(q.shape[2]),
            item_shape=attention_item_shape(q.dtype, k.dtype, v.dtype, k_split_rows=split, device=q.device))
    return dict(case=case, call=dict(
        q=q, persisted_k=sk, persisted_v=sv, segment_starts=st, segment_ends=en, segment_counts=ct, current_k=k,
        current_v=v, softmax_scale=_softmax_scale(case), return_lse=case["lse"], out_dtype=_types(case["dtypes"])[2],
        work_plan=plan, k_split_rows=split))


def _prepare_pack(case, seed):
    _, sched = _schedule(case)
    qk, vt, _ = _types(case["dtypes"])
    gen, ranges, B, H = _gen(seed), _ranges(case), case["batch"], case["heads"]
    dk = torch.zeros((B, sched.capacity, D), device=DEVICE, dtype=qk)
    dv = torch.zeros((B, sched.capacity, D), device=DEVICE, dtype=vt)
    calls = []
    for s in range(case["scale"]):
        plan = sched.append_plans.get((s, s + 1))
        if plan is None or len(plan) == 0:
            continue
        n = ranges[s][1] - ranges[s][0]
        starts, sources, lengths = sched.device_plan(plan, dk.device, ("append", s))
        calls.append(dict(dst_k=dk, dst_v=dv, src_k=_randn(gen, B, H * n, D).to(qk),
                          src_v=_randn(gen, B, H * n, D).to(vt), dst_starts=starts, src_starts=sources,
                          lengths=lengths, max_length=plan.max_length))
    return dict(case=case, calls=calls, slab=(dk, dv))


def _produce_offsets(case):
    """Every other head appends, its rows back to back in the slab."""
    n, at, offsets = case["length"], 0, []
    for h in range(case["heads"]):
        offsets.append(at if h % 2 == 0 else -1)
        at += n if h % 2 == 0 else 0
    return offsets, at


def _prepare_produce(case, seed):
    gen, B, H, L = _gen(seed), case["batch"], case["heads"], case["length"]
    qk, vt, _ = _types(case["dtypes"])
    side = math.isqrt(L - 1) + 1 if L > 1 else 1
    table = rope2d_freqs_table(D, [(1, side, side)]).to(DEVICE)
    offsets, capacity = _produce_offsets(case)
    append = None
    if case["append"]:
        append = (torch.zeros((B, capacity, D), device=DEVICE, dtype=qk),
                  torch.zeros((B, capacity, D), device=DEVICE, dtype=vt),
                  torch.tensor(offsets, dtype=torch.int32, device=DEVICE))
    return dict(case=case, qkv=_randn(gen, B, L, 3 * H * D).to(vt), append=append, table=table,
                scale_mul=_head_scale(H))


def _generation_keep(case):
    return _keep(dict(case, scale=case["scales"] - 1, aspect=1.0, policy="budget"),
                 torch.Generator().manual_seed(_policy_seed(case)))


def _prepare_generation(case, seed):
    c = dict(case, scale=case["scales"] - 1, aspect=1.0, policy="budget")
    keep, sched = _schedule(c)
    dropped = {s: {h for h in range(keep.shape[0]) if not keep[h, s]} for s in range(keep.shape[1])}
    cache = SegmentedLayerCache(sched, lambda t: {s: dropped[s] for s in range(min(t, keep.shape[1]))},
                                num_heads=case["heads"], num_scales=case["scales"])
    gen = _gen(seed)
    steps = [_qkv(case, gen, case["batch"], case["heads"], s * s) for s in SIDES_1M[:case["scales"]]]
    if case["dtypes"] == "model":
        steps = [(q, _split_rows(k), v) for q, k, v in steps]
    return dict(case=case, cache=cache, steps=steps)


def _layer_model(case, seed):
    sides = SIDES_1M[:case["scales"]]
    orders = harness.seeded_orders(1, case["heads"], max(0, len(SIDES_1M) - 1 - FORCED), _policy_seed(case))
    model = harness.build_model(harness.METHOD_NAME, device=DEVICE, num_layers=1, num_heads=case["heads"],
                                embed_dim=case["heads"] * D, budget=case["budget"], initial_scales=FORCED,
                                orders=orders, seed=seed)
    schedule = [(1, s, s) for s in SIDES_1M]
    grid = precompute_rope2d_freqs_grid(D, {1.0: {"1M": {"scales": schedule}}}, 2, pad_to_multiplier=128,
                                        device=DEVICE)
    gen = _gen(seed)
    xs = [_randn(gen, case["batch"], s * s, case["heads"] * D).to(torch.bfloat16) for s in sides]
    return model, schedule, grid, xs


def prepare(case, seed):
    if case["kind"] == "layer":
        model, schedule, grid, xs = _layer_model(case, seed)
        return dict(case=case, model=model, schedule=schedule, grid=grid, xs=xs)
    return {"attn": _prepare_attn, "pack": _prepare_pack, "produce": _prepare_produce,
            "generation": _prepare_generation}[case["kind"]](case, seed)


# ---------------------------------------------------------------- run

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        return fused_real_pruning_flat_segmented_attention(**state["call"])
    if kind == "pack":
        for c in state["calls"]:
            pack_flat_segments_kv(**c)
        return state["slab"]
    if kind == "produce":
        qkv = qkv_produce(state["qkv"], case["heads"], scale_mul=state["scale_mul"], rope_table=state["table"],
                          qk_dtype=_types(case["dtypes"])[0], append=state["append"],
                          k_split_rows=case["dtypes"] == "model")
        out = _bytes_of_k(case, *qkv)
        return out + (_bytes_of_k(case, None, *state["append"][:2])[1:] if state["append"] is not None else ())
    if kind == "generation":
        out_dtype = _types(case["dtypes"])[2]
        return [state["cache"].step(q, k, v, t, _softmax_scale(case), out_dtype=out_dtype,
                                    k_split_rows=case["dtypes"] == "model")
                for t, (q, k, v) in enumerate(state["steps"])]
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        for layer in state["model"]:
            layer.kv_caching(True)
        out = []
        for t, x in enumerate(state["xs"]):
            for layer in state["model"]:
                x = layer(x, None, None, state["schedule"], state["grid"], t)
            out.append(x)
    return out


def _bytes_of_k(case, q, k, v):
    """Split rows are pairs of bf16 parts: seen as such (a view), not as the fp32 they are typed."""
    return q, (k.view(torch.bfloat16) if case["dtypes"] == "model" else k), v


# ---------------------------------------------------------------- work and tolerance

def _retained(keep, ranges, t):
    """Prior rows over all heads at target t."""
    return sum(ranges[s][1] - ranges[s][0] for h in range(keep.shape[0]) for s in range(min(t, keep.shape[1]))
               if keep[h, s])


def _step_work(case, length, rows, size):
    """One attention step: ``rows`` = retained prior rows over all heads."""
    B, H = case["batch"], case["heads"]
    sq, sv, so = size
    return (B * D * (H * length * (2 * sq + sv + so) + rows * (sq + sv)), 4 * B * length * D * (rows + H * length))


def work(case):
    size = [torch.empty((), dtype=t).element_size() for t in _types(case.get("dtypes", "model"))]
    B, H = case["batch"], case["heads"]
    if case["kind"] == "produce":
        rows = B * case["length"] * H
        kept = rows // 2 if case["append"] else 0
        return {"bytes": D * (rows * (3 * size[1] + 2 * size[0] + size[1]) + kept * (size[0] + size[1]))
                + case["length"] * D * 4, "flops": 0}
    if case["kind"] in ("attn", "pack"):
        keep, sched = _schedule(case)
        ranges = _ranges(case)
        if case["kind"] == "pack":
            slots = sum(p.slots for (s, _), p in sched.append_plans.items() if s < case["scale"])
            return {"bytes": 2 * B * slots * D * (size[0] + size[1]), "flops": 0}
        a, b = ranges[case["scale"]]
        n, f = _step_work(case, b - a, _retained(keep, ranges, case["scale"]), size)
        return {"bytes": n + (4 * B * H * (b - a) if case["lse"] else 0), "flops": f}
    c = dict(case, scale=case["scales"] - 1, aspect=1.0, policy="budget")
    ranges, nbytes, flops = _ranges(c), 0, 0
    if case["kind"] == "generation":
        keep = _generation_keep(case)
        for t in range(case["scales"]):
            a, b = ranges[t]
            n, f = _step_work(case, b - a, _retained(keep, ranges, t), size)
            nbytes, flops = nbytes + n, flops + f
        return {"bytes": nbytes, "flops": flops}
    tokens, width = ranges[case["scales"] - 1][1], H * D
    removed = _layer_removed(case)
    for t in range(case["scales"]):
        a, b = ranges[t]
        rows = sum(ranges[s][1] - ranges[s][0] for s in range(t) for h in range(H) if h not in removed(t).get(s, ()))
        flops += 4 * B * (b - a) * D * (rows + H * (b - a))
    return {"bytes": 2 * (2 * B * tokens * width + 4 * width * width), "flops": flops + 8 * B * tokens * width * width}


def tolerance(case):
    if case["kind"] == "pack":
        return "exact"
    kind = case.get("dtypes", "model")
    if case["kind"] == "produce":
        # 32-bit arithmetic, off by 6e-8 from 64 bits; the parts of split rows
        # and 16-bit results move by a rounding step where that crosses a tie
        return {"rel": 1e-6, "max": 1e-5} if kind == "fp32" else {"rel": 1e-3, "max": 0.02}
    # Off by this much from 64 bits (2-norm): 1.4e-5 for fp32 (products of 16
    # significand bits), 2.9e-4 with probabilities and results in fp16, 2.1e-3
    # to 2.6e-3 with either in bf16.  About four times that:
    return {"fp32": {"rel": 6e-5, "max": 3e-3}, "fp16": {"rel": 1.2e-3, "max": 0.03}}.get(
        kind, {"rel": 1e-2, "max": 0.25})


# ---------------------------------------------------------------- 64-bit results

def _attend64(q, keys, values, scale):
    """softmax(scale q k^T) v of one (batch, head) in 64 bits; the log-sum-exp beside it."""
    out, lse = [], []
    for part in q.double().split(1024):
        s = part @ keys.T * scale
        top = s.max(dim=1, keepdim=True).values
        p = (s - top).exp()
        total = p.sum(dim=1, keepdim=True)
        out.append(p @ values / total)
        lse.append((top + total.log()).squeeze(1))
    return torch.cat(out), torch.cat(lse)


def _exact_attn(case, seed):
    sched, q, k, v, sk, sv = _attn_inputs(case, seed)
    st, en, ct = sched.tables[case["scale"]]
    B, H, L, _ = q.shape
    out = torch.empty((B, L, H * D), device=DEVICE, dtype=torch.float64)
    lse = torch.empty((B, H, L), device=DEVICE, dtype=torch.float64)
    for h in range(H):
        rows = torch.cat([torch.arange(int(st[h, i]), int(en[h, i])) for i in range(int(ct[h]))]
                         or [torch.zeros(0, dtype=torch.int64)]).to(DEVICE)
        for b in range(B):
            keys = torch.cat((sk[b, rows], k[b, h])).double()
            vals = torch.cat((sv[b, rows], v[b, h])).double()
            out[b, :, h * D:(h + 1) * D], lse[b, h] = _attend64(q[b, h], keys, vals, _softmax_scale(case))
    return (out, lse) if case["lse"] else out


def _exact_kept(steps, kept, scale):
    """Every step of a generation: ``steps`` of (q, k, v) [B, H, n, D], ``kept(t, h)`` the prior scales head h attends to."""
    outs = []
    for t, (q, k, v) in enumerate(steps):
        B, H, L, _ = q.shape
        out = torch.empty((B, L, H * D), device=DEVICE, dtype=torch.float64)
        for h in range(H):
            of = kept(t, h) + [t]
            for b in range(B):
                keys = torch.cat([steps[s][1][b, h] for s in of]).double()
                vals = torch.cat([steps[s][2][b, h] for s in of]).double()
                out[b, :, h * D:(h + 1) * D], _ = _attend64(q[b, h], keys, vals, scale)
        outs.append(out)
    return outs


def _rotate64(x, table, start):
    c, s = (table[i, start:start + x.shape[2]].double() for i in range(2))
    x = x.reshape(*x.shape[:-1], D // 2, 2)
    return torch.stack((c * x[..., 0] - s * x[..., 1], s * x[..., 0] + c * x[..., 1]), dim=-1).flatten(-2)


def _prologue64(qkv, heads, scale_mul, table, start):
    """[B, L, 3HD] -> q, k, v [B, H, L, D] in 64 bits."""
    B, L, _ = qkv.shape
    q, k, v = qkv.double().reshape(B, L, 3, heads, D).permute(2, 0, 3, 1, 4)
    q = q / q.norm(dim=-1, keepdim=True) * scale_mul.double().view(1, heads, 1, 1)
    k = k / k.norm(dim=-1, keepdim=True)
    return _rotate64(q, table, start), _rotate64(k, table, start), v


def _exact_produce(case, seed):
    state = _prepare_produce(case, seed)
    q, k, v = _prologue64(state["qkv"], case["heads"], state["scale_mul"], state["table"], 0)
    if case["dtypes"] == "model":
        hi = k.float().to(torch.bfloat16).double()
        k = torch.cat((hi, k - hi), dim=-1)
    out = [q, None if case["dtypes"] == "model" else k, v]
    if case["append"]:
        offsets, capacity = _produce_offsets(case)
        sv = torch.zeros((case["batch"], capacity, D), device=DEVICE, dtype=torch.float64)
        for h, off in enumerate(offsets):
            if off >= 0:
                sv[:, off:off + case["length"]] = v[:, h]
        out += [None, sv]
    return tuple(out)


def _layer_removed(case):
    from heatkv_amd.policy import controller_for_budget

    orders = harness.seeded_orders(1, case["heads"], max(0, len(SIDES_1M) - 1 - FORCED), _policy_seed(case))
    ctrl = controller_for_budget(case["budget"], orders, num_layers=1, num_heads=case["heads"],
                                 protected_prefix_scales=FORCED, source_scale_start=FORCED)
    return lambda t: ctrl.removed_heads_by_source_for(0, t)


def _exact_layer(case, seed):
    model, _, grid, xs = _layer_model(case, seed)
    layer, H = model[0], case["heads"]
    table = next(iter(grid.values())).reshape(2, -1, D // 2)
    bias = torch.cat((layer.q_bias, layer.zero_k_bias, layer.v_bias)).double()
    mul = layer.scale_mul_1H11.detach().reshape(-1).float().clamp_max(layer.max_scale_mul).exp()
    steps, at = [], 0
    with torch.no_grad():
        for x in xs:
            # autocast's projection is bf16: rounded here too, the rest in 64 bits
            qkv = (x.double() @ layer.mat_qkv.weight.double().T + bias).to(torch.bfloat16)
            steps.append(_prologue64(qkv, H, mul, table, at))
            at += x.shape[1]
        removed = _layer_removed(case)
        outs = _exact_kept(steps, lambda t, h: [s for s in range(t) if h not in removed(t).get(s, ())], 1.0)
        return [o @ layer.proj.weight.double().T + layer.proj.bias.double() for o in outs]


def exact(case, seed):
    if case["kind"] == "attn":
        return _exact_attn(case, seed)
    if case["kind"] == "produce":
        return _exact_produce(case, seed)
    if case["kind"] == "generation":
        gen, keep = _gen(seed), _generation_keep(case)
        steps = [_qkv(case, gen, case["batch"], case["heads"], s * s) for s in SIDES_1M[:case["scales"]]]
        return _exact_kept(steps, lambda t, h: [s for s in range(min(t, keep.shape[1])) if keep[h, s]],
                           _softmax_scale(case))
    if case["kind"] == "layer":
        return _exact_layer(case, seed)
    return None  # copies
