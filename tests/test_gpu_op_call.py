"""The operators' native call path (csrc/op_call.cpp) against their Python
bodies: the same bits where it takes a call, the same errors and results where
it leaves the call to the body."""

from __future__ import annotations

import pytest
import torch

from heatkv_amd import (
    _lib,
    attention_item_shape,
    fused_real_pruning_flat_segmented_attention,
    pack_flat_segments_kv,
    segmented_attention_plan,
)
from heatkv_amd.produce import qkv_produce, rope2d_freqs_table

pytestmark = pytest.mark.gpu
D = 128


def split_rows(x):
    hi = x.to(torch.bfloat16)
    return torch.cat((hi, (x - hi.float()).to(torch.bfloat16)), dim=-1).view(torch.float32)


def attention_args(device, dtypes=(torch.bfloat16,) * 3, B=2, H=3, L=33, cap=50, planned=False, **kw):
    g = torch.Generator().manual_seed(5)
    rand = lambda *s: torch.randn(s, generator=g).to(device)  # noqa: E731
    qd, kd, vd = dtypes
    st = torch.tensor([[0, 20], [5, 40], [30, 30]][:H], dtype=torch.int32)
    en = torch.tensor([[10, 33], [6, 50], [30, 49]][:H], dtype=torch.int32)
    ct = torch.tensor([2, 2, 1][:H], dtype=torch.int32)
    plan = None
    if planned:
        qpi, slots = attention_item_shape(qd, kd, vd, k_split_rows=kw.get("k_split_rows", False), device=device)
        plan = segmented_attention_plan(st, en, ct, batch_size=B, current_len=L, capacity=cap, device=device,
                                        queries_per_item=qpi, slots=slots)
    if kw.get("k_split_rows"):  # K as split rows: bf16 high parts, then low parts
        rand_k = lambda *s: split_rows(rand(*s))  # noqa: E731
    else:
        rand_k = rand
    return dict(q=rand(B, H, L, D).to(qd), persisted_k=rand_k(B, cap, D).to(kd), persisted_v=rand(B, cap, D).to(vd),
                segment_starts=st.to(device), segment_ends=en.to(device), segment_counts=ct.to(device),
                current_k=rand_k(B, H, L, D).to(kd), current_v=rand(B, H, L, D).to(vd), softmax_scale=0.09,
                work_plan=plan, **kw)


def native(a):
    return _lib.op_call.attention(
        a["q"], a["persisted_k"], a["persisted_v"], a["segment_starts"], a["segment_ends"], a["segment_counts"],
        a["current_k"], a["current_v"], a["softmax_scale"], a.get("softmax_mode", "exp"), a.get("return_lse", False),
        a.get("out_dtype"), a.get("work_plan"), a.get("k_split_rows", False), 4096, 65536)


def body(fn, *args, **kw):
    """The call through the Python body; an error as its type and text."""
    saved, _lib.op_call = _lib.op_call, None
    try:
        return fn(*args, **kw)
    except Exception as e:  # noqa: BLE001 - compared with the other path's
        return type(e), str(e)
    finally:
        _lib.op_call = saved


def public(fn, *args, **kw):
    try:
        return fn(*args, **kw)
    except Exception as e:  # noqa: BLE001
        return type(e), str(e)


def same(x, y):
    if isinstance(x, torch.Tensor):
        return (isinstance(y, torch.Tensor) and x.dtype == y.dtype and x.shape == y.shape and x.device == y.device
                and x.requires_grad == y.requires_grad and torch.equal(x, y))
    if isinstance(x, tuple):
        return isinstance(y, tuple) and len(x) == len(y) and all(same(a, b) for a, b in zip(x, y))
    return x == y


BF, FP, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(autouse=True)
def ready(device):
    _lib.load()
    assert _lib.op_call is not None
    body(fused_real_pruning_flat_segmented_attention, **attention_args(device))  # checks the device, workspace


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("kw", [{}, {"return_lse": True, "softmax_mode": "exp2"}, {"out_dtype": F32}])
@pytest.mark.parametrize("dtypes", [(BF, BF, BF), (FP, FP, BF), (F32, F32, BF), (F32, F32, F32), "split"], ids=str)
def test_attention_taken(device, dtypes, kw, planned):
    if dtypes == "split":
        dtypes, kw = (F32, F32, BF), dict(kw, k_split_rows=True)
    a = attention_args(device, dtypes, planned=planned, **kw)
    got = native(a)
    assert got is not None
    torch.cuda.synchronize(device)
    want = body(fused_real_pruning_flat_segmented_attention, **a)
    assert same(got, want)
    if dtypes[2] == F32 and not planned:  # a small call on a slab whose split copies would be large: staged kernel
        big = dict(a, **{n: torch.cat((a[n], a[n].new_zeros(2, 40000, D)), dim=1) for n in ("persisted_k", "persisted_v")})
        got = native(big)
        torch.cuda.synchronize(device)
        assert same(got, body(fused_real_pruning_flat_segmented_attention, **big)) and not same(got, want)


@pytest.mark.parametrize("B,H,L,cap,split", [
    (1, 2, 16, 65536, True), (1, 2, 16, 65537, False),         # few rows: the slab's own limit
    (4, 16, 64, 4096, True), (4, 16, 64, 4097, False),         # 4096 rows: 4 slab rows each
    (1, 16, 256, 16384, True), (1, 16, 256, 16385, False),
    (1, 16, 257, 32896, True), (1, 16, 257, 32897, False),     # 8 above 256 tokens
    (8, 32, 16, 25000, False),                                 # rows a pool of kept slabs would have
    (5, 13, 126, 8, True), (5, 13, 127, 8, False),             # one round of the staged kernel
    (4, 16, 128, 8, True), (8, 32, 128, 8, False), (8, 33, 128, 8, True), (8, 32, 129, 8, True)])
def test_fp32_split_copies_only_where_they_pay(device, B, H, L, cap, split, monkeypatch):
    """All-fp32 calls make split copies on the inner side of each limit and run
    as they are, with no memory beside their outputs, on the other: both paths
    of the operator alike."""
    g = torch.Generator(device=device).manual_seed(3)
    rand = lambda *s: torch.randn(s, generator=g, device=device)  # noqa: E731
    table = torch.zeros((H, 1), dtype=torch.int32, device=device)
    a = dict(q=rand(B, H, L, D), persisted_k=rand(B, cap, D), persisted_v=rand(B, cap, D), segment_starts=table,
             segment_ends=table + min(cap, 8), segment_counts=torch.ones(H, dtype=torch.int32, device=device),
             current_k=rand(B, H, L, D), current_v=rand(B, H, L, D), softmax_scale=0.09)

    def measured(fn):
        torch.cuda.synchronize(device)
        torch.cuda.reset_peak_memory_stats(device)
        before = torch.cuda.memory_allocated(device)
        out = fn()
        torch.cuda.synchronize(device)
        return out, torch.cuda.max_memory_allocated(device) - before - out.numel() * out.element_size()

    got, used = measured(lambda: native(a))
    want, body_used = measured(lambda: body(fused_real_pruning_flat_segmented_attention, **a))
    monkeypatch.setenv("HKV_ATTN_SPLIT_ROWS", "0")
    staged, _ = measured(lambda: fused_real_pruning_flat_segmented_attention(**a))
    assert same(got, want) and same(got, staged) != split
    copies = 2 * 512 * B * (cap + H * L)
    # torch's allocator leaves up to 1 MB of a cached block on one of over 1 MB, and rounds new ones up to 2 MB
    rounding = 2 << 20
    assert copies > 3 * rounding or split
    for n in (used, body_used):
        assert (n >= copies) if split else (n < rounding)


def test_fp32_call_without_room_for_split_copies(device, monkeypatch):
    """Where the split copies cannot be allocated the call runs as it does
    without them."""
    a = attention_args(device, (F32, F32, F32), L=300)
    for n in ("persisted_k", "persisted_v"):
        a[n] = torch.cat((a[n], a[n].new_zeros(2, 30000, D)), dim=1)
    fn = fused_real_pruning_flat_segmented_attention
    with monkeypatch.context() as m:
        m.setenv("HKV_ATTN_SPLIT_ROWS", "0")
        want = fn(**a)
    assert not same(fn(**a), want)  # split where there is room
    torch.cuda.synchronize(device)
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved(device) + (24 << 20)
    held = []
    try:
        torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(device).total_memory, device)
        # fill what earlier tests left in the allocator's segments, then leave one hole: it and
        # the free rest beside it take the output, not 64 MB of copies
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                held.append(torch.empty(8 << 20, dtype=torch.uint8, device=device))
        held.pop()
        for call in (fn, lambda **kw: body(fn, **kw)):
            got = call(**a)
            torch.cuda.synchronize(device)
            assert same(got, want)
            del got
    finally:
        held.clear()
        torch.cuda.set_per_process_memory_fraction(1.0, device)


def _changes(device):
    """Calls outside the native path, or refused: name -> changed arguments."""
    a = attention_args(device)
    wide = torch.randn((2, 33, 3, D), device=device).to(BF).transpose(1, 2)  # [B, H, L, D], strided
    plan = attention_args(device, planned=True)["work_plan"]
    other = attention_args(device, L=65, planned=True)["work_plan"]
    return {
        "strided q": dict(q=wide), "strided v": dict(current_v=wide),
        "int64 tables": {k: a[k].long() for k in ("segment_starts", "segment_ends", "segment_counts")},
        "strided tables": dict(segment_starts=a["segment_starts"].t().contiguous().t()),
        "no slab": dict(persisted_k=None, persisted_v=None, segment_starts=a["segment_starts"][:, :0],
                        segment_ends=a["segment_ends"][:, :0], segment_counts=torch.zeros_like(a["segment_counts"])),
        "empty slab": dict(persisted_k=a["persisted_k"][:, :0], persisted_v=a["persisted_v"][:, :0]),
        "whole number scale": dict(softmax_scale=1), "negative scale": dict(softmax_scale=-0.1),
        "requires grad": dict(q=a["q"].clone().requires_grad_()),
        "parameter": dict(current_k=torch.nn.Parameter(a["current_k"])),
        "truthy flag": dict(return_lse=1),
        # refused
        "plan without its record": dict(work_plan=plan.clone()), "plan of another length": dict(work_plan=other),
        "plan of another shape": dict(work_plan=plan[:, :4]), "q on the host": dict(q=a["q"].cpu()),
        "tables on the host": dict(segment_counts=a["segment_counts"].cpu()), "mode": dict(softmax_mode="softmax"),
        "mixed q and k": dict(q=a["q"].half()), "slab of another type": dict(persisted_k=a["persisted_k"].half()),
        "shape": dict(current_k=a["current_k"][:, :, :20]), "out type": dict(out_dtype=torch.float64),
        "slab batch": dict(persisted_k=a["persisted_k"][:1], persisted_v=a["persisted_v"][:1]),
        "no queries": {k: a[k][:, :, :0] for k in ("q", "current_k", "current_v")},
        "head dim": {k: a[k][..., :64] for k in ("q", "current_k", "current_v", "persisted_k", "persisted_v")},
        "split rows of bf16": dict(k_split_rows=True), "counts": dict(segment_counts=a["segment_counts"][:2]),
        "double": {k: a[k].double() for k in ("q", "current_k", "persisted_k")},
    }


def test_attention_other_calls_match_the_body(device):
    for name, change in _changes(device).items():
        print(f"[op_call] {name}", flush=True)
        a = dict(attention_args(device), **change)
        got, want = (public(fused_real_pruning_flat_segmented_attention, **a),
                     body(fused_real_pruning_flat_segmented_attention, **a))
        torch.cuda.synchronize(device)
        assert same(got, want), name


@pytest.mark.parametrize("knob,value", [("REAL_PRUNING_FUSED_QK_DOT_MODE", "fp32"), ("HKV_ATTN_SPLIT", "0"),
                                        ("REAL_PRUNING_FUSED_VALUE_DOT_MODE", "bad"), ("HKV_ATTN_SPLIT_ROWS", "0")])
def test_knobs_are_read_at_each_call(device, knob, value, monkeypatch):
    a = attention_args(device, (F32, F32, BF))
    assert native(a) is not None
    monkeypatch.setenv(knob, value)
    assert native(a) is None
    assert same(public(fused_real_pruning_flat_segmented_attention, **a),
                body(fused_real_pruning_flat_segmented_attention, **a))
    monkeypatch.delenv(knob)
    assert native(a) is not None


def test_modes_streams_and_capture_are_left_to_the_body(device):
    a = attention_args(device)
    want = body(fused_real_pruning_flat_segmented_attention, **a)

    class Count(torch.overrides.TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Count.seen += 1
            return func(*args, **(kwargs or {}))

    with Count():
        assert native(a) is None
        assert same(fused_real_pruning_flat_segmented_attention(**a), want)
    assert Count.seen > 0
    with torch.inference_mode():
        assert fused_real_pruning_flat_segmented_attention(**a).is_inference()
    side = torch.cuda.Stream(device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        first = fused_real_pruning_flat_segmented_attention(**a)  # the stream's first call: the body
        assert native(a) is not None
        second = fused_real_pruning_flat_segmented_attention(**a)
    side.synchronize()
    assert same(first, want) and same(second, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert native(a) is None
        out = fused_real_pruning_flat_segmented_attention(**a)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize(device)
        assert same(out, want)
        assert same(fused_real_pruning_flat_segmented_attention(**a), want)


@pytest.mark.parametrize("proj,qk,k_split,append", [(BF, F32, True, True), (BF, F32, False, False), (F32, F32, False, True),
                                                    (FP, FP, False, True), (BF, BF, False, False)])
def test_produce_taken(device, proj, qk, k_split, append):
    B, L, H = 2, 37, 3
    g = torch.Generator().manual_seed(9)
    qkv = torch.randn((B, L, 3 * H * D), generator=g).to(proj).to(device)
    kw = dict(scale_mul=torch.rand(H, generator=g).to(device), rope_table=rope2d_freqs_table(D, [(1, 7, 7)]).to(device),
              rope_start_row=3, qk_dtype=qk, k_split_rows=k_split)

    def slab():
        return (torch.zeros((B, 200, D), device=device, dtype=qk), torch.zeros((B, 200, D), device=device, dtype=proj),
                torch.tensor([100, -1, 4], dtype=torch.int32, device=device))

    s1, s2 = (slab(), slab()) if append else (None, None)
    got = _lib.op_call.produce(qkv, H, kw["scale_mul"], kw["rope_table"], 3, True, 1e-12, qk, s1, k_split)
    assert got is not None
    want = body(qkv_produce, qkv, H, append=s2, **kw)
    torch.cuda.synchronize(device)
    assert same(got, want) and same(s1, s2)
    assert same(public(qkv_produce, qkv.view(B, L, 3, H, D), H, **kw), want)
    for change in (dict(rope_table=kw["rope_table"].double()), dict(scale_mul=kw["scale_mul"].view(1, H, 1, 1)),
                   dict(rope_start_row=13), dict(scale_mul=kw["scale_mul"][:2]), dict(qk_dtype=torch.float64),
                   dict(rope_table=kw["rope_table"].cpu()), dict(k_split_rows=True, qk_dtype=FP)):
        c = dict(kw, **change)
        assert same(public(qkv_produce, qkv, H, **c), body(qkv_produce, qkv, H, **c)), change


def test_pack_taken(device):
    g = torch.Generator().manual_seed(2)
    src = [torch.randn((2, 70, D), generator=g).to(device).to(t) for t in (F32, BF)]
    meta = [torch.tensor(x, device=device) for x in ([0, 40], [3, 30], [20, 33])]

    def run(fn, slab, **kw):
        return fn(pack_flat_segments_kv, **dict(dict(dst_k=slab[0], dst_v=slab[1], src_k=src[0], src_v=src[1],
                                                     dst_starts=meta[0], src_starts=meta[1], lengths=meta[2],
                                                     max_length=33), **kw))

    def slab():
        return [torch.zeros((2, 90, D), device=device, dtype=t) for t in (F32, BF)]

    assert _lib.op_call.pack(*slab(), *src, *meta, 33, 32) is True
    for kw in ({}, dict(max_length=10), dict(max_length=None), dict(block_t=1, max_length=5), dict(max_length=0),
               dict(block_t=0), dict(lengths=meta[2].int()), dict(lengths=meta[2][:1]), dict(src_k=src[0].half()),
               dict(src_k=src[0][:, :60]), dict(lengths=meta[2].cpu()),
               dict(src_k=src[0].transpose(1, 2).contiguous().transpose(1, 2)),
               dict(dst_starts=meta[0][:0], src_starts=meta[1][:0], lengths=meta[2][:0])):
        a, b = slab(), slab()
        got, want = run(public, a, **kw), run(body, b, **kw)
        torch.cuda.synchronize(device)
        assert same(got, want) and same(tuple(a), tuple(b)), kw
