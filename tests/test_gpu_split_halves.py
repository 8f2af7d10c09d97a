"""The split-row kernel's two forms, 128-query halves (small launches, fp32 V)
and 256-query workgroups (large ones), against the oracle at the sizes where
they can go wrong: lengths around the 32-key halves, 64-key tiles and 128- and
256-query items, empty and full tables, planned (items cut in two) and not,
with and without the workspace, the fused append, and tensors that do not
start on a 16-byte boundary."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import heatkv_amd.real_pruning_fused_attention as op
from heatkv_amd import attention_item_shape, fused_real_pruning_flat_segmented_attention, segmented_attention_plan
from oracle import segmented_attention as oattn
from support import assert_attention_close, to_np

pytestmark = pytest.mark.gpu

SCALE = 1.0 / np.sqrt(128.0)


def make(seed, B, H, L, cap, S, vdtype):
    """fp32 q and k (N(0, 1): scores of O(1) to O(4)), v of ``vdtype``, and
    disjoint segments: head h owns rows of the slab, cut at random, some empty."""
    g = torch.Generator().manual_seed(seed)
    q, ck, cv = (torch.randn((B, H, L, 128), generator=g) for _ in range(3))
    sk, sv = (torch.randn((B, cap, 128), generator=g) for _ in range(2))
    st = torch.zeros((H, S), dtype=torch.int32)
    en = torch.zeros((H, S), dtype=torch.int32)
    ct = torch.zeros((H,), dtype=torch.int32)
    own = cap // H if H else 0
    for h in range(H):
        n = int(torch.randint(0, S + 1, (1,), generator=g)) if S and own else 0
        cuts = sorted(int(x) for x in torch.randint(0, own + 1, (2 * n,), generator=g))
        for i in range(n):
            st[h, i], en[h, i] = h * own + cuts[2 * i], h * own + cuts[2 * i + 1]
        ct[h] = n
    return q, sk, sv.to(vdtype), (st, en, ct), ck, cv.to(vdtype)


def reference(q, sk, sv, tables, ck, cv):
    return oattn.flat_segmented_attention(
        *(to_np(t).astype(np.float64) for t in (q, sk, sv)), *(t.numpy() for t in tables),
        *(to_np(t).astype(np.float64) for t in (ck, cv)), SCALE, dtype=np.float64, workers=16)


def call(device, q, sk, sv, tables, ck, cv, **kw):
    st, en, ct = (t.to(device) for t in tables)
    return fused_real_pruning_flat_segmented_attention(
        q=q.to(device), persisted_k=sk.to(device), persisted_v=sv.to(device), segment_starts=st, segment_ends=en,
        segment_counts=ct, current_k=ck.to(device), current_v=cv.to(device), softmax_scale=float(SCALE), **kw)


def check(out, lse, ref_out, ref_lse, q, ck, cv, vdtype, what):
    if vdtype != torch.float32:
        assert_attention_close(to_np(out), to_np(lse), ref_out, ref_lse, what=what)
        return
    # Two bf16 pieces leave 2^-16 of an operand, so a product of two carries at
    # most 3 * 2^-16 of |q||k| (the dropped low-low product included); a score
    # off by d moves every weight by a factor within e^{2d}, and the P V
    # product adds its own 3 * 2^-16 of max |v|.
    unit = 3.0 * 2.0 ** -16
    d = unit * SCALE * float(q.norm(dim=-1).max() * ck.norm(dim=-1).max())
    bound = (2.0 * d + unit) * float(cv.abs().max()) * 1.3  # slab rows are drawn alike: a little longer than the current ones
    err = np.abs(to_np(out).astype(np.float64) - ref_out).max()
    assert err <= bound, f"{what}: {err:.2e} > {bound:.2e}"
    assert np.abs(to_np(lse).astype(np.float64) - ref_lse).max() <= 1.3 * d + 1e-5, what


# (B, H, L, cap, S): halves of items around every boundary ...
SMALL = [(1, 1, 1, 0, 0), (2, 3, 31, 64, 3), (1, 4, 32, 500, 2), (2, 3, 33, 900, 4), (1, 5, 64, 333, 1),
         (2, 2, 65, 700, 5), (1, 3, 127, 400, 3), (2, 3, 128, 5000, 6), (1, 2, 129, 2000, 40), (3, 2, 256, 3000, 4),
         (1, 3, 257, 100, 2), (2, 5, 700, 6000, 7)]
# ... and more 256-query items than CUs: the 256-query form
LARGE = [(2, 65, 400, 6500, 3), (2, 131, 250, 1310, 2)]


@pytest.mark.parametrize("vdtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", SMALL + LARGE, ids=lambda s: "x".join(map(str, s)))
def test_split_forms_against_fp64(shape, vdtype, device, monkeypatch):
    monkeypatch.setattr(op, "_SPLIT_VALUES_ROWS", 0)  # fp32 V: the split kernel at every size
    B, H, L, cap, S = shape
    case = make(500 + L, B, H, L, cap, S, vdtype)
    ref_out, ref_lse = reference(*case)
    q, ck, cv, tables = case[0], case[4], case[5], case[3]
    qpi, slots = attention_item_shape(torch.float32, torch.float32, vdtype, device=device)
    for name, plan_slots, ws in (("planned", slots, "1"), ("cut", 4 * slots, "1"), ("no workspace", slots, "0"),
                                 ("unplanned", None, "1")):
        monkeypatch.setenv("HKV_ATTN_SPLIT", ws)
        print(f"[attn] split forms {shape} v={vdtype} {name}", flush=True)
        plan = (None if plan_slots is None else
                segmented_attention_plan(*tables, batch_size=B, current_len=L, capacity=cap, device=device,
                                         queries_per_item=qpi, slots=plan_slots))
        out, lse = call(device, *case, work_plan=plan, return_lse=True, out_dtype=torch.float32)
        torch.cuda.synchronize(device)
        check(out, lse, ref_out, ref_lse, q, ck, cv, vdtype, f"{shape} {name}")


@pytest.mark.parametrize("L", [40, 300])
def test_fp32_values_append_and_misaligned_rows(L, device, monkeypatch):
    """The fp32 call's append writes the fp32 rows themselves, to both
    destinations, and leaves every other row; rows that start off a 16-byte
    boundary give the same bits."""
    monkeypatch.setattr(op, "_SPLIT_VALUES_ROWS", 0)
    B, H, cap = 2, 3, 1500
    q, sk, sv, tables, ck, cv = (t.to(device) if isinstance(t, torch.Tensor) else t
                                 for t in make(77, B, H, L, 600, 3, torch.float32))
    grow = torch.full((B, cap - 600, 128), 7.0, device=device)
    slab_k, slab_v = torch.cat((sk, grow), dim=1), torch.cat((sv, grow), dim=1)
    plain, lse = call(device, q, slab_k, slab_v, tables, ck, cv, return_lse=True)
    offs = torch.tensor([600, -1, 600 + L], dtype=torch.int32, device=device)
    offs2 = torch.tensor([-1, 0, L], dtype=torch.int32, device=device)
    k1, v1 = slab_k.clone(), slab_v.clone()
    k2, v2 = (torch.zeros((B, 2 * L, 128), device=device) for _ in range(2))
    st, en, ct = (t.to(device) for t in tables)
    out = fused_real_pruning_flat_segmented_attention(
        q=q, persisted_k=k1, persisted_v=v1, segment_starts=st, segment_ends=en, segment_counts=ct, current_k=ck,
        current_v=cv, softmax_scale=float(SCALE), append_offsets=offs, append_also=(k2, v2, offs2))
    torch.cuda.synchronize(device)
    assert torch.equal(out, plain)
    for got, want, cur in ((k1, slab_k.clone(), ck), (v1, slab_v.clone(), cv)):
        want[:, 600:600 + L] = cur[:, 0]
        want[:, 600 + L:600 + 2 * L] = cur[:, 2]
        assert torch.equal(got, want)
    for got, cur in ((k2, ck), (v2, cv)):
        assert torch.equal(got, torch.cat((cur[:, 1], cur[:, 2]), dim=1))

    def off_boundary(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=device)
        buf[1:] = t.reshape(-1)
        return buf[1:].view(t.shape)

    moved = [off_boundary(t) for t in (q, slab_k, slab_v, ck, cv)]
    assert all(t.data_ptr() % 16 for t in moved)
    out2, lse2 = call(device, moved[0], moved[1], moved[2], tables, moved[3], moved[4], return_lse=True)
    torch.cuda.synchronize(device)
    assert torch.equal(out2, plain) and torch.equal(lse2, lse)
