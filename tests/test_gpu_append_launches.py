"""The append inside the attention launches, at the lines between kernels: small
16-bit launches (64-query workgroups, as far as the CUs and the copy blocks
allow) and the split-row kernel's 128- and 256-query forms, planned (whole and
cut items) and not, one and two destinations: the attention against the oracle,
the written rows exactly and every other row untouched."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from heatkv_amd import attention_item_shape, fused_real_pruning_flat_segmented_attention, segmented_attention_plan
from heatkv_amd.real_pruning_fused_attention import _split_rows
from oracle import segmented_attention as oattn
from support import assert_attention_close, to_np

pytestmark = pytest.mark.gpu
SCALE = float(1.0 / np.sqrt(128.0))


def check_append(device, B, H, L, qk, kept, dests, plans):
    """``kept``: retained rows of head h, ``plans``: name -> slots per resident
    workgroup (None: no plan).  fp32 q and k: K as split rows."""
    split = qk == torch.float32
    g = torch.Generator().manual_seed(L * 31 + H)
    rows = [kept(h) for h in range(H)]
    first = np.concatenate(([0], np.cumsum(rows))).astype(np.int32)
    used = int(first[-1])
    st, en = (torch.from_numpy(a.copy()).reshape(H, 1) for a in (first[:-1], first[1:]))
    ct = torch.ones(H, dtype=torch.int32)
    # the first destination takes every third head, the second the others and one of those again
    offs, offs2 = (torch.full((H,), -1, dtype=torch.int32) for _ in range(2))
    for i, h in enumerate(range(0, H, 3)):
        offs[h] = used + i * L
    others = [0] + [h for h in range(H) if h % 3]
    for i, h in enumerate(others):
        offs2[h] = i * L
    cap, cap2 = used + -(-H // 3) * L, len(others) * L
    q, ck, cv = (torch.randn((B, H, L, 128), generator=g).to(t) for t in (qk, qk, torch.bfloat16))
    sk, sv = (torch.randn((B, cap, 128), generator=g).to(t) for t in (qk, torch.bfloat16))
    want = oattn.flat_segmented_attention(*(to_np(t.float()) for t in (q, sk, sv)), st.numpy(), en.numpy(), ct.numpy(),
                                          *(to_np(t.float()) for t in (ck, cv)), SCALE, workers=16)
    q, ck, cv, sk, sv = (t.to(device) for t in (q, ck, cv, sk, sv))
    if split:
        stream = torch.cuda.current_stream(device)
        ck, sk = (_split_rows(t, stream).view(torch.float32) for t in (ck, sk))
    qpi, slots = attention_item_shape(qk, qk, torch.bfloat16, k_split_rows=split, device=device)
    bits = lambda t: t.view(torch.int32) if t.dtype == torch.float32 else t.view(torch.int16)  # noqa: E731
    for name, share in plans.items():
        print(f"[attn] append B={B} H={H} L={L} {qk} {dests} destinations {name}", flush=True)
        plan = None if share is None else segmented_attention_plan(
            st, en, ct, batch_size=B, current_len=L, capacity=cap, device=device, queries_per_item=qpi,
            slots=share * slots)
        k1, v1 = sk.clone(), sv.clone()
        k2 = torch.full((B, cap2, 128), 7.0, device=device, dtype=qk)
        v2 = torch.full((B, cap2, 128), 7.0, device=device, dtype=torch.bfloat16)
        out, lse = fused_real_pruning_flat_segmented_attention(
            q=q, persisted_k=k1, persisted_v=v1, segment_starts=st.to(device), segment_ends=en.to(device),
            segment_counts=ct.to(device), current_k=ck, current_v=cv, softmax_scale=SCALE, return_lse=True,
            work_plan=plan, append_offsets=offs.to(device), k_split_rows=split,
            append_also=(k2, v2, offs2.to(device)) if dests == 2 else None)
        torch.cuda.synchronize(device)
        assert_attention_close(to_np(out.float()), to_np(lse), *want, what=f"L={L} {name}")
        pairs = [(k1, sk.clone(), ck, offs), (v1, sv.clone(), cv, offs)]
        if dests == 2:
            pairs += [(k2, torch.full_like(k2, 7.0), ck, offs2), (v2, torch.full_like(v2, 7.0), cv, offs2)]
        for got, rest, cur, at in pairs:
            for h in range(H):
                if at[h] >= 0:
                    rest[:, at[h]:at[h] + L] = cur[:, h]
            assert torch.equal(bits(got), bits(rest)), name


# copy blocks (16 rows each) against the CUs that the 64-query workgroups leave:
# 256 workgroups (none left), just within and past 16 copies a CU, a plan of
# 128-query units with a half-empty last one in each item, and more workgroups
# than CUs with such units
@pytest.mark.parametrize("B,H,L,dests", [(8, 32, 4, 1), (8, 32, 64, 2), (6, 30, 36, 2), (6, 30, 64, 1), (6, 30, 64, 2),
                                         (5, 16, 128, 2), (3, 16, 144, 2), (4, 16, 144, 1), (5, 16, 192, 1),
                                         (2, 5, 65, 2), (1, 3, 192, 2), (1, 2, 193, 1)])
def test_small_launches_with_the_append(B, H, L, dests, device):
    check_append(device, B, H, L, torch.bfloat16, lambda h: (h * 13) % 40, dests, {"planned": 1, "unplanned": None})


# 128-query form (plan units of 256 queries as two workgroups, the last one empty
# at L % 256 in 1 .. 128), then past its two lines: 2560 tokens, two items a CU
@pytest.mark.parametrize("B,H,L", [(2, 3, 100), (2, 3, 300), (1, 5, 129), (2, 2, 1000), (1, 13, 2700), (4, 131, 250)])
@pytest.mark.parametrize("dests", [1, 2])
def test_split_row_launches_with_the_append(B, H, L, dests, device):
    plans = {"planned": 1, "cut": 4, "unplanned": None} if H < 10 else {"planned": 1}
    check_append(device, B, H, L, torch.float32, lambda h: (h * 97) % 700 if H < 100 else h % 7, dests, plans)
