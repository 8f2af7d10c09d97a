"""The mixed tile of the 16-bit kernels (128-query items, and 64-query items for
few queries without cut items) and the split-row kernel: the last current rows and the first prior
rows in one 64-key tile, at lengths and retained rows around the tile's edge,
planned (whole, cut) and not, against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import heatkv_amd.real_pruning_fused_attention as op
from heatkv_amd import attention_item_shape, fused_real_pruning_flat_segmented_attention, segmented_attention_plan
from oracle import segmented_attention as oattn
from support import assert_attention_close, to_np

pytestmark = pytest.mark.gpu
SCALE = float(1.0 / np.sqrt(128.0))


@pytest.mark.parametrize("qk,vt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                   (torch.float32, torch.bfloat16), (torch.float32, torch.float32)], ids=str)
@pytest.mark.parametrize("L", [1, 8, 16, 31, 33, 63, 64, 65, 120, 128, 129, 191, 192, 193, 639, 641])
def test_mixed_tile_against_oracle(L, qk, vt, device, monkeypatch):
    monkeypatch.setattr(op, "_SPLIT_VALUES_ROWS", 0)  # fp32 v: the split-row kernel at every size
    # per head: no prior rows, one, those that fill the tile less one / exactly
    # / plus one, a whole tile more, and many, in segments of uneven length
    rest = 64 - L % 64
    rows = [0, 1, rest - 1, rest, rest + 1, rest + 64, 700]
    H, B = len(rows), 2
    st, en, at = torch.zeros((H, 3), dtype=torch.int32), torch.zeros((H, 3), dtype=torch.int32), 3
    for h, n in enumerate(rows):
        cuts = [0, n // 3, n // 3 + n // 5, n]
        for i in range(3):
            st[h, i], en[h, i] = at, at + cuts[i + 1] - cuts[i]
            at += cuts[i + 1] - cuts[i] + 2  # rows of no segment between
    ct = torch.full((H,), 3, dtype=torch.int32)
    g = torch.Generator().manual_seed(L)
    q, ck, cv = (torch.randn((B, H, L, 128), generator=g).to(t) for t in (qk, qk, vt))
    sk, sv = (torch.randn((B, at, 128), generator=g).to(t) for t in (qk, vt))
    live = torch.zeros(at, dtype=torch.bool)
    for s, e in zip(st.flatten().tolist(), en.flatten().tolist()):
        live[s:e] = True
    sk[:, ~live], sv[:, ~live] = float("nan"), float("nan")  # never read
    want = oattn.flat_segmented_attention(*(to_np(t.float()) for t in (q, sk.nan_to_num(), sv.nan_to_num())),
                                          st.numpy(), en.numpy(), ct.numpy(),
                                          *(to_np(t.float()) for t in (ck, cv)), SCALE)
    dev = [t.to(device) for t in (q, sk, sv, st, en, ct, ck, cv)]
    queries, resident = attention_item_shape(qk, qk, vt, device=device)
    outs = {}
    for name, slots in (("unplanned", None), ("planned", 1), ("cut", 16), ("whole", 0)):
        print(f"[attn] mixed tile L={L} {qk} {vt} {name}", flush=True)
        plan = None if slots is None else segmented_attention_plan(
            st, en, ct, batch_size=B, current_len=L, capacity=at, device=device, queries_per_item=queries,
            slots=slots * resident)
        out, lse = fused_real_pruning_flat_segmented_attention(
            q=dev[0], persisted_k=dev[1], persisted_v=dev[2], segment_starts=dev[3], segment_ends=dev[4],
            segment_counts=dev[5], current_k=dev[6], current_v=dev[7], softmax_scale=SCALE, return_lse=True,
            work_plan=plan)
        torch.cuda.synchronize(device)
        assert_attention_close(to_np(out.float()), to_np(lse), *want, what=f"L={L} {name}")
        outs[name] = out
    assert torch.isfinite(outs["unplanned"].float()).all()
