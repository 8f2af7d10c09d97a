"""All-fp32 calls against 64 bits, tightly enough that no product of the split
operands can go missing: each of q, K, P and V is two bf16 pieces, and a call
that dropped the low piece of any of them would be ~1e-3 off (2-norm, relative),
the sum of all pieces ~1e-5 (tests/test_gpu_split_halves.py bounds the largest
element by the worst case, which a dropped piece can stay under)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import heatkv_amd.real_pruning_fused_attention as op
from heatkv_amd import attention_item_shape, segmented_attention_plan
from support import to_np
from test_gpu_split_halves import SCALE, call, make, reference

# Four times the error of the two-piece products at these shapes (largest 1.4e-5, see the emulation below).
REL = 6e-5
# (B, H, L, cap, S): lengths around the 32-key halves, the tiles and 128-query
# items, on both sides of the mixed tile's limit of 640 rows
SHAPES = [(2, 3, 31, 64, 3), (1, 4, 32, 500, 2), (2, 3, 33, 900, 4), (2, 2, 65, 700, 5), (1, 3, 127, 400, 3),
          (2, 3, 128, 5000, 6), (1, 2, 129, 2000, 40), (1, 3, 257, 100, 2), (1, 2, 639, 900, 3), (1, 2, 641, 900, 3),
          (1, 3, 672, 0, 0)]


def relative(out, want):
    return float(np.linalg.norm(out.astype(np.float64) - want) / np.linalg.norm(want))


def pieces(x, low):
    hi = x.bfloat16().float()
    return hi, (x - hi).bfloat16().float() if low else torch.zeros_like(x)


def product(a, b):
    """a b^T of two-piece operands without the low-low product."""
    return a[0] @ b[0].mT + a[1] @ b[0].mT + a[0] @ b[1].mT


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_a_dropped_piece_would_show(shape):
    B, H, L, cap, S = shape
    q, sk, sv, tables, ck, cv = case = make(900 + L, B, H, L, cap, S, torch.float32)
    want, _ = reference(*case)

    def emulated(dropped):
        out = torch.empty((B, L, H, 128))
        for h in range(H):
            rows = [r for i in range(int(tables[2][h])) for r in range(int(tables[0][h, i]), int(tables[1][h, i]))]
            k, v = (torch.cat((c[:, h], s[:, rows]), dim=1) for c, s in ((ck, sk), (cv, sv)))
            s = product(pieces(q[:, h], dropped != "q"), pieces(k, dropped != "k")) * SCALE
            p = torch.exp(s - s.amax(dim=-1, keepdim=True))
            o = product(pieces(p, dropped != "p"), pieces(v.mT, dropped != "v"))
            out[:, :, h] = o / p.sum(dim=-1, keepdim=True)
        return relative(out.reshape(B, L, H * 128).numpy(), want)

    assert emulated(None) <= REL / 2
    for piece in "qkpv":
        assert emulated(piece) > 4 * REL, piece


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_fp32_values_relative_error(shape, device, monkeypatch):
    monkeypatch.setattr(op, "_split_values_pays", lambda *a: True)  # the split-row kernel at every size
    monkeypatch.setattr(op._lib, "op_call", None)  # (the native path has the rule's own copy)
    B, H, L, cap, S = shape
    case = make(900 + L, B, H, L, cap, S, torch.float32)
    want, want_lse = reference(*case)
    qpi, slots = attention_item_shape(torch.float32, torch.float32, torch.float32, device=device)
    for name, plan_slots in (("planned", slots), ("cut", 4 * slots), ("unplanned", None)):
        print(f"[attn] fp32 values {shape} {name}", flush=True)
        plan = (None if plan_slots is None else
                segmented_attention_plan(*case[3], batch_size=B, current_len=L, capacity=cap, device=device,
                                         queries_per_item=qpi, slots=plan_slots))
        out, lse = call(device, *case, work_plan=plan, return_lse=True)
        torch.cuda.synchronize(device)
        assert relative(to_np(out), want) <= REL, name
        # scores of O(4) with the same relative error, and a 32-bit logarithm of O(8)
        assert np.abs(to_np(lse) - want_lse).max() <= 5 * REL, name
