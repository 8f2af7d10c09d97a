"""Slab pack at the edges of its 16-row chunks and of its grid."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from heatkv_amd import pack_flat_segments_kv
from oracle import pack as opack
from support import bits

pytestmark = pytest.mark.gpu


# Among them: a list uneven enough for 64-row chunks (33 items x 700 rows against
# 1388 that move) and one that is not (33 x 130 against 930).
# The last two: so many items that 16-row chunks would pass the launch grid
# (64-row chunks run: 66000 x 256 chunks of 16 rows), and 2-byte units.
@pytest.mark.parametrize("lengths,D,max_length", [
    ([1, 15, 16, 17, 31, 32, 33, 64, 65], 128, 65), ([2], 128, 2), ([47, 0, 48], 128, 48),
    ([700] + [1, 3, 17, 65] * 8, 128, 700), ([130] + [1, 3, 31, 65] * 8, 128, 130),
    ([5, 70, 16, 64, 4000, 65] + [0] * 66000 + [17, 130], 6, 4096), ([17, 16, 3], 5, 17)])
@pytest.mark.parametrize("kdt,vdt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16)])
def test_pack_chunk_edges(lengths, D, max_length, kdt, vdt, device):
    print(f"[pack] chunk edges {lengths[:9]} D={D} max_length={max_length} {kdt} {vdt}", flush=True)
    gen = torch.Generator().manual_seed(3)
    B, src_rows, cap = 2, sum(lengths) + 7, sum(lengths) + 11
    src = [torch.randn((B, src_rows, D), generator=gen).to(t) for t in (kdt, vdt)]
    dst = [torch.randn((B, cap, D), generator=gen).to(t) for t in (kdt, vdt)]
    src_starts = np.concatenate(([4], 4 + np.cumsum(lengths)[:-1])).tolist()
    dst_starts = np.concatenate(([3], 3 + np.cumsum(lengths)[:-1])).tolist()
    got = [t.clone().to(device) for t in dst]
    meta = [torch.tensor(x, dtype=torch.int64, device=device) for x in (dst_starts, src_starts, lengths)]
    pack_flat_segments_kv(dst_k=got[0], dst_v=got[1], src_k=src[0].to(device), src_v=src[1].to(device),
                          dst_starts=meta[0], src_starts=meta[1], lengths=meta[2], max_length=max_length)
    torch.cuda.synchronize(device)
    for g, d, s in zip(got, dst, src):
        want = opack.pack_flat_segments(d.clone(), s, dst_starts, src_starts, lengths)
        assert np.array_equal(bits(g), bits(want))
