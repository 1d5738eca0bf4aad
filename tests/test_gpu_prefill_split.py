"""HCA prefill launches whose last row blocks are split over their source tiles: against the unsplit
launch (a workspace without room for the pieces) and, where small enough, the oracle.

Tolerance: the path's 1e-2 relative / 2e-3 absolute in bf16 (split and unsplit sum the same bf16 weights
relative to different maxima, so both are within it of the oracle and of each other here)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import aetherkv._lib as L
import oracle as O
from aetherkv import PolarQuant
from aetherkv.prefill import _device_sources, prefill_workspace
from aetherkv.synthetic import normal
from conftest import to_np_f32

pytestmark = pytest.mark.gpu


def _run(q, codes, scale, counts, win, sink, pq, room):
    B, T, H, D = q.shape
    S, Wt = codes.size(1), win.size(1)
    blocks = -(-B * S * 256 // 256) * 256
    n = L.lib().aekv_quant_prefill_workspace_size(B, T, H, S, Wt) if room else blocks
    assert not room or n > blocks
    ws = torch.full((n,), 0x7F, dtype=torch.uint8, device=q.device)  # (NaN patterns: prior contents never matter)
    out = torch.empty_like(q)
    vis, _, w0, wl = counts
    with torch.cuda.device(q.device):
        L.check(L.lib().aekv_quant_prefill_attention(
            L.ptr(q), L.ptr(codes), L.ptr(scale), None, L.ptr(vis), L.ptr(win), L.ptr(w0), L.ptr(wl), L.ptr(sink),
            L.ptr(pq._diag(D, q.device)), B, T, H, D, S, -1, Wt, pq.bits, D ** -0.5, L.ptr(ws), n, L.ptr(out),
            L.stream_of(q)), "prefill")
    torch.cuda.synchronize()
    return out


# every block split (one partial round), a partial last block; two sequences; a full round (512 blocks of 64 rows)
# and a split remainder; early targets whose pieces see no tile
@pytest.mark.parametrize("B,T,H,S,start", [(1, 40, 12, 1300, 1300 * 128 - 40), (2, 33, 5, 1100, 60000), (1, 1, 12, 900, 115000),
                                           (1, 2200, 16, 1100, 138000), (1, 100, 12, 800, 0)])
def test_split_matches_unsplit(dev, B, T, H, S, start):
    print(f"B={B} T={T} H={H} S={S} start={start}", flush=True)
    pq = PolarQuant(4)
    codes, scale = pq.encode(normal((B, S, 128), 3).to(dev))
    q, win, sink = normal((B, T, H, 128), 4).to(dev), normal((B, T + 127, 128), 5).to(dev), torch.randn(H).to(dev)
    base = max(0, start - 127)
    counts = _device_sources(q, win, start, S, 128, 128, base, 0)
    old = L.lib().aekv_set_flash_rows(64)
    try:
        got, want = (_run(q, codes, scale, counts, win, sink, pq, room) for room in (True, False))
    finally:
        L.lib().aekv_set_flash_rows(old)
    torch.testing.assert_close(got.float(), want.float(), rtol=1e-2, atol=2e-3)
    if T > 100:
        return
    vis, _, w0, wl = counts.cpu().tolist()
    for b in range(B):
        for t in range(0, T, 13):
            sel = np.arange(vis[b][t], dtype=np.int64)[None]
            w = to_np_f32(win[b : b + 1, w0[b][t] : w0[b][t] + wl[b][t]])
            ref = O.quant_attention(to_np_f32(q[b : b + 1, t]), codes[b : b + 1].cpu().numpy(),
                                    scale[b : b + 1].cpu().numpy(), sel, w, to_np_f32(sink), O.diag(42, 128), 4, 128 ** -0.5)
            np.testing.assert_allclose(to_np_f32(got[b, t]), ref[0], rtol=1e-2, atol=2e-3)
