"""GPU parity of the fp32-key indexer's matrix-core path (IC 64 / 128, up to 16 heads, k up to 1024)
against the oracle and against the generic kernels.

Bar as tests/test_gpu_indexer.py: the oracle's top-k up to entries within the fp32 rounding bound of the
k-th score.  Scores against the generic kernel's: both are fp32 sums of at most IC products per head
in different orders, so within twice 4 IC 2^-24 of the sum of magnitudes.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import aetherkv._lib as L
import oracle as O
from aetherkv import csa_indexer_topk
from test_gpu_indexer import w_act
from topk_check import assert_topk_matches, score_error_bound

pytestmark = pytest.mark.gpu


def _inputs(seed, B, S, IH, IC):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(B, IH, IC, generator=g), torch.randn(B, S, IC, generator=g), torch.randn(B, IH, generator=g) * 2


# partial and whole 16-key slots and 64-key groups, 1 to 16 heads (one to four per lane group), both head widths
@pytest.mark.parametrize("mode", ["softplus", "raw", "relu_w"])
@pytest.mark.parametrize("IH,IC,S,k", [(1, 64, 15, 15), (4, 64, 65, 64), (5, 64, 1000, 256), (16, 64, 4099, 512),
                                       (4, 128, 16, 1), (12, 128, 2050, 1024)])
def test_shapes_match_oracle(dev, mode, IH, IC, S, k):
    q, kv, w = _inputs(S + IH, 3, S, IH, IC)
    idx = csa_indexer_topk(q.to(dev), kv.to(dev), w.to(dev), k, mode=mode).cpu().numpy()
    scores = O.index_scores(q.numpy(), w.numpy(), kv.numpy(), mode=mode)
    assert_topk_matches(idx, scores, k, score_error_bound(q.numpy(), w_act(w.numpy(), mode), kv.numpy()))


def _call(dev, q, kv, w, valid, k, mode, generic):
    B, IH, IC = q.shape
    S = kv.size(1)
    lib = L.lib()
    out = torch.empty(B, k, dtype=torch.int64, device=dev)
    sc = torch.empty(B, k, dtype=torch.float32, device=dev)
    ws = torch.full((lib.aekv_csa_indexer_workspace_size(B, S, k),), 0xA5, dtype=torch.uint8, device=dev)
    old = lib.aekv_set_generic_kernels(1 if generic else 0)
    try:
        with torch.cuda.device(dev):
            L.check(lib.aekv_csa_indexer_topk(L.ptr(q), L.ptr(kv), L.ptr(w), L.ptr(valid), B, S, IH, IC, k, mode,
                                              L.ptr(ws), ws.numel(), L.ptr(out), L.ptr(sc), L.stream_of(q)), "indexer")
    finally:
        lib.aekv_set_generic_kernels(old)
    torch.cuda.synchronize()
    return out.cpu(), sc.cpu()


# visible counts at slot edges; B * S large enough for two groups per wave; rows past their count padded
@pytest.mark.parametrize("B,S,k,valid", [(6, 700, 64, [0, 1, 16, 17, 699, 5000]), (20, 65537, 256, None)])
def test_counts_and_scores_match_generic(dev, B, S, k, valid):
    g = torch.Generator(device=dev).manual_seed(B)
    q, w = torch.randn(B, 4, 64, generator=g, device=dev), torch.randn(B, 4, generator=g, device=dev)
    kv = torch.randn(B, S, 64, generator=g, device=dev)
    v = None if valid is None else torch.tensor(valid, dtype=torch.int32, device=dev)
    idx, sc = _call(dev, q, kv, w, v, k, 0, False)
    idx_g, sc_g = _call(dev, q, kv, w, v, k, 0, True)
    n = torch.full((B,), k) if valid is None else torch.tensor(valid).clamp(0, min(k, S))
    pad = torch.arange(k)[None] >= n[:, None]
    assert bool((idx[pad] == -1).all()) and bool((idx_g[pad] == -1).all())
    # |q| |k| <= 64 * 5^2 per head, weights below 8: the magnitudes sum to less than 64 * 25 * 4 * 8 / 8
    torch.testing.assert_close(sc[~pad], sc_g[~pad], rtol=0, atol=2 * 4 * 64 * 2.0 ** -24 * 400)
    same = torch.tensor([len(set(a.tolist()) ^ set(b.tolist())) for a, b in zip(idx, idx_g)])
    assert int(same.max()) <= 2  # at most one entry of a row exchanged with a near tie at the k-th place


def test_infinite_keys_and_ties(dev):
    # absent heads' products meet infinite keys as 0 * inf and must not enter; equal keys resolve to the lower index
    q, kv, w = _inputs(3, 1, 400, 3, 64)
    kv[0, 37, 5], kv[0, 38, 6] = float("inf"), float("-inf")
    kv[0, 100:200] = kv[0, 100]
    for mode in (0, 1, 2):
        a, _ = _call(dev, q.to(dev), kv.to(dev), w.to(dev), None, 300, mode, False)
        b, _ = _call(dev, q.to(dev), kv.to(dev), w.to(dev), None, 300, mode, True)
        tied = [i for i in a[0].tolist() if 100 <= i < 200]
        assert tied == sorted(tied)
        assert len(set(a[0].tolist()) ^ set(b[0].tolist())) <= 2
        assert (37 in a[0]) == (37 in b[0]) and (38 in a[0]) == (38 in b[0])


def test_misaligned_keys_are_accepted(dev):
    q, kv, w = _inputs(9, 2, 300, 4, 64)
    flat = torch.empty(kv.numel() + 1, device=dev)
    view = flat[1:].view(kv.shape)
    view.copy_(kv)
    a = csa_indexer_topk(q.to(dev), view, w.to(dev), 32)
    b = csa_indexer_topk(q.to(dev), kv.to(dev), w.to(dev), 32)
    assert len(set(a[0].tolist()) ^ set(b[0].tolist())) <= 2


# More equal keys than a row's workgroup collects: the passes over all stored keys, whose parts per wave
# end inside, at and past the row (4 keys per lane, 256 per wave step).  All scores are zero except a few
# larger ones scattered over the parts: those come first, then the lowest indices.
@pytest.mark.parametrize("S,k,top", [(65536, 256, [65535, 7, 40000]), (16387, 1000, []), (60001, 300, [60000, 59999])])
def test_many_equal_scores(dev, S, k, top):
    q = torch.zeros(2, 4, 64)
    q[:, :, 0] = 1.0
    kv = torch.zeros(2, S, 64)
    for n, j in enumerate(top):
        kv[:, j, 0] = float(len(top) - n)
    w = torch.ones(2, 4)
    idx = csa_indexer_topk(q.to(dev), kv.to(dev), w.to(dev), k, mode="raw").cpu()
    want = (top + [j for j in range(k + len(top)) if j not in top])[:k]
    assert idx.tolist() == [want, want]


# Rows with fewer 16-key slots than k and more keys than a workgroup collects: every stored key is counted.
# Whole-number scores, so that the selection is exact: mostly distinct ones, a few hundred values, and a few
# values (where whole waves meet in one bin).  1024 rows take the 512-thread select (1536 candidates), 2 rows
# the 1024-thread one (4096).
@pytest.mark.parametrize("B,S,k", [(1024, 1537, 256), (1024, 2049, 129), (1024, 3001, 200), (1024, 2047, 512),
                                   (2, 4097, 1024), (2, 8190, 513), (2, 16383, 1024)])
@pytest.mark.parametrize("values", [1 << 20, 300, 3])
def test_fewer_slots_than_k(dev, B, S, k, values):
    g = torch.Generator(device=dev).manual_seed(S + values)
    s = torch.randint(-values // 8, values, (B, S), generator=g, device=dev).float()
    s[0] = s[0].sort().values  # (ordered along the row: whole waves above or below the k-th key)
    kv = torch.zeros(B, S, 64, device=dev)
    kv[:, :, 5] = s
    q = torch.zeros(B, 1, 64, device=dev)
    q[:, :, 5] = 1.0
    idx = csa_indexer_topk(q, kv, torch.ones(B, 1, device=dev), k, mode="relu_w")
    want = s.sort(dim=1, descending=True, stable=True).indices[:, :k]
    assert torch.equal(idx, want)
