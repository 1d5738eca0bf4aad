"""Split workspaces of the drop-in attention calls (aetherkv._lib.workspace) under graph capture.

A captured call keeps its buffer's address for every replay, so the buffer must be the graph's own:
not the one that the eager calls of the same stream share and replace when a larger call comes.
"""
from __future__ import annotations

import pytest
import torch

import aetherkv._lib as L
from aetherkv import sparse_sink_attention, tiled_prefill_attention
from aetherkv.decode import attention_workspace, decode_workspace, indexer_workspace


def test_captured_calls_get_buffers_of_their_own(monkeypatch):
    monkeypatch.setattr(L, "_ws_cache", {})
    capturing = [False]
    monkeypatch.setattr(L, "_capturing", lambda: capturing[0])
    cpu = torch.device("cpu")
    eager = L.workspace(1000, cpu, 7)
    assert L.workspace(600, cpu, 7) is eager  # reused
    capturing[0] = True  # on the stream that was warmed up, with a sufficient buffer there
    captured = [L.workspace(600, cpu, 7) for _ in range(2)]
    capturing[0] = False
    grown = L.workspace(5000, cpu, 7)  # replaces the cached buffer
    ptrs = {t.data_ptr() for t in (eager, grown, *captured)}
    assert len(ptrs) == 4 and all(t.numel() == 600 for t in captured)
    assert L.workspace(100, cpu, 7) is grown and L.workspace(100, cpu, 8) is not grown
    assert L.workspace(0, cpu, 7) is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.float32, 64), (torch.bfloat16, 64), (torch.bfloat16, 128)])
def test_replays_after_a_larger_eager_call_on_the_capture_stream(dev, dtype, D):
    # warm up and capture on one stream, then a larger eager call there, then other tensors on it: the
    # replays give the eager result and write nothing that is not theirs
    g = torch.Generator().manual_seed(D)
    q = torch.randn(1, 2, 12, D, generator=g).to(dtype).to(dev)
    kv = torch.randn(1, 1500, 2, D, generator=g).to(dtype).to(dev)
    sink = torch.randn(12, generator=g).to(dtype).to(dev)
    idx = torch.randint(0, 1500, (1, 2, 1400), generator=g).to(dev)
    qb = torch.randn(1, 40, 12, D, generator=g).to(dtype).to(dev)
    kvb = torch.randn(1, 2176, 2, D, generator=g).to(dtype).to(dev)
    code = L.TORCH_TO_AEKV[dtype]
    size = lambda T, S: L.lib().aekv_sink_attention_workspace_size(code, 1, T, 12, D, S, -1)  # noqa: E731
    assert 0 < size(2, 1500) < size(40, 2176)

    def calls():
        return (tiled_prefill_attention(q, kv, sink, D ** -0.5), sparse_sink_attention(q, kv, idx, sink, D ** -0.5))

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        want = calls()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            outs = calls()
        held = []
        for rep in range(3):
            tiled_prefill_attention(qb, kvb, sink, D ** -0.5)
            held += [torch.full((n // 4,), float(rep), device=dev) for n in (1 << 12, 1 << 15, 1 << 17, 1 << 19) for _ in range(4)]
            for o in outs:
                o.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert all(torch.equal(o, w) for o, w in zip(outs, want)), rep
            assert all(bool((t == float(i // 16)).all()) for i, t in enumerate(held)), rep


def test_sizes_follow_a_tensor_count_changed_in_place():
    # counts given as 0-d tensors: the size is that of the present value
    k = torch.tensor(16)
    small = indexer_workspace(4, 300, k, "cpu").numel()
    k.fill_(2000)
    assert indexer_workspace(4, 300, k, "cpu").numel() == L.lib().aekv_csa_indexer_workspace_size(4, 300, 2000) > small
    n = torch.tensor(64)
    small = decode_workspace(1, 300, 64, 12, 128, n, "cpu").numel()
    n.fill_(4096)
    assert decode_workspace(1, 300, 64, 12, 128, n, "cpu").numel() > small
    n.fill_(64)
    small = attention_workspace(1, 12, 128, n, 0, "cpu").numel()
    n.fill_(4096)
    assert attention_workspace(1, 12, 128, n, 0, "cpu").numel() > small
