"""aekv_prefill_counts and the prefill calls that use it: the counts of prefill_sources, on the device;
the arguments that were refused before any device work stay refused."""
from __future__ import annotations

import pytest
import torch

import aetherkv._lib as L
from aetherkv import PolarQuant
from aetherkv.prefill import _device_sources, csa_prefill, hca_prefill, prefill_sources


@pytest.mark.gpu
# the first targets of a prompt, block edges, counts past a workgroup, a window buffer that starts earlier
@pytest.mark.parametrize("B,T,start,nb,M,W,extra,k", [(1, 1, 0, 0, 4, 3, 0, 0), (3, 10, 0, 2, 4, 3, 0, 1),
                                                     (2, 300, 127, 5, 128, 128, 0, 256), (8, 257, 5000, 3000, 4, 128, 9, 256)])
def test_counts_match_host(dev, B, T, start, nb, M, W, extra, k):
    first = max(0, start - W + 1) - extra if start >= W - 1 + extra else 0
    Wt = start + T - first
    want = prefill_sources(T, start, nb, compression=M, sliding_window=W, window_base=first, window_len=Wt)
    q = torch.zeros(B, T, 2, 128, dtype=torch.bfloat16, device=dev)
    got = _device_sources(q, torch.zeros(B, Wt, 1, device=dev), start, nb, M, W, first, k).cpu()
    for row, w in zip((got[0], got[1], got[2], got[3]), (want[0], want[0].clamp(max=k), want[1], want[2])):
        assert torch.equal(row, w.expand(B, T))


def test_host_checks():
    lib = L.lib()
    assert lib.aekv_prefill_counts(1, 4, 0, 1, 0, 3, 0, 0, 256, 512, 768, 1024, None) == L.ERR_VALUE
    assert lib.aekv_prefill_counts(1, 4, -1, 1, 4, 3, 0, 0, 256, 512, 768, 1024, None) == L.ERR_VALUE
    assert lib.aekv_prefill_counts(1 << 20, 1 << 20, 0, 1, 4, 3, 0, 0, 256, 512, 768, 1024, None) == L.ERR_UNSUPPORTED
    assert lib.aekv_prefill_counts(1, 4, 0, 1, 4, 3, 0, 0, None, None, 768, 1024, None) == L.ERR_VALUE
    assert lib.aekv_prefill_counts(0, 4, 0, 1, 4, 3, 0, 0, None, None, None, None, None) == L.OK
    # host tensors are refused before anything is launched; a window that does not cover the chunk comes first
    q, win = torch.zeros(1, 2, 4, 128, dtype=torch.bfloat16), torch.zeros(1, 5, 128, dtype=torch.bfloat16)
    codes, scale, sink, pq = torch.zeros(1, 3, 64, dtype=torch.uint8), torch.ones(1, 3), torch.zeros(4), PolarQuant(4)
    iq, iw, ix = torch.zeros(1, 2, 4, 64), torch.zeros(1, 2, 4), torch.zeros(1, 3, 32, dtype=torch.uint8)
    with pytest.raises(ValueError, match="does not cover"):
        hca_prefill(q, codes, scale, win, sink, 0.1, kv_quant=pq, start=200)
    with pytest.raises(RuntimeError, match="HIP device"):
        hca_prefill(q, codes, scale, win, sink, 0.1, kv_quant=pq, start=3)
    with pytest.raises(RuntimeError, match="HIP device"):
        csa_prefill(q, iq, iw, ix, scale, codes, scale, win, sink, 0.1, kv_quant=pq, start=3)
