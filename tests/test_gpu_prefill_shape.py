"""The workgroup shape that an HCA prefill chunk's attention takes: the 96-row shape, which rounds each
row's weights at four running maxima, wherever it leaves no CU with more rows than the 64-row shape's two
maxima would.  Chunks of one round and chunks just past one are the ones where another choice is faster
and further from 64 bits."""
from __future__ import annotations

import pytest
import torch

import aetherkv._lib as L
from aetherkv import PolarQuant
from aetherkv.prefill import hca_prefill
from aetherkv.synthetic import normal

pytestmark = pytest.mark.gpu


# 12 heads: one workgroup per CU or fewer, the last 64-row blocks few; the 64-row shape's own range
@pytest.mark.parametrize("B,T,S,rows", [(1, 128, 2048, 96), (1, 1360, 700, 96), (2, 170, 2048, 96), (8, 375, 100, 96),
                                        (1, 3001, 2021, 96), (1, 2400, 300, 64)])
def test_shape(dev, B, T, S, rows):
    pq = PolarQuant(4)
    codes, scale = pq.encode(normal((B, S, 128), 3).to(dev))
    q, win = normal((B, T, 12, 128), 4).to(dev), normal((B, T + 127, 128), 5).to(dev)
    sink = normal((12,), 6, dtype=torch.float32).to(dev)
    start = S * 128 - T

    def call(shape):
        old = L.lib().aekv_set_flash_rows(shape)
        try:
            return hca_prefill(q, codes, scale, win, sink, 128 ** -0.5, kv_quant=pq, start=start)
        finally:
            L.lib().aekv_set_flash_rows(old)

    assert torch.equal(call(0), call(rows))
