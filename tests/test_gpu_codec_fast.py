"""The fast encodes of D = 64 and 128 from bf16 and fp16, bit for bit against the generic kernel (which the
oracle pins); the encode of fp32 inputs, which has the generic kernel alone, against the oracle on the same
vectors; and the 4-element decode layout of fp32 outputs against the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import aetherkv._lib as L
import oracle as O
from aetherkv import PolarQuant
from aetherkv.synthetic import normal_with_outliers

pytestmark = pytest.mark.gpu


def _both(pq, x):
    prev = L.lib().aekv_set_generic_kernels(1)
    try:
        g = pq.encode(x)
    finally:
        L.lib().aekv_set_generic_kernels(prev)
    return g, pq.encode(x)


def _same(pq, x):
    if x.dtype == torch.float32:
        codes, scale = pq.encode(x)
        want_c, want_s = O.encode(x.cpu().numpy(), "f32", pq.bits, O.diag(42, x.shape[-1]))
        np.testing.assert_array_equal(codes.cpu().numpy(), want_c)
        np.testing.assert_array_equal(scale.cpu().numpy(), want_s)
        return
    if x.dtype == torch.float16:  # (the fast fp16 encode starts at 3 * 2^20 elements: whole waves ahead of x)
        ahead = torch.randn((3 << 20) // x.shape[-1], x.shape[-1], generator=torch.Generator(device=x.device).manual_seed(0),
                            device=x.device)
        x = torch.cat([ahead.to(x.dtype), x])
    (cg, sg), (cf, sf) = _both(pq, x)
    assert torch.equal(cg, cf)
    assert torch.equal(sg.view(torch.int32), sf.view(torch.int32))  # (bits: NaN scales compare too)


CASES = [(dt, bits, d) for dt in (torch.bfloat16, torch.float16, torch.float32) for bits in (4, 8) for d in (64, 128)]


# a lone vector, partial and whole waves, thousands of waves (some hold undecided roundings)
@pytest.mark.parametrize("dtype,bits,d", CASES)
@pytest.mark.parametrize("n", [1, 15, 33, 200003])
def test_random_vectors(dev, dtype, bits, d, n):
    _same(PolarQuant(bits), normal_with_outliers((n, d), n + d + bits, dtype=dtype, trailing_dims=1).to(dev))


# vectors of a few small integers: their transforms take few values, whose ratios to the largest are often exact
# halves of a code step (3 +- 1 gives 2 / 4 * 7 = 3.5 and 2 / 4 * 127 = 63.5): ties and near ties throughout
@pytest.mark.parametrize("dtype,bits,d", CASES)
def test_ties(dev, dtype, bits, d):
    g = torch.Generator().manual_seed(d + bits)
    x = torch.zeros(20000, d)
    for n in range(1, 5):
        rows = slice(5000 * (n - 1), 5000 * n)
        at = torch.rand(5000, d, generator=g).argsort(1)[:, :n]
        x[rows].scatter_(1, at, torch.randint(-9, 10, (5000, n), generator=g).float())
    _same(PolarQuant(bits), x.to(dtype).to(dev))
    _same(PolarQuant(bits), (x * 0.1).to(dtype).to(dev))  # rounded inputs: near ties


# zero, tiny and huge vectors, infinities and NaN, and (bf16) sums that overflow, between ordinary vectors of one wave.
# (The oracle converts a NaN ratio to a whole number, which C leaves undefined: fp32 vectors with one are left out.
# The 4-bit D = 128 bf16 kernel is another one, which takes finite vectors of ordinary range: zero and tiny ones.)
@pytest.mark.parametrize("dtype,bits,d", CASES)
def test_extreme_vectors(dev, dtype, bits, d):
    x = torch.randn(64, d, generator=torch.Generator().manual_seed(d))
    big = 6e4 if dtype == torch.float16 else 3e38
    x[3] = 0.0
    x[5] *= 1e-7
    x[7] *= 1e-12
    x[20] *= big / 200
    x[22, :3] = big
    x[40] = big
    x[41, ::2], x[41, 1::2] = big, -big
    x[50, 9] = float("inf")
    x[51, 10], x[51, 11] = float("inf"), float("-inf")
    x[60, 12] = float("nan")
    if dtype != torch.float16:
        x[30] *= 1e31  # above the fast quantiser's range, sums still finite
        x[31] *= 1e-36
    if dtype == torch.float32:
        x = x[[i for i in range(64) if i not in (22, 40, 41, 50, 51, 60)]]
    elif (dtype, bits, d) == (torch.bfloat16, 4, 128):
        x = x[:20]
    for rows in (slice(0, 16), slice(16, 35), slice(0, 64)):
        if len(x[rows]):
            _same(PolarQuant(bits), x[rows].to(dtype).to(dev))


# the fp16 line between the generic and the fast encode: either side of 3 * 2^20 elements
@pytest.mark.parametrize("bits,d", [(4, 64), (8, 64), (4, 128), (8, 128)])
def test_fp16_line(dev, bits, d):
    n = (3 << 20) // d
    x = normal_with_outliers((n, d), d + bits, dtype=torch.float16, trailing_dims=1).to(dev)
    pq = PolarQuant(bits)
    for rows in (n - 1, n):
        (cg, sg), (cf, sf) = _both(pq, x[:rows])
        assert torch.equal(cg, cf) and torch.equal(sg, sf)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("d", [16, 32, 64, 128, 256, 512])
def test_decode_to_fp32(dev, bits, d):
    rng = np.random.default_rng(d)
    for n in (1, 37, 3001):
        if bits == 8:
            codes = rng.integers(-127, 128, (n, d)).astype(np.int8)
        else:
            codes = rng.integers(0, 256, (n, d // 2)).astype(np.uint8)
        scale = (rng.random((n, 1)) + 1e-3).astype(np.float32)
        got = PolarQuant(bits).decode(torch.from_numpy(codes).to(dev), torch.from_numpy(scale).to(dev), torch.float32)
        np.testing.assert_array_equal(got.cpu().numpy(), O.decode(codes, scale, bits, O.diag(42, d), "f32"))


# streamed decodes (160 MB of codes and output; 400 MB: past the caches), with a last wave and group partly filled
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bits,d", [(4, 64), (8, 64), (4, 128), (8, 128)])
@pytest.mark.parametrize("line", [160_000_000, 400_000_000])
def test_streamed_decode(dev, dtype, bits, d, line):
    es = 4 if dtype == torch.float32 else 2
    n = -(-line // (d * es + d * bits // 8)) + 37
    g = torch.Generator(device=dev).manual_seed(n + bits)
    lo, hi = (0, 256) if bits == 4 else (-127, 128)
    codes = torch.randint(lo, hi, (n, d * bits // 8), generator=g, device=dev, dtype=torch.uint8 if bits == 4 else torch.int8)
    scale = torch.rand(n, 1, generator=g, device=dev)
    scale[::1000] = 0.0
    pq = PolarQuant(bits)
    got = pq.decode(codes, scale, dtype)
    prev = L.lib().aekv_set_generic_kernels(1)
    try:
        want = pq.decode(codes, scale, dtype)
    finally:
        L.lib().aekv_set_generic_kernels(prev)
    assert torch.equal(got, want)
    small = pq.decode(codes[-100:], scale[-100:], dtype)  # (below the line)
    assert torch.equal(small, got[-100:])
