"""GPU parity of hca_compress over the launch forms of its row kernel and the general one, against the
oracle.  fp32: at most 200 terms weighted to one, each weight within 2^-21 relative for |z| < 12; 16-bit
outputs round once (2^-9 in bf16)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from aetherkv import hca_compress
from conftest import to_np_f32

pytestmark = pytest.mark.gpu


# one entry, a wave's and a workgroup's fits with ragged entries and rows, entries past every fit, widths outside it
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,M,D", [(1, 1, 128), (5, 8, 128), (7, 7, 64), (3, 31, 64), (9, 128, 128), (2, 127, 64),
                                   (2, 200, 128), (3, 33, 512), (4, 300, 128), (3, 10, 24), (2, 5, 7)])
def test_shapes(dev, dtype, B, M, D):
    g = torch.Generator().manual_seed(M + D)
    c, z = torch.randn(B, M, D, generator=g).to(dtype), (torch.randn(B, M, D, generator=g) * 2).to(dtype)
    got = hca_compress(c.to(dev), z.to(dev))
    assert got.dtype == dtype and got.shape == (B, D)
    tol = 1e-5 if dtype == torch.float32 else 5e-3
    np.testing.assert_allclose(to_np_f32(got), O.hca_compress(to_np_f32(c), to_np_f32(z)), rtol=tol, atol=tol)


def test_infinities_stay_in_their_column(dev):
    # 7 entries leave an eighth lane slot that repeats the last entry: an infinite value there enters once, a
    # -inf logit gives its entry no weight, and other columns are untouched
    g = torch.Generator().manual_seed(1)
    c, z = torch.randn(2, 7, 64, generator=g), torch.randn(2, 7, 64, generator=g)
    z[0, 3, 5] = float("-inf")
    c[0, 6, 9] = float("inf")
    got = hca_compress(c.to(dev), z.to(dev)).cpu()
    want = (torch.softmax(z.double(), 1) * c.double()).sum(1).float()
    assert got[0, 9] == float("inf")
    got[0, 9] = want[0, 9] = 0.0
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5)
    flat = torch.empty(c.numel() + 1, device=dev)  # 4-byte aligned inputs take the general kernel
    view = flat[1:].view(c.shape)
    view.copy_(z)
    torch.testing.assert_close(hca_compress(view, z.to(dev)), hca_compress(z.to(dev), z.to(dev)), rtol=1e-5, atol=1e-5,
                               equal_nan=True)


def test_more_rows_than_a_launch_of_whole_waves(dev):
    # 2^26 rows of 16 bytes: a wave each would be 2^32 work-items, past what a launch takes; the general
    # kernel serves them (one entry per row: the result is the row itself)
    B, D = 1 << 26, 8
    c = torch.randint(-100, 100, (B, 1, D), device=dev, dtype=torch.int8).to(torch.bfloat16)
    z = torch.zeros_like(c)
    got = hca_compress(c, z)
    assert torch.equal(got, c[:, 0])


# the lines between the kernels, below and above them, by rows, entries and columns
@pytest.mark.parametrize("dtype,B,M,D", [(torch.bfloat16, B, M, D) for B, M, D in (
    (5, 22, 8), (5, 23, 8), (8192, 91, 8), (8192, 92, 8), (5, 7, 64), (5, 8, 64), (1024, 8, 64), (1025, 8, 64), (2048, 11, 64),
    (2048, 12, 64), (5, 1, 512), (5, 3, 256), (5, 4, 256), (1025, 1, 256), (16383, 3, 128), (16384, 3, 128), (16384, 2, 128))]
                         + [(torch.float32, B, M, D) for B, M, D in (
    (5, 11, 4), (5, 12, 4), (8192, 91, 4), (8192, 92, 4), (2048, 15, 4), (2048, 16, 4), (5, 1, 256), (1025, 1, 128))])
def test_lines_between_the_kernels(dev, dtype, B, M, D):
    g = torch.Generator().manual_seed(B + M * D)
    c, z = torch.randn(B, M, D, generator=g).to(dtype), (torch.randn(B, M, D, generator=g) * 2).to(dtype)
    tol = 1e-5 if dtype == torch.float32 else 5e-3
    np.testing.assert_allclose(to_np_f32(hca_compress(c.to(dev), z.to(dev))), O.hca_compress(to_np_f32(c), to_np_f32(z)),
                               rtol=tol, atol=tol)
