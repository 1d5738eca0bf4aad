"""GPU parity of the drop-in attention entry points on their fp32 matrix-core path (fp32 at head_dim
64 and 128, bf16 / fp16 at 64) against the oracle.

Tolerances: fp32 1e-5 of the values' range (sums of up to 3000 terms weighted to one, each product
within 2^-24 and the exponent's argument within 2^-23 of |logit| < 40, so below 5e-6), 16-bit outputs
the reference's own 5e-3.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import aetherkv._lib as L
import oracle as O
from aetherkv import sparse_sink_attention, tiled_prefill_attention
from conftest import to_np_f32

pytestmark = pytest.mark.gpu


def _tol(dtype):
    return 1e-5 if dtype == torch.float32 else 5e-3


def _inputs(seed, B, T, H, D, S, dtype):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, T, H, D, generator=g).to(dtype)
    kv = torch.randn(B, S, 2, D, generator=g).to(dtype)
    sink = torch.randn(H, generator=g).to(dtype)
    return g, q, kv, sink


def _check(got, q, kv, idx, sink, scale):
    assert got.dtype == q.dtype and got.shape == q.shape
    want = O.sink_attention(to_np_f32(q), to_np_f32(kv), idx, to_np_f32(sink), scale, threads=8)
    np.testing.assert_allclose(to_np_f32(got), want, rtol=_tol(q.dtype), atol=_tol(q.dtype))


# one partial group, whole groups, 4 and 8 waves, several groups per wave, a split (> 640 sources), two head groups
@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.float32, 64), (torch.bfloat16, 64), (torch.float16, 64)])
@pytest.mark.parametrize("H,K,idx_dtype", [(12, 1, torch.int32), (16, 17, torch.int64), (20, 256, torch.int32),
                                           (3, 1100, torch.int64)])
def test_sparse_shapes(dev, dtype, D, H, K, idx_dtype):
    g, q, kv, sink = _inputs(H + K, 2, 3, H, D, 700, dtype)
    idx = torch.randint(-30, 730, (2, 3, K), generator=g, dtype=idx_dtype)  # some skipped, some repeated
    idx[1, 2] = -1                                                         # no valid source
    got = sparse_sink_attention(q.to(dev), kv.to(dev), idx.to(dev), sink.to(dev), D ** -0.5)
    _check(got, q, kv, idx.numpy(), sink, D ** -0.5)
    assert not bool(got[1, 2].float().abs().sum())


# fewer rows than a block, both row-group counts, ragged rows and sources, split and not
@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.float32, 64), (torch.bfloat16, 64)])
@pytest.mark.parametrize("B,T,H,S", [(1, 1, 12, 640), (2, 1, 3, 1), (1, 5, 12, 2176), (3, 67, 16, 131), (1, 173, 12, 1003)])
def test_dense_shapes(dev, dtype, D, B, T, H, S):
    _, q, kv, sink = _inputs(T + S, B, T, H, D, S, dtype)
    got = tiled_prefill_attention(q.to(dev), kv.to(dev), sink.to(dev), D ** -0.5)
    _check(got, q, kv, np.broadcast_to(np.arange(S), (B, T, S)), sink, D ** -0.5)


def test_skipped_values_and_extreme_logits(dev):
    # values of skipped sources never enter (row 0 stands in for them and is not finite), large logits
    # are exact maxima, a scalar sink of -inf leaves the softmax without one, a dominant one empties it
    g, q, kv, _ = _inputs(5, 1, 4, 16, 128, 90, torch.float32)
    kv[:, 0] = float("inf")
    idx = torch.randint(1, 90, (1, 4, 50), generator=g)
    idx[0, :, ::3] = 95
    q = q * 30.0
    for sink in (torch.tensor([float("-inf")]), torch.tensor([1e4])):
        got = sparse_sink_attention(q.to(dev), kv.to(dev), idx.to(dev), sink.to(dev), 128 ** -0.5)
        kv0 = kv.clone()
        kv0[:, 0] = 0.0
        want = O.sink_attention(to_np_f32(q), to_np_f32(kv0), idx.numpy(), to_np_f32(sink), 128 ** -0.5)
        # |logit| up to ~150: the exponent's argument is within 150 * 2^-22 = 4e-5
        np.testing.assert_allclose(to_np_f32(got), want, rtol=1e-4, atol=1e-4)


def test_unsplit_and_small_workspace_agree(dev):
    # the entry point without a workspace, and one with a workspace below the split's, run unsplit
    B, T, H, D, S = 1, 2, 12, 128, 1500
    _, q, kv, sink = _inputs(9, B, T, H, D, S, torch.float32)
    assert L.lib().aekv_sink_attention_workspace_size(L.F32, B, T, H, D, S, -1) > 256
    qd, kvd, sd = q.to(dev), kv.to(dev), sink.to(dev)
    outs = [torch.empty_like(qd) for _ in range(2)]
    small = torch.empty(256, dtype=torch.uint8, device=dev)
    with torch.cuda.device(dev):
        for out, ws, n in ((outs[0], None, 0), (outs[1], small, 256)):
            L.check(L.lib().aekv_tiled_prefill_attention_ws(
                L.ptr(qd), L.ptr(kvd), L.ptr(sd), H, L.F32, B, T, H, D, S, D ** -0.5, 256, L.ptr(ws), n, L.ptr(out),
                L.stream_of(qd)), "tiled")
    for out in outs:
        _check(out, q, kv, np.broadcast_to(np.arange(S), (B, T, S)), sink, D ** -0.5)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("K", [50, 1500])  # whole, and split into pieces
def test_no_sink_and_no_maximum(dev, K):
    # a sink of -inf leaves a target without sources at zero, and one whose logits are all NaN at NaN
    g, q, kv, _ = _inputs(11, 1, 2, 12, 128, 900, torch.float32)
    q[0, 1] = float("nan")
    idx = torch.randint(0, 900, (1, 2, K), generator=g)
    idx[0, 0] = -1
    got = sparse_sink_attention(q.to(dev), kv.to(dev), idx.to(dev), torch.full((12,), float("-inf"), device=dev), 128 ** -0.5)
    assert bool((got[0, 0] == 0).all()) and bool(torch.isnan(got[0, 1]).all())


def test_more_targets_than_a_launch_of_whole_workgroups(dev):
    # 2^24 targets of one head: a workgroup of 256 threads each would be 2^32 work-items, past what a
    # launch takes, so the call runs on the kernel of one wave per row; its parts fit
    T, D, S = 1 << 24, 64, 512
    g = torch.Generator(device=dev).manual_seed(3)
    q = torch.randn(1, T, 1, D, generator=g, device=dev, dtype=torch.bfloat16)
    kv = torch.randn(1, S, 2, D, generator=g, device=dev, dtype=torch.bfloat16)
    idx = torch.randint(0, S, (1, T, 130), generator=g, device=dev, dtype=torch.int32)
    sink = torch.zeros(1, device=dev, dtype=torch.bfloat16)
    got = sparse_sink_attention(q, kv, idx, sink, D ** -0.5)
    for lo in (0, T // 2, T - 4096):
        part = slice(lo, lo + 4096)
        want = sparse_sink_attention(q[:, part].contiguous(), kv, idx[:, part].contiguous(), sink, D ** -0.5)
        # both in fp32 from the same inputs: at most one bf16 rounding apart
        torch.testing.assert_close(got[:, part], want, rtol=2 ** -7, atol=1e-5)


# Sparse calls either side of the lines between the VALU kernel, one wave and four waves per workgroup (targets,
# heads, sources), none of them at all, and two head groups of a target.
@pytest.mark.parametrize("dtype,D", [(torch.float32, 64), (torch.float32, 128), (torch.bfloat16, 64)])
@pytest.mark.parametrize("T,H,K", [(1023, 3, 128), (1024, 3, 128), (1024, 3, 129), (1025, 6, 1), (1025, 7, 1), (513, 17, 1), (2047, 1, 4), (2048, 1, 4),
                                   (2048, 1, 5), (6144, 1, 12), (6144, 1, 13), (6143, 2, 3), (6144, 2, 3), (6144, 2, 4),
                                   (3000, 1, 0)])
def test_lines_between_kernels(dev, dtype, D, T, H, K):
    g = torch.Generator(device=dev).manual_seed(T + H + K)
    q = torch.randn(1, T, H, D, generator=g, device=dev).to(dtype)
    kv = torch.randn(1, 300, 2, D, generator=g, device=dev).to(dtype)
    idx = torch.randint(-20, 320, (1, T, K), generator=g, device=dev)  # some skipped
    sink = torch.randn(H, generator=g, device=dev).to(dtype)
    got = sparse_sink_attention(q, kv, idx, sink, D ** -0.5)
    for lo in (0, T // 2, T - 100):
        part = slice(lo, lo + 100)
        want = O.sink_attention(to_np_f32(q[:, part]), to_np_f32(kv), idx[:, part].cpu().numpy(), to_np_f32(sink), D ** -0.5,
                                threads=8)
        np.testing.assert_allclose(to_np_f32(got[:, part]), want, rtol=_tol(dtype), atol=_tol(dtype))
