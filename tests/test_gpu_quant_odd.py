"""GPU parity of the quantizers on contiguous rows of any length and alignment
(row lengths that are no multiple of 8, odd pitches, unaligned bases): fp8
bytes and scales bit-identical to the CPU oracle. The inputs are views into
buffers of infinities, so an element read from outside a row shows in its
scale."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from practice_cuda_amd.fp8_bmm import fp8_quant
from practice_cuda_amd.impls.hip_per_block import hip_per_block_quant
from practice_cuda_amd.impls.hip_per_channel import hip_per_channel_quant
from practice_cuda_amd.impls.hip_per_tensor import hip_per_tensor_quant

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
# row lengths at the edges of a chunk (8), a group (128), a unit of two chunks
# per lane (1024), a wave's row (2048) and the longest register row (16384)
COLS = [1, 7, 9, 127, 129, 1023, 1031, 2047, 2049, 4099, 16379]


def _view(x, pad, offset, dev):
    """x's values on the device with row pitch n + pad, `offset` elements into a buffer of inf."""
    *lead, m, n = x.shape
    b = lead[0] if lead else 1
    buf = torch.full((offset + b * m * (n + pad) + 16,), float("inf"), dtype=x.dtype, device=dev)
    strides = ((m * (n + pad),) if lead else ()) + (n + pad, 1)
    v = torch.as_strided(buf, x.shape, strides, offset)
    v.copy_(x)
    return v


def _same(q, s, q_ref, s_ref, label):
    assert np.array_equal(q.contiguous().view(torch.uint8).cpu().numpy(), q_ref), f"{label}: fp8 bytes differ"
    s = s.float().cpu().numpy().reshape(-1).view(np.uint32)
    assert np.array_equal(s, np.asarray(s_ref, np.float32).reshape(-1).view(np.uint32)), f"{label}: scales differ"


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("n", COLS)
def test_odd_rows_match_oracle(dev, n, dtype):
    g = torch.Generator().manual_seed(n)
    for shape, pad, offset in (((5, n), 0, 0), ((2, 131, n) if n < 5000 else (3, n), 3, 1)):
        x = (torch.randn(*shape, generator=g) * 0.3).to(DT[dtype])
        xd = _view(x, pad, offset, dev)
        print(f"odd rows {shape} {dtype} pad={pad} offset={offset}", flush=True)
        for bm, bn in ((1, 128), (1, 8), (1, 512), (128, 128), (16, 64)):
            r = hip_per_block_quant(xd, block_m=bm, block_n=bn)
            _same(r.tensor, r.dequant_scale, *O.quant_block(x, bm, bn), f"block {bm}x{bn}")
        for axis in (-2, -1):
            r = hip_per_channel_quant(xd, channel_axis=axis)
            _same(r.tensor, r.dequant_scale, *O.quant_channel(x, axis), f"channel {axis}")
        r = hip_per_tensor_quant(xd, fp8_dtype=torch.float8_e5m2)
        _same(r.tensor, r.dequant_scale, *O.quant_tensor(x, "e5m2")[:2], "tensor")


@pytest.mark.parametrize("total", [1, 7, 8, 1025, 32771, 70003])
@pytest.mark.parametrize("offset", [0, 1])
def test_odd_runs_per_tensor(dev, total, offset):
    """One contiguous run of `total` elements, aligned or not."""
    x = torch.randn(1, total, generator=torch.Generator().manual_seed(total)).bfloat16()
    print(f"odd run {total} offset={offset}", flush=True)
    xd = _view(x, 0, offset, dev)
    r = hip_per_tensor_quant(xd)
    _same(r.tensor, r.dequant_scale, *O.quant_tensor(x)[:2], "tensor")
    q, s = fp8_quant(xd)
    _same(q, s, *O.quant_tensor(x, scale_dt="input")[:2], "legacy")


def test_odd_e5m2_reduced_range(dev):
    """A caller's fp8_range below the format maximum keeps its clamp."""
    x = torch.randn(33, 1031, generator=torch.Generator().manual_seed(4))
    q, s = fp8_quant(x.to(dev), fp8_range=100.0)
    _same(q, s, *O.quant_tensor(x, scale_dt="input", fp8_max=100.0)[:2], "legacy fp8_range")


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
def test_odd_rows_skip_nan_in_the_maxima(dev, dtype):
    """A NaN does not count in the maximum of what it is quantized with, and no
    other element's byte depends on it: every scale and byte but its own are
    those of the tensor with 0 in its place. (128 consecutive NaN: whole chunks
    and a whole group of them; [8, 1031] is also one run of whole chunks.)"""
    x = torch.randn(8, 1031, generator=torch.Generator().manual_seed(5)).to(DT[dtype])
    nan = torch.zeros(x.shape, dtype=torch.bool)
    nan[0, 3] = nan[1, 256:384] = nan[2, 1030] = nan[3, 8:16] = True
    clean, dirty = x.masked_fill(nan, 0.0).to(dev), x.masked_fill(nan, float("nan")).to(dev)
    nan = nan.to(dev)
    cases = {f"block {bm}x{bn}": lambda t, bm=bm, bn=bn: hip_per_block_quant(t, block_m=bm, block_n=bn)
             for bm, bn in ((1, 8), (1, 128), (1, 512), (128, 128), (16, 64))}
    cases.update({f"channel {a}": lambda t, a=a: hip_per_channel_quant(t, channel_axis=a) for a in (-2, -1)})
    cases["tensor"] = hip_per_tensor_quant
    for name, fn in cases.items():
        print(f"odd rows NaN {name} {dtype}", flush=True)
        want, got = fn(clean), fn(dirty)
        assert torch.equal(want.dequant_scale, got.dequant_scale), name
        assert torch.equal(want.tensor.view(torch.uint8)[~nan], got.tensor.view(torch.uint8)[~nan]), name
    want, got = fp8_quant(clean), fp8_quant(dirty)
    assert torch.equal(want[1], got[1])
    assert torch.equal(want[0].view(torch.uint8)[~nan], got[0].view(torch.uint8)[~nan])
