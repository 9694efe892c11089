"""The per-tensor and per-column C entry points with and without a workspace
(two and four launches) give the same bytes and scales."""
from __future__ import annotations

import pytest
import torch

from practice_cuda_amd import _lib
from practice_cuda_amd.impls.hip_per_channel import hip_per_channel_quant

pytestmark = pytest.mark.gpu


def _head(x, y):
    b, m, n = x.shape
    return (_lib.ptr(x), _lib.dtype_code(x.dtype), b, m, n, *x.stride(), _lib.ptr(y), _lib.E4M3FN, *y.stride())


def _x(shape, dtype, dev):
    x = torch.randn(*shape, generator=torch.Generator().manual_seed(shape[1])) * 0.3
    return x.to(dtype).to(dev)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 1, 8), (1, 3, 5), (2, 100, 1024), (1, 4096, 1031), (1, 2100, 4096)])
def test_per_tensor_workspace(dev, shape, dtype):
    """One workgroup, a few, and more chunks than the amax grid's 256 workgroups take in one step."""
    x = _x(shape, dtype, dev)
    L, st = _lib.lib(), _lib.stream_of(x)
    got = []
    for ws in (False, True):
        y = torch.zeros(shape, dtype=torch.float8_e4m3fn, device=dev)
        s = torch.full((4 + 256,), float("nan"), device=dev)  # stale slots must not count
        cast = torch.zeros((), dtype=dtype, device=dev)
        args = (*_head(x, y), s.data_ptr(), s.data_ptr() + 4, 448.0, 1e-12, _lib.dtype_code(dtype))
        if ws:
            rc = L.pcamd_quant_tensor_ws(*args, cast.data_ptr(), s.data_ptr() + 16, 1024, st)
        else:
            rc = L.pcamd_quant_tensor(*args, st)
        _lib.check(rc, "per-tensor")
        torch.cuda.synchronize()
        if ws:
            assert torch.equal(cast.float(), s[0].to(dtype).float())
        got.append((y.view(torch.uint8), s[:2].view(torch.int32)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("total", [262144 - 8, 262144, 262144 + 8, 262144 + 2049, 3 * 262144 - 3, 40 * 262144 + 11])
def test_per_tensor_workspace_span_edges(dev, total):
    """The quantize pass takes the tensor in spans of 262144 elements, the last one first: whole
    spans, a piece more or less, odd ends. Bytes and scales as without a workspace, nothing behind the end."""
    x = _x((1, 1, total), torch.bfloat16, dev)
    L, st = _lib.lib(), _lib.stream_of(x)
    got = []
    for ws in (False, True):
        buf = torch.full((total + 64,), 0x55, dtype=torch.uint8, device=dev)
        y = buf[:total].view(torch.float8_e4m3fn).view(1, 1, total)
        s = torch.full((4 + 256,), float("nan"), device=dev)
        args = (*_head(x, y), s.data_ptr(), s.data_ptr() + 4, 448.0, 1e-12, _lib.F32)
        if ws:
            rc = L.pcamd_quant_tensor_ws(*args, 0, s.data_ptr() + 16, 1024, st)
        else:
            rc = L.pcamd_quant_tensor(*args, st)
        _lib.check(rc, "per-tensor")
        torch.cuda.synchronize()
        got.append((buf, s[:2].view(torch.int32)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("shape", [(1, 257, 8), (1, 300, 130), (2, 1281, 264), (1, 4300, 1024), (3, 700, 1031)])
def test_per_column_workspace(dev, shape):
    """Parts of one slab and of several, a ragged last part, batches, odd rows."""
    x = _x(shape, torch.bfloat16, dev)
    b, m, n = shape
    L, st = _lib.lib(), _lib.stream_of(x)
    size = L.pcamd_quant_channel_workspace(b, m, n, -1)
    assert size > 0 and L.pcamd_quant_channel_workspace(b, m, n, -2) == 0
    got = []
    for ws in (None, torch.full((size // 4,), float("nan"), device=dev)):
        y = torch.zeros(shape, dtype=torch.float8_e4m3fn, device=dev)
        s = torch.zeros(b, n, device=dev)
        rc = L.pcamd_quant_channel_ws(*_head(x, y), s.data_ptr(), n, 1, -1, 448.0, 1e-12, _lib.ptr(ws),
                                      0 if ws is None else size, st)
        _lib.check(rc, "per-column")
        torch.cuda.synchronize()
        got.append((y.view(torch.uint8), s.view(torch.int32)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("shape", [(1, 24578, 130), (1, 30000, 8), (2, 25000, 3), (1, 70000, 264)])
def test_per_column_workspace_tall(dev, shape):
    """Tall, narrow tensors: more than 64 parts per column, reduced to one before the quantize pass."""
    x = _x(shape, torch.bfloat16, dev)
    b, m, n = shape
    L, st = _lib.lib(), _lib.stream_of(x)
    size = L.pcamd_quant_channel_workspace(b, m, n, -1)
    assert size > 64 * b * n * 4
    got = []
    for ws in (None, torch.full((size // 4 + 16,), float("nan"), device=dev)):
        y = torch.zeros(shape, dtype=torch.float8_e4m3fn, device=dev)
        s = torch.zeros(b, n, device=dev)
        rc = L.pcamd_quant_channel_ws(*_head(x, y), s.data_ptr(), n, 1, -1, 448.0, 1e-12, _lib.ptr(ws),
                                      0 if ws is None else size, st)
        _lib.check(rc, "per-column")
        torch.cuda.synchronize()
        assert ws is None or torch.isnan(ws[size // 4:]).all()
        got.append((y.view(torch.uint8), s.view(torch.int32)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("shape", [(1, 200, 1031), (1, 200, 4099), (1, 2, 16383), (3, 256, 2047)])
def test_per_column_few_odd_rows(dev, shape):
    """At most 256 odd rows: element-wise without a workspace, in slabs with one; same bytes as the aligned
    columns of a wider tensor."""
    b, m, n = shape
    wide = _x((b, m, -(-n // 8) * 8), torch.bfloat16, dev)
    x = wide[:, :, :n].contiguous()
    r, w = hip_per_channel_quant(x, channel_axis=-1), hip_per_channel_quant(wide, channel_axis=-1)
    assert torch.equal(r.tensor.view(torch.uint8), w.tensor.view(torch.uint8)[:, :, :n])
    assert torch.equal(r.dequant_scale, w.dequant_scale[:, :n])


def test_workspace_too_small(dev):
    x = _x((1, 512, 256), torch.bfloat16, dev)
    y = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=dev)
    s = torch.empty(1, 256, device=dev)
    L, st = _lib.lib(), _lib.stream_of(x)
    assert L.pcamd_quant_channel_ws(*_head(x, y), s.data_ptr(), 256, 1, -1, 448.0, 1e-12, s.data_ptr(), 64,
                                    st) == _lib.ERR_INVALID
    assert L.pcamd_quant_tensor_ws(*_head(x, y), s.data_ptr(), 0, 448.0, 1e-12, 0, 0, s.data_ptr(), 64,
                                   st) == _lib.ERR_INVALID
