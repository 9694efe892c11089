"""Bias in the staged epilogue of the tiled BMM (csrc/bmm_epilogue.h): row
pieces of the bias pass through the staging slots that the outputs take.

Operands are small integers, scales powers of two and the bias a multiple of
1/4, so the scaled product plus the bias is exact in fp32 and the 16-bit
output must be its single rounding, bit for bit.
"""
from __future__ import annotations

import pytest
import torch

from practice_cuda_amd.impls.hip_per_block import hip_per_block_bmm
from practice_cuda_amd.impls.hip_per_channel import hip_per_channel_bmm
from practice_cuda_amd.registry import QuantResult

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn

# 128 x 128 tiles (first and last) and whole tiles, partial ones in both
# directions (half tiles: test_gpu_tiles.py)
SHAPES = [(1, 1000, 2056, 160), (3, 1030, 8200, 256), (2, 512, 8192, 144)]


def _bias(kind, b, m, n, dtype, g, dev):
    v = (torch.randint(-64, 65, (b, m, n), generator=g) / 4).to(dtype).to(dev)
    if kind == "rows":      # one row broadcast over M
        return v[:, :1].expand(b, m, n)
    if kind == "batch":     # one matrix broadcast over the batch
        return v[:1].expand(b, m, n)
    if kind == "offset8":   # rows 8-byte aligned only
        buf = torch.zeros(b, m, n + 4, dtype=dtype, device=dev)
        buf[:, :, 4:] = v
        return buf[:, :, 4:]
    if kind == "offset2":   # unaligned rows: the element-wise epilogue
        buf = torch.zeros(b, m, n + 3, dtype=dtype, device=dev)
        buf[:, :, 3:] = v
        return buf[:, :, 3:]
    return v


@pytest.mark.parametrize("kind", ["full", "rows", "batch", "offset8", "offset2"])
@pytest.mark.parametrize("scheme", ["channel", "block128", "block1"])
@pytest.mark.parametrize("shape", SHAPES)
def test_staged_bias_exact(dev, shape, scheme, kind):
    b, m, n, k = shape
    g = torch.Generator().manual_seed(1)
    va = torch.randint(-4, 5, (b, m, k), generator=g).float()
    vb = torch.randint(-4, 5, (b, k, n), generator=g).float()
    va, vb = va.to(dev), vb.to(dev)
    qa, qb = va.to(E4M3), vb.to(E4M3)
    two = lambda *s: 2.0 ** torch.randint(-2, 3, s, generator=g).float().to(dev)  # noqa: E731
    print(f"bias {scheme} {shape} {kind}", flush=True)
    if scheme == "channel":
        sa, sb = two(b, m), two(b, n)
        ref = torch.bmm(va, vb) * sa[:, :, None] * sb[:, None]
        ra = QuantResult(qa, sa, "t", "channel", {"channel_axis": -2})
        rb = QuantResult(qb, sb, "t", "channel", {"channel_axis": -1})
        fn = hip_per_channel_bmm
    else:
        qbn = int(scheme[5:])
        kb = -(-k // 128)
        sa, sb = two(b, m, kb), two(b, kb, -(-n // qbn))
        ref = torch.zeros(b, m, n, device=dev)
        for i in range(kb):
            s = slice(128 * i, min(128 * i + 128, k))
            ref += torch.bmm(va[:, :, s].contiguous(), vb[:, s].contiguous()) * sa[:, :, i, None] * \
                sb[:, i].repeat_interleave(qbn, dim=1)[:, None, :n]
        ra = QuantResult(qa, sa, "t", "block", {"block_m": 1, "block_n": 128})
        rb = QuantResult(qb, sb, "t", "block", {"block_m": 128, "block_n": qbn})
        fn = hip_per_block_bmm
    for dtype in (torch.bfloat16, torch.float16):
        bias = _bias(kind, b, m, n, dtype, g, dev)
        out = fn(ra, rb, out_dtype=dtype, bias=bias)
        assert torch.equal(out, (ref + bias.float()).to(dtype))
