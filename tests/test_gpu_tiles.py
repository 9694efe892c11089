"""The tile forms of the wide BMM kernel, each on a grid that takes it, and the
general kernel, exactly.

Grids are sized from the CU count: 128 x 128 tiles where 256 x 256 ones leave
CUs idle, one wave of whole tiles, and two waves with a short third that runs as
half tiles; all past the K-split kernel's range (two 64 x 64 tiles per CU). The
general kernel takes e5m2 operands whose rows are not 16-byte aligned, and large
e4m3fn products with aligned rows and a K that is no multiple of 4.

Operands are small integers, scales powers of two and biases multiples of 1/4,
so every product and sum is exact in fp32 in any order: an fp32 output equals the
reference, a 16-bit one its single rounding. Every row's padding, which a masked
last K step loads too, holds NaN codes.
"""
from __future__ import annotations

import pytest
import torch

from practice_cuda_amd import _lib

pytestmark = pytest.mark.gpu
E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2
LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]
MODES = {"block128": _lib.SCALE_BLOCK, "block16": _lib.SCALE_BLOCK, "block1": _lib.SCALE_BLOCK,
         "channel": _lib.SCALE_CHANNEL, "tensor": _lib.SCALE_TENSOR}


def _size(form, dev):
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    if form == "small":  # 18 rows of 64 x 64 tiles, a little more than two per CU
        return 1104, (2 * cus // 18 + 2) * 64 - 16
    if form == "whole":  # 16 x (cus / 16) tiles
        return 4080, cus // 16 * 256 - 48
    if form == "halves":  # two waves and an eighth
        return (2 * cus + cus // 8) // 16 * 256 - 16, 4096 - 48
    if form == "odd_k":  # 32 rows of 64 x 64 tiles, a little more than six per CU
        return 2032, (6 * cus // 32 + 2) * 64 - 16
    return 33, 47


def _operand(rows, cols, last, pad, dtype, g, dev):
    """(values [1, rows, cols], a view of them contiguous along the last dim or the one before, NaN codes behind each row)"""
    v = torch.randint(-4, 5, (1, rows, cols), generator=g, device=dev).float()
    s = v if last else v.transpose(1, 2)
    buf = torch.full((1, s.shape[1], s.shape[2] + pad), 0x7F, dtype=torch.uint8, device=dev).view(dtype)
    buf[:, :, :s.shape[2]] = s.to(dtype)
    q = buf[:, :, :s.shape[2]]
    return v, q if last else q.transpose(1, 2)


def _pow2(shape, g, dev):
    return 2.0 ** torch.randint(-2, 3, shape, generator=g, device=dev).float()


def _case(form, mode, k, a_k, b_k, dev, out_dtype=torch.float32, bias=False, quant_scales=False, gelu=False):
    m, n = _size(form, dev)
    dtype, pad = (E5M2, 1) if form == "general" else (E4M3, 16)
    g = torch.Generator(device=dev).manual_seed(k)
    pad_of = lambda last, c, r: pad if form == "general" else pad + -(c if last else r) % 16  # noqa: E731
    va, qa = _operand(m, k, a_k, pad_of(a_k, k, m), dtype, g, dev)
    vb, qb = _operand(k, n, not b_k, pad_of(not b_k, n, k), dtype, g, dev)
    qbn, kb = int(mode[5:]) if mode.startswith("block") else 1, -(-k // 128)
    if mode.startswith("block"):
        sa, sb = _pow2((1, m, kb), g, dev), _pow2((1, kb, -(-n // qbn)), g, dev)
        ref = torch.zeros(1, m, n, device=dev)
        for i in range(kb):
            s = slice(128 * i, min(128 * i + 128, k))
            ref += (va[:, :, s].contiguous() @ vb[:, s].contiguous()) * sa[:, :, i, None] * \
                sb[:, i].repeat_interleave(qbn, dim=1)[:, None, :n]
    else:
        shapes = ((1, m), (1, n)) if mode == "channel" else ((1, 1), (1, 1))
        sa, sb = (_pow2(s, g, dev) for s in shapes)
        scale = sa[:, :, None] * sb[:, None] if mode == "channel" or quant_scales else sa[:, :, None]
        ref = (va @ vb) * (1 / scale if quant_scales else scale)
    bv = None
    if bias:
        bv = (torch.randint(-64, 65, (1, m, n), generator=g, device=dev) / 4).to(torch.float16)
        ref = ref + bv.float()
    if gelu:
        ref = torch.nn.functional.gelu(ref.double()).float()
    c = torch.empty(1, m, n, dtype=out_dtype, device=dev)
    st = lambda t: tuple(t.stride()) + (0,) * (3 - t.dim())  # noqa: E731
    print(f"tiles {form} {mode} {m}x{n}x{k} a_k={a_k} b_k={b_k} {out_dtype}", flush=True)
    rc = _lib.lib().pcamd_bmm_scaled(
        _lib.ptr(qa), _lib.ptr(qb), _lib.dtype_code(dtype), 1, m, n, k, *qa.stride(), *qb.stride(), _lib.ptr(c),
        _lib.dtype_code(out_dtype), *c.stride(), _lib.ptr(bv), 0 if bv is None else _lib.F16,
        *((0, 0, 0) if bv is None else bv.stride()), _lib.ptr(sa), *st(sa), _lib.ptr(sb), *st(sb), MODES[mode],
        int(quant_scales), 1, 128, qbn, _lib.ACT_GELU if gelu else _lib.ACT_NONE, _lib.stream_of(c))
    _lib.check(rc, "pcamd_bmm_scaled")
    return c, ref


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("k", [256, 272, 388])
@pytest.mark.parametrize("form", ["small", "whole", "halves", "general"])
def test_tile_forms_exact(dev, form, k, mode, a_k, b_k):
    """Whole K steps, and last ones of 16 and 4 valid k (388 of an even and an odd number of steps)."""
    out, ref = _case(form, mode, k, a_k, b_k, dev)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("mode", ["block128", "channel", "tensor"])
@pytest.mark.parametrize("k", [100, 1031])
def test_large_odd_k_exact(dev, k, mode, a_k, b_k):
    """Aligned rows that the wide kernel does not take: the general kernel with one scale (and, from K =
    1024 on, channel scales unless both operands are K-major), else the K-split kernel."""
    out, ref = _case("odd_k", mode, k, a_k, b_k, dev)
    assert torch.equal(out, ref)


@pytest.mark.parametrize("mode", ["channel", "tensor"])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", ["small", "whole", "halves", "general"])
def test_scales_are_quant(dev, form, out_dtype, mode):
    """The epilogues that multiply by 1 / (sa sb): element by element and through LDS."""
    out, ref = _case(form, mode, 256, True, False, dev, out_dtype=out_dtype, quant_scales=True)
    assert torch.equal(out, ref.to(out_dtype))


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("form", ["small", "whole", "halves", "general"])
def test_fp16_bias(dev, form, mode):
    """The per-tensor product of the legacy API and the other schemes, fp16 bias and output."""
    out, ref = _case(form, mode, 272, True, False, dev, out_dtype=torch.float16, bias=True)
    assert torch.equal(out, ref.to(torch.float16))


@pytest.mark.parametrize("form", ["small", "whole", "halves", "general"])
def test_fp16_bias_gelu(dev, form):
    """GELU against 64 bits: half an ulp of fp16 (2^-11 of the value, 2^-25 below its
    normal range), a few fp32 roundings (2^-20 of it), and for negative x, where 1 +
    erf(x / sqrt 2) cancels, erff's error near -1: below 4 ulp of 1 (2^-21) times |x| / 2
    < 3 wherever the sum is not 0: 1.5e-6."""
    out, ref = _case(form, "tensor", 272, True, False, dev, out_dtype=torch.float16, bias=True, gelu=True)
    err = (out.double() - ref.double()).abs()
    assert torch.all(err <= ref.double().abs() * (2 ** -11 + 2 ** -20) + 1.5e-6 + 2 ** -25)
