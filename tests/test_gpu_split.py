"""GPU parity of the K-split BMM kernel (csrc/bmm_split.h): short grids and
operands of any alignment.

Operands are small integers and scales powers of two, so every product and
every partial sum is exact in fp32 whatever the order (|a b| <= 16, K <= 4200:
sums below 2^17, scales in [1/4, 4], far inside 24 bits): the fp32 output must
equal the 64-bit product bit for bit, and a 16-bit one its single rounding.
Each operand is a view into a larger buffer of NaN codes, at an odd byte
offset and with a padded pitch where `pad` says so, so a byte taken from
outside the operand shows.
"""
from __future__ import annotations

import pytest
import torch

from practice_cuda_amd.impls.hip_per_block import hip_per_block_bmm
from practice_cuda_amd.impls.hip_per_channel import hip_per_channel_bmm
from practice_cuda_amd.impls.hip_per_tensor import hip_per_tensor_bmm
from practice_cuda_amd.registry import QuantResult

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


def _embed(values: torch.Tensor, pad: int, offset: int, dev) -> torch.Tensor:
    """values [B, R, C] (fp8) as a view with row pitch C + pad, `offset` bytes into a buffer of NaN codes."""
    b, r, c = values.shape
    pitch = c + pad
    buf = torch.full((offset + b * r * pitch + 64,), 0x7F, dtype=torch.uint8, device=dev)
    view = torch.as_strided(buf, (b, r, c), (r * pitch, pitch, 1), offset)
    view.copy_(values.view(torch.uint8).to(dev))
    return view.view(E4M3)


def _operand(b, rows, cols, major_last, pad, offset, g, dev):
    """(fp64 values [b, rows, cols], fp8 view contiguous along the last dim or the one before)."""
    v = torch.randint(-4, 5, (b, rows, cols), generator=g).float()
    store = v if major_last else v.transpose(-1, -2).contiguous()
    q = _embed(store.to(E4M3), pad, offset, dev)
    return v.double(), q if major_last else q.transpose(-1, -2)


def _pow2(shape, g):
    return 2.0 ** torch.randint(-2, 3, shape, generator=g).float()


def _case(scheme, shape, a_k, b_k, dev, pad=0, offset=0, bias=None, activation="none", out_dtype=torch.float32,
          seed=0):
    b, m, n, k = shape
    g = torch.Generator().manual_seed(seed)
    va, qa = _operand(b, m, k, a_k, pad, offset, g, dev)
    vb, qb = _operand(b, k, n, not b_k, pad, offset, g, dev)
    if scheme.startswith("block"):
        qbn = int(scheme[5:])
        kb = -(-k // 128)
        sa, sb = _pow2((b, m, kb), g), _pow2((b, kb, -(-n // qbn)), g)
        ref = torch.zeros(b, m, n, dtype=torch.float64)
        for i in range(kb):
            s = slice(128 * i, min(128 * i + 128, k))
            cols = sb[:, i].double().repeat_interleave(qbn, dim=1)[:, None, :n]
            ref += (va[:, :, s] @ vb[:, s]) * sa[:, :, i, None].double() * cols
        ra = QuantResult(qa, sa.to(dev), "t", "block", {"block_m": 1, "block_n": 128})
        rb = QuantResult(qb, sb.to(dev), "t", "block", {"block_m": 128, "block_n": qbn})
        fn = hip_per_block_bmm
    elif scheme == "channel":
        sa, sb = _pow2((b, m), g), _pow2((b, n), g)
        ref = (va @ vb) * sa[:, :, None].double() * sb[:, None].double()
        ra = QuantResult(qa, sa.to(dev), "t", "channel", {"channel_axis": -2})
        rb = QuantResult(qb, sb.to(dev), "t", "channel", {"channel_axis": -1})
        fn = hip_per_channel_bmm
    else:
        sa, sb = _pow2((), g), _pow2((), g)
        ref = (va @ vb) * float(sa * sb)
        ra, rb = QuantResult(qa, sa.to(dev), "t", "tensor"), QuantResult(qb, sb.to(dev), "t", "tensor")
        fn = hip_per_tensor_bmm
    if bias is not None:
        ref = ref + bias.double()
    if activation == "gelu":
        ref = torch.nn.functional.gelu(ref)
    print(f"split {scheme} {shape} a_k={a_k} b_k={b_k} pad={pad} offset={offset}", flush=True)
    out = fn(ra, rb, out_dtype=out_dtype, bias=None if bias is None else bias.to(dev), activation=activation)
    torch.cuda.synchronize()
    return out.cpu(), ref


LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]
SCHEMES = ["block128", "block16", "block1", "channel", "tensor"]
# every tile of the kernel (rows <= 16 / 32 / more; few, about one and several
# workgroups per CU), its edges, and K below, at and past whole K steps and
# the eight waves' shares
SHAPES = [(1, 16, 32, 256), (1, 17, 64, 1024), (2, 33, 80, 1040), (1, 64, 16384, 256), (1, 130, 6656, 272),
          (1, 32, 16400, 144), (1, 16, 16384, 144), (1, 512, 4096, 384), (1, 16, 48, 4096)]
# nothing aligned: the smallest rows, one byte past and short of a K step / tile
ODD = [(1, 16, 16, 16), (1, 17, 17, 17), (3, 16, 31, 127), (2, 65, 33, 129), (1, 63, 65, 255), (2, 200, 301, 1031),
       (1, 1025, 1027, 130)]


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("shape", SHAPES)
def test_split_exact(dev, shape, scheme, a_k, b_k):
    out, ref = _case(scheme, shape, a_k, b_k, dev, pad=16)
    assert torch.equal(out, ref.float())


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("scheme", ["block128", "block1", "channel", "tensor"])
@pytest.mark.parametrize("shape", ODD)
def test_split_unaligned_exact(dev, shape, scheme, a_k, b_k):
    for pad, offset in ((0, 0), (3, 5)):
        out, ref = _case(scheme, shape, a_k, b_k, dev, pad=pad, offset=offset)
        assert torch.equal(out, ref.float())


@pytest.mark.parametrize("rows", [1, 5])
def test_split_few_rows(dev, rows):
    """One and a few rows (K-major A), which the MN-major layout cannot hold."""
    for scheme in SCHEMES:
        out, ref = _case(scheme, (2, rows, 100, 1031), True, False, dev)
        assert torch.equal(out, ref.float())


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float8_e4m3fn])
@pytest.mark.parametrize("n", [64, 77])
def test_split_epilogue(dev, out_dtype, n):
    """Bias (16-bit, fp32, broadcast rows) and every output type: one rounding of
    the exact sum. The bias is a multiple of 1/4, so the sum stays exact."""
    g = torch.Generator().manual_seed(3)
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        bias = (torch.randint(-64, 65, (1, 1, n), generator=g) / 4).to(dt).expand(1, 40, n)
        out, ref = _case("channel", (1, 40, n, 300), True, False, dev, bias=bias, out_dtype=out_dtype)
        want = ref.float()
        if out_dtype == torch.float8_e4m3fn:
            want = want.clamp(-448, 448)
        assert torch.equal(out.float(), want.to(out_dtype).float())


def test_split_gelu(dev):
    """GELU against 64 bits: the bf16 rounding (8 significant bits: half an ulp is
    at most 2^-8 of the value), a few fp32 roundings (2^-20 of it), and for
    negative x, where 1 + erf(x / sqrt 2) cancels, erff's error near -1: below
    4 ulp of 1 (2^-21) times |x| / 2 < 3 wherever the sum is not 0: 1.5e-6."""
    out, ref = _case("tensor", (1, 40, 77, 300), True, False, dev, activation="gelu", out_dtype=torch.bfloat16)
    assert torch.all((out.double() - ref).abs() <= ref.abs() * (2 ** -8 + 2 ** -20) + 1.5e-6)


def test_split_deterministic(dev):
    """The partial sums meet in a fixed order: the same bits on every call."""
    g = torch.Generator().manual_seed(9)
    a = torch.randn(1, 48, 4096, generator=g).to(E4M3).to(dev)
    b = torch.randn(1, 4096, 1024, generator=g).to(E4M3).to(dev)
    s = torch.full((), 0.37, device=dev)
    qa, qb = QuantResult(a, s, "t", "tensor"), QuantResult(b, s, "t", "tensor")
    first = hip_per_tensor_bmm(qa, qb, out_dtype=torch.float32)
    for _ in range(3):
        assert torch.equal(hip_per_tensor_bmm(qa, qb, out_dtype=torch.float32), first)
