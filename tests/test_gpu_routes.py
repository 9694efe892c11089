"""Which kernel a product takes, seen in its bits: with channel scales the tiled
kernels sum K in one accumulator per output and the K-split kernel sums its
waves' shares, so on random operands their results differ. A product whose
own grid is in question is compared with the same product as one of a batch
that is far past the K-split kernel's range."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest
import torch

from practice_cuda_amd.impls.hip_per_channel import hip_per_channel_bmm
from practice_cuda_amd.registry import QuantResult

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _operands(m, n, k, dev, batch):
    g = torch.Generator(device=dev).manual_seed(m + n + k)
    # exponents over most of the format's range, so that fp32 sums round
    spread = lambda *s: (torch.randn(s, generator=g, device=dev) *  # noqa: E731
                         2.0 ** torch.randint(-6, 7, s, generator=g, device=dev)).to(E4M3)
    a, b = spread(1, m, k), spread(1, k, n)
    sa, sb = ((torch.rand(1, d, generator=g, device=dev) + 0.5) / 64 for d in (m, n))
    rep = lambda t: t.repeat(batch, *([1] * (t.dim() - 1)))  # noqa: E731
    return (QuantResult(rep(a.view(torch.uint8)).view(E4M3), rep(sa), "t", "channel", {"channel_axis": -2}),
            QuantResult(rep(b.view(torch.uint8)).view(E4M3), rep(sb), "t", "channel", {"channel_axis": -1}))


def same_bits_as_tiled(m, n, k, dev, out_dtype=torch.float16):
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    tiles = -(-m // 64) * -(-n // 64)
    out = hip_per_channel_bmm(*_operands(m, n, k, dev, 1), out_dtype=out_dtype)
    tiled = hip_per_channel_bmm(*_operands(m, n, k, dev, 4 * cus // tiles + 1), out_dtype=out_dtype)
    return torch.equal(out[0], tiled[0])


def _columns(dev, tiles_per_cu):
    """Columns of a 128-row product with that many 64 x 64 tiles per CU."""
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    return int(tiles_per_cu * cus) // 2 * 64


@pytest.mark.parametrize("tiles_per_cu,k,tiled", [
    (0.5, 256, False), (1, 256, True), (1, 512, False), (1.25, 512, True), (2, 1024, True), (2, 4096, False),
    (2.25, 4096, True)])
def test_short_grid_rule(dev, tiles_per_cu, k, tiled):
    n = _columns(dev, tiles_per_cu)
    print(f"route 128 x {n} x {k}", flush=True)
    assert same_bits_as_tiled(128, n, k, dev) is tiled


def test_short_grid_rule_element_wise_outputs(dev):
    """Outputs that the tiled kernels store element by element, and few rows, keep the wider range."""
    assert not same_bits_as_tiled(128, _columns(dev, 2), 1024, dev, out_dtype=torch.float32)
    assert not same_bits_as_tiled(32, 2 * _columns(dev, 2), 1024, dev)


@pytest.mark.parametrize("switch", ["PCAMD_BMM_SPLIT", "PCAMD_BMM_HALVES"])
def test_switches_keep_short_grids_on_tiles(dev, switch):
    """Each is read once per process, so it runs in one of its own."""
    assert not same_bits_as_tiled(64, 512, 1024, dev)
    code = ("import torch, sys; sys.path[:0] = ['.', 'tests']; from test_gpu_routes import same_bits_as_tiled\n"
            "assert same_bits_as_tiled(64, 512, 1024, torch.device('cuda:0'))")
    print(f"route with {switch}=0", flush=True)
    run = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**os.environ, switch: "0"}, capture_output=True,
                         text=True, timeout=110)
    assert run.returncode == 0, run.stderr
