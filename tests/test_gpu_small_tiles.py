"""GPU parity of the 128 x 128-tile form of the wide BMM kernel (two
workgroups per CU): grids past the K-split kernel's that 256 x 256 tiles would
not fill. Exact-integer operands, as in test_gpu_split.py: the fp32 output
equals the 64-bit product bit for bit."""
from __future__ import annotations

import pytest
import torch

from test_gpu_split import LAYOUTS, SCHEMES, _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a_k,b_k", LAYOUTS)
@pytest.mark.parametrize("scheme", SCHEMES)
@pytest.mark.parametrize("shape", [(1, 1104, 2304, 272), (2, 1040, 1168, 256)])
def test_small_tiles_exact(dev, shape, scheme, a_k, b_k):
    """A ragged and a whole last K step, partial last tiles in both directions."""
    out, ref = _case(scheme, shape, a_k, b_k, dev, pad=16)
    assert torch.equal(out, ref.float())
    out, ref = _case(scheme, shape, a_k, b_k, dev, pad=16, out_dtype=torch.bfloat16)
    assert torch.equal(out, ref.to(torch.bfloat16))
