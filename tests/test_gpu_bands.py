"""Frequency bands on both sides of the line between eight channels a thread and
one: the same sums in the same order, so a channels-last map gives the bits that the
same map in another layout gives, which runs one channel a thread."""

import pytest
import torch
import torch.nn.functional as F

from trifusion_amd.ops import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,c,t,f", [(1, 64, 3, 64), (1, 64, 3, 63), (2, 72, 5, 129), (1, 64, 512, 9), (1, 64, 511, 9),
                                     (2, 16, 1024, 17), (1, 16, 2047, 17), (8, 8, 2000, 65), (1, 12, 3000, 65)])
def test_layouts_agree(b, c, t, f, dtype):
    x = torch.randn(b, t, f, c, device=DEV, generator=torch.Generator(DEV).manual_seed(c + t)).to(dtype)
    x = x.permute(0, 3, 1, 2)
    y = ops.bands(x)
    assert torch.equal(y, ops.bands(x.contiguous()))
    ref = F.adaptive_avg_pool2d(x.double(), (t, 8)).permute(0, 2, 3, 1)
    # fp32 sums of up to 18 values, then a rounding
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-23
    assert ((y.double() - ref).abs() <= unit * ref.abs() + 20 * 2.0**-24 * x.double().abs().max()).all()
