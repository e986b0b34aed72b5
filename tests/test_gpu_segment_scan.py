"""Segment scans over growing steps: a segment whose decay factor leaves the fp32
range on its own, applied to a state of 0 or a small one, gives what the serial walk
gives, whose factors stay finite chunk by chunk."""

import ctypes

import pytest
import torch

from oracle.recurrence import max_rel
from trifusion_amd import _lib
from trifusion_amd.mamba_fused import build_args, fused_mamba
from trifusion_amd.synthetic import clip_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("entering", ["zero", "small"])
@pytest.mark.parametrize("state,dtype", [(64, torch.float32), (128, torch.bfloat16)])
def test_growth_past_the_fp32_range(state, dtype, entering):
    t = 640  # segments of two chunks
    args = [x.to(DEV) for x in clip_inputs(1, t, heads=2, head_dim=64, state=state, dtype=dtype,
                                           ctrl_dtype=torch.float32, seed=6)]
    v, adt = args[2].clone(), args[3].clone()
    # the second segment grows by 2^200, 2^100 a chunk; nothing is added meanwhile
    adt[..., 128:256] = 100 / 64 / 1.4427
    adt[..., :128] = -1e-3
    v[:, 128:256] = 0
    v[:, :128] = 0 if entering == "zero" else v[:, :128] * 2.0**-100
    args[2], args[3] = v, adt
    out = torch.empty(v.shape, device=DEV)
    y = fused_mamba(*args, out=out)
    serial = torch.empty_like(out)
    a = build_args(*args, serial, None, "auto")
    assert _lib.load().tf_fused_mamba_split_size(ctypes.byref(a)) > 0  # the operator splits this shape
    _lib.check(_lib.load().tf_fused_mamba(ctypes.byref(a), _lib.stream_of(out)), "fused_mamba")
    assert serial.isfinite().all() and y.isfinite().all()
    for part in (slice(0, 128), slice(128, 256), slice(256, 320), slice(576, t)):
        assert max_rel(y[:, part], serial[:, part]) <= (1e-5 if dtype == torch.float32 else 1e-3)
