"""The native fused_mamba operator refuses what build_args refuses, with the same
exception type, and takes outputs and layouts as it does."""

import pytest
import torch

from trifusion_amd import fused_mamba
from trifusion_amd.mamba_fused import build_args
from trifusion_amd.synthetic import clip_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("q", "k", "v", "adt", "dt", "trap", "qb", "kb", "angles", "d", "z")


def operands():
    return dict(zip(NAMES, clip_inputs(2, 70, heads=4, seed=2, device=DEV)))


def bad(name):
    x, kw = operands(), {}
    h = torch.ones(4, device=DEV)
    n = torch.ones(64, device=DEV)
    if name == "dims":
        x["q"] = x["q"][0]
    elif name == "control_dims":
        x["dt"] = x["dt"][0]
    elif name == "state":
        x["q"] = x["q"][..., :24]
        x["k"] = x["k"][..., :24]
    elif name == "rotary":
        x["angles"] = torch.zeros(2, 70, 4, 33, device=DEV)
    elif name == "qk_shape":
        x["k"] = x["k"][:, :69]
    elif name == "heads":
        x["q"] = x["q"].expand(2, 70, 3, 64)
        x["k"] = x["k"].expand(2, 70, 3, 64)
    elif name == "gate":
        x["z"] = x["z"][:, :, :3]
    elif name == "controls":
        x["trap"] = x["trap"][:, :, :69]
    elif name == "angles":
        x["angles"] = x["angles"][:1]
    elif name == "bias_dtype":
        x["qb"] = x["qb"].double()
    elif name == "bias_stride":
        x["kb"] = x["kb"].t().contiguous().t()
    elif name == "skip":
        x["d"] = x["d"][:3]
    elif name == "lengths":
        kw["lengths"] = torch.ones(2, dtype=torch.int32, device=DEV)
    elif name == "lengths_shape":
        kw["lengths"] = torch.ones(3, dtype=torch.int64, device=DEV)
    elif name == "step_bias":
        kw["dt_bias"] = h[:3]
    elif name == "raw_dtypes":
        x["dt"], kw["dt_bias"] = x["dt"].bfloat16(), h
    elif name == "one_norm":
        kw["q_norm"] = n
    elif name == "norm_shape":
        kw["q_norm"], kw["k_norm"] = n, n[:32]
    elif name == "out_shape":
        kw["out"] = torch.empty(2, 70, 4, 32, device=DEV)
    elif name == "out_dtype":
        kw["out"] = torch.empty(2, 70, 4, 64, device=DEV, dtype=torch.float64)
    elif name == "dtype":
        x["trap"] = x["trap"].double()
    elif name == "device":
        x["d"] = x["d"].cpu()
    elif name == "variant":
        kw["variant"] = "fast"
    return x, kw


@pytest.mark.parametrize("name", ["dims", "control_dims", "state", "rotary", "qk_shape", "heads", "gate", "controls",
                                  "angles", "bias_dtype", "bias_stride", "skip", "lengths", "lengths_shape",
                                  "step_bias", "raw_dtypes", "one_norm", "norm_shape", "out_shape", "out_dtype",
                                  "dtype", "device", "variant"])
def test_refusals_match(name):
    x, kw = bad(name)
    packed = dict(kw)
    out = packed.pop("out", None)
    with pytest.raises(Exception) as want:
        build_args(**x, out=torch.empty_like(x["v"]) if out is None else out, **packed)
    with pytest.raises(Exception) as got:
        fused_mamba(**x, **kw)
    assert type(got.value) is type(want.value)


def test_refused_variant_and_strided_output():
    x = operands()
    with pytest.raises(ValueError):
        fused_mamba(**clip(32), variant="pipe")
    wide = torch.zeros(2, 70, 4, 96, device=DEV, dtype=torch.bfloat16)
    y = fused_mamba(**x, out=wide[..., :64])
    assert y.data_ptr() == wide.data_ptr() and not wide[..., 64:].any()
    assert torch.equal(y, fused_mamba(**x))


def clip(state):
    return dict(zip(NAMES, clip_inputs(1, 20, heads=4, state=state, seed=2, device=DEV)))
