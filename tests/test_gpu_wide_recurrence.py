"""The N = 128, P = 64 recurrence kernel at the edges of its chunks, segments and
input forms, against the oracle and its own serial walk."""

import ctypes

import pytest
import torch

from oracle.recurrence import fused_mamba_chunked, fused_mamba_reversed, max_rel, rel_fro
from trifusion_amd import _lib
from trifusion_amd.mamba_fused import build_args, fused_mamba
from trifusion_amd.synthetic import clip_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"
MAX_REL = 1e-3  # the recurrence's tolerance


def padded(x, before, after):
    """``x`` inside a wider buffer of NaN: rows of another stride and alignment."""
    wide = torch.full((*x.shape[:-1], before + x.shape[-1] + after), float("nan"), device=x.device, dtype=x.dtype)
    wide[..., before : before + x.shape[-1]] = x
    return wide[..., before : before + x.shape[-1]]


# rotary: a full table of 32, above it (64 rows of table), not a multiple of 8,
# none in the last piece; angles: aligned pieces or single elements; controls fp32
# or (as the model's raw projection) bf16; q/k/v/z rows 16- or 8-byte aligned
@pytest.mark.parametrize("rotary", [32, 64, 33, 9, 1])
@pytest.mark.parametrize("form", ["fp32", "bf16", "odd"])
@pytest.mark.parametrize("reverse", [False, True])
def test_forms_and_edges(rotary, form, reverse):
    lens = [400, 0, 1, 16, 17, 63, 64, 65, 129]
    b, t, h = len(lens), 400, 2
    print(f"case rotary={rotary} form={form} reverse={reverse}", flush=True)
    args = list(clip_inputs(b, t, heads=h, head_dim=64, state=128, rotary=rotary, seed=rotary))
    if form == "bf16":  # trapezoid and angles bf16; raw bf16 controls are the model's own tests
        args[5], args[8] = args[5].to(torch.bfloat16), args[8].to(torch.bfloat16)
    dev = [x.to(DEV) for x in args]
    if form == "odd":
        dev[8] = padded(dev[8], 1, 2)
        for i in (0, 1, 2, 10):
            dev[i] = padded(dev[i], 4, 8)
    lengths = torch.tensor(lens, dtype=torch.int64)
    ref = (fused_mamba_reversed if reverse else fused_mamba_chunked)(*args, lengths=lengths, out_dtype=torch.float32)
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((b, t, h, 64), float("nan"), device=DEV, dtype=dtype)
        y = fused_mamba(*dev, lengths=lengths.to(DEV), reverse=reverse, out=out)  # segments
        a = build_args(*dev, torch.full_like(out, float("nan")), lengths.to(DEV), "auto", reverse=reverse)
        assert _lib.load().tf_fused_mamba_workspace_size(ctypes.byref(a)) > 0
        serial = torch.full_like(out, float("nan"))
        a = build_args(*dev, serial, lengths.to(DEV), "auto", reverse=reverse)  # no workspace: one workgroup a unit
        _lib.check(_lib.load().tf_fused_mamba(ctypes.byref(a), _lib.stream_of(out)), "fused_mamba")
        for got in (y, serial):
            # fp32: the tolerance; bf16: half a unit of the rounded result more
            assert max_rel(got.float().cpu(), ref) <= MAX_REL + (2.0**-8 if dtype == torch.bfloat16 else 0)
            for i, length in enumerate(lens):
                assert not got[i, length:].any()


def test_nan_angle_stays_in_later_rows():
    args = [x.to(DEV) for x in clip_inputs(1, 400, heads=1, head_dim=64, state=128, seed=4)]
    clean = fused_mamba(*args)
    args[8] = args[8].clone()
    args[8][0, 200, 0, 5] = float("nan")
    y = fused_mamba(*args)
    assert torch.equal(y[:, :200], clean[:, :200]) and y[0, 200:].isnan().any(-1).all()


def serial_walk(dev, out, lengths=None, **kw):
    """The C entry without a workspace: one workgroup a unit."""
    a = build_args(*dev, out, lengths, "auto", **kw)
    assert _lib.load().tf_fused_mamba_workspace_size(ctypes.byref(a)) > 0  # the operator splits this shape
    _lib.check(_lib.load().tf_fused_mamba(ctypes.byref(a), _lib.stream_of(out)), "fused_mamba")
    return out


def test_phase_of_many_small_steps():
    """28 800 steps that all turn the same way by ~1e-3 revolutions: the phase sum
    is held to the fp64 one by the results it moves. With every increment rounded
    to the nearest 2^-32 revolutions the sum strays by 0.3 sqrt(28 800) units, 7e-8
    rad, less than the fp32 phase itself, so what remains are q and k elements that
    round to the other bf16 neighbour, in the segmented form also because it rounds
    keys in each segment's own phase. Rounding towards 0 would add 2e-5 rad."""
    args = list(clip_inputs(1, 28800, heads=1, head_dim=64, state=128, rotary=32, seed=3))
    args[8] = args[8].abs() * 0.02
    dev = [x.to(DEV) for x in args]
    out = torch.empty(dev[2].shape, device=DEV)
    split = fused_mamba(*dev, out=out).cpu()
    serial = serial_walk(dev, torch.empty_like(out)).cpu()
    ref = fused_mamba_chunked(*args)
    print(f"rel_fro segments {rel_fro(split, ref):.3e} serial {rel_fro(serial, ref):.3e}", flush=True)
    assert rel_fro(split, ref) <= 1.2e-4 and rel_fro(serial, ref) <= 1.2e-4
