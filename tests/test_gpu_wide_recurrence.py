"""The N = 128, P = 64 recurrence kernel at the edges of its chunks, segments and
input forms, against the oracle and its own serial walk."""

import ctypes

import pytest
import torch

from oracle.elementwise import mamba_controls, rms_norm
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
# none in the last piece; angles: aligned pieces or single elements; fp32 controls
# (test_model_form has the model's raw bf16 ones); q/k/v/z rows 16- or 8-byte aligned
@pytest.mark.parametrize("rotary", [32, 64, 33, 9, 1])
@pytest.mark.parametrize("form", ["fp32", "bf16", "odd"])
@pytest.mark.parametrize("reverse", [False, True])
def test_forms_and_edges(rotary, form, reverse):
    lens = [400, 0, 1, 16, 17, 63, 64, 65, 129]
    b, t, h = len(lens), 400, 2
    print(f"case rotary={rotary} form={form} reverse={reverse}", flush=True)
    args = list(clip_inputs(b, t, heads=h, head_dim=64, state=128, rotary=rotary, seed=rotary))
    if form == "bf16":  # trapezoid and angles bf16 beside fp32 controls: read element by element
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


def model_operands(b, t, h, rotary, seed):
    """What a Mamba layer's projection hands the recurrence: columns [z | v | k | q |
    ddt | a | trap | angles] of one bf16 buffer, the angles shared by all heads, with
    an fp32 step bias and B/C norm weights. The kernel's packed form reads them."""
    g = torch.Generator().manual_seed(seed)
    n, p = 128, 64
    x = torch.randn(b, t, 2 * h * p + 2 * n + 3 * h + rotary, generator=g)
    x[..., -rotary:] *= 0.3
    x = x.to(torch.bfloat16).to(DEV)
    z, v, k, q, ddt, a, trap, angles = x.split([h * p, h * p, n, n, h, h, h, rotary], -1)
    assert angles.data_ptr() % 16 == 0 and x.shape[-1] % 8 == 0 and rotary % 8 == 0  # pieces of eight angles
    qb, kb = (1 + 0.1 * torch.randn(h, n, generator=g) for _ in range(2))
    wq, wk = (0.5 + torch.rand(n, generator=g) for _ in range(2))
    bias, d = torch.randn(h, generator=g) - 4, torch.ones(h)
    args = (q.unsqueeze(2), k.unsqueeze(2), v.unflatten(-1, (h, p)), a.transpose(1, 2), ddt.transpose(1, 2),
            trap.transpose(1, 2), qb.to(DEV), kb.to(DEV), angles.unsqueeze(2).expand(-1, -1, h, -1), d.to(DEV),
            z.unflatten(-1, (h, p)))
    kw = dict(dt_bias=bias.to(DEV), a_floor=1e-4, q_norm=wq.to(DEV), k_norm=wk.to(DEV), norm_eps=1e-5)
    adt, dt = mamba_controls(a.cpu(), ddt.cpu(), bias, 1e-4)
    ref = [x.cpu() for x in args]
    ref[0], ref[1], ref[3], ref[4] = rms_norm(ref[0], wq, 1e-5), rms_norm(ref[1], wk, 1e-5), adt, dt
    return args, kw, ref


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("rotary", [32, 64, 24])
@pytest.mark.parametrize("b,t,h,lens", [(24, 130, 8, "ragged"), (2, 700, 8, (700, 333)), (1, 1300, 16, None)])
def test_model_form(b, t, h, lens, rotary, reverse):
    """Raw bf16 controls, bf16 trapezoid and angles and fused norms, as every layer of
    the models passes them: 192 units of up to three chunks in one walk each, and few
    units in segments, against the oracle and the serial walk. Where the norm, the
    rotation or the phase differs in its last fp32 bit, a q or k element near the
    middle of two bf16 values rounds to the other one: 2^-8 of that element, so of one
    term of a result (no larger than the largest result), for one element in some 2^13
    (2^-22 against a step of 2^-8, both sides), which is 2^-8 2^-6.5 = 4e-5 of the
    norm; five times that is allowed. Segments round every key in another frame than
    the oracle: two roundings of a key, 2^-9 / sqrt(3) of it at most in root mean
    square, differ by 1.6e-3 of it, and so does what a state hands on, part of a
    result (2e-4 here)."""
    print(f"case B{b} T{t} H{h} R{rotary} reverse={reverse}", flush=True)
    args, kw, ref = model_operands(b, t, h, rotary, seed=b + rotary)
    if lens == "ragged":
        lens = [(37 * i) % (t + 1) for i in range(b - 1)] + [t]
    lengths = None if lens is None else torch.tensor(lens)
    dl = None if lengths is None else lengths.to(DEV)
    out = torch.full((b, t, h, 64), float("nan"), device=DEV)
    y = fused_mamba(*args, out=out, lengths=dl, reverse=reverse, **kw).cpu()
    expect = (fused_mamba_reversed if reverse else fused_mamba_chunked)(*ref, lengths=lengths)
    split = b * h <= 128
    got = [(y, 1.6e-3 if split else 2e-4)]
    if split:
        got.append((serial_walk(args, torch.full_like(out, float("nan")), dl, reverse=reverse, **kw).cpu(), 2e-4))
    for x, bound in got:
        print(f"  max_rel {max_rel(x, expect):.3e} rel_fro {rel_fro(x, expect):.3e}", flush=True)
        assert max_rel(x, expect) <= 2.0**-8 and rel_fro(x, expect) <= bound
    for i, length in enumerate(lens or ()):
        assert not y[i, length:].any()


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("b,t,h", [(24, 130, 8), (1, 700, 8)])
def test_positive_decay(b, t, h, reverse):
    """A fifth of the steps grow: scores are capped at weight 1 inside a chunk, the
    carried state is not (as tests/test_gpu_positive_decay.py has it for N = 64)."""
    args = list(clip_inputs(b, t, heads=h, head_dim=64, state=128, rotary=32, seed=43))
    flip = torch.rand(args[3].shape, generator=torch.Generator().manual_seed(1)) < 0.2
    args[3] = torch.where(flip, -0.25 * args[3], args[3])
    out = torch.empty(b, t, h, 64, device=DEV)
    dev = [x.to(DEV) for x in args]
    got = [fused_mamba(*dev, out=out, reverse=reverse)]
    if b == 1:
        got.append(serial_walk(dev, torch.empty_like(out), reverse=reverse))
    ref = (fused_mamba_reversed if reverse else fused_mamba_chunked)(*args)
    for y in got:
        assert y.isfinite().all() and max_rel(y.cpu(), ref) <= MAX_REL
