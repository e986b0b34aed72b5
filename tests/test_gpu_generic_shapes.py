"""The generic recurrence kernel at the edges of its tiles: state dims that are
not a multiple of 32 (through the C ABI, which takes any even N <= 128 and any
P <= 64), strides it cannot read four elements at a time, every dtype, ragged
lengths, both directions, and values that are not finite."""

import ctypes
import math

import pytest
import torch

from oracle.recurrence import fused_mamba_chunked, fused_mamba_f64, fused_mamba_reversed, max_rel
from trifusion_amd import _lib
from trifusion_amd.mamba_fused import fused_mamba
from trifusion_amd.synthetic import clip_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def call(args, out, lengths=None, reverse=False):
    """The C entry directly: the Python wrapper takes only N and P of the model."""
    q, k, v, adt, dt, trap, qb, kb, angles, d, z = args
    a = _lib.MambaArgs()
    for name, t in (("q", q), ("k", k), ("v", v), ("adt", adt), ("dt", dt), ("trap", trap), ("angles", angles),
                    ("z", z), ("out", out)):
        setattr(a, name, t.data_ptr())
        setattr(a, name + "_dtype", _lib.dtype_code(t, "test"))
        getattr(a, name + "_stride")[:] = t.stride()
    a.qb, a.kb, a.d = qb.data_ptr(), kb.data_ptr(), d.data_ptr()
    a.lengths = None if lengths is None else lengths.data_ptr()
    a.batch, a.time, a.heads, a.head_dim = v.shape
    a.qk_heads, a.state, a.rotary = q.shape[2], q.shape[3], angles.shape[3]
    a.variant, a.reverse = _lib.VARIANTS["generic"], int(reverse)
    _lib.check(_lib.load().tf_fused_mamba(ctypes.byref(a), _lib.stream_of(v)), "fused_mamba")
    return out


def on(args):
    return tuple(x.to(DEV) for x in args)


@pytest.mark.parametrize("n,p,r", [(2, 1, 1), (6, 5, 3), (18, 33, 9), (32, 32, 16), (34, 64, 17), (66, 63, 20),
                                   (96, 32, 24), (98, 64, 49), (128, 64, 64)])
@pytest.mark.parametrize("t", [1, 64, 97])
def test_shapes_against_float64(n, p, r, t):
    args = clip_inputs(2, t, heads=2, head_dim=p, state=n, rotary=r, dtype=torch.float32, seed=n + t)
    out = torch.full((2, t, 2, p), math.nan, device=DEV)
    call(on(args), out)
    ref = fused_mamba_f64(*args)
    # 32-bit sums of up to 128 + 64 terms; the walk carries them over two chunks
    assert max_rel(out.cpu(), ref) <= 5e-6


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_lengths_and_strides(dtype, reverse):
    args = clip_inputs(5, 130, heads=4, head_dim=64, state=64, dtype=dtype, ctrl_dtype=torch.float32, qk_heads=2,
                       seed=3)
    lengths = torch.tensor([130, 0, 1, 33, 64])
    # rows of every operand at odd offsets and strides: no four-element loads
    odd = []
    for i, x in enumerate(on(args)):
        if i in (0, 1, 2, 10):
            wide = torch.full((*x.shape[:-1], x.shape[-1] + 3), math.nan, device=DEV, dtype=x.dtype)
            wide[..., 1 : 1 + x.shape[-1]] = x
            x = wide[..., 1 : 1 + x.shape[-1]]
        odd.append(x)
    even = torch.full((5, 130, 4, 64), math.nan, device=DEV)
    strided = torch.full((5, 130, 4, 65), math.nan, device=DEV)[..., 1:]
    call(on(args), even, lengths.to(DEV), reverse)
    call(tuple(odd), strided, lengths.to(DEV), reverse)
    assert torch.equal(even, strided)  # the same arithmetic whatever the loads
    ref = (fused_mamba_reversed if reverse else fused_mamba_chunked)(*args, lengths=lengths)
    assert max_rel(even.cpu(), ref) <= (1e-5 if dtype == torch.float32 else 1e-3)
    for i, length in enumerate(lengths.tolist()):
        assert not even[i, length:].any()


def test_infinite_value_is_causal():
    """A row of v that is not finite leaves every earlier row as it was."""
    args = on(clip_inputs(1, 100, heads=1, head_dim=64, state=64, dtype=torch.float32, seed=9))
    clean = fused_mamba(*args)
    for at, bad in ((40, math.inf), (70, math.nan)):
        v = args[2].clone()
        v[0, at, 0, 3] = bad
        y = fused_mamba(*args[:2], v, *args[3:])
        assert max_rel(y[:, :at].cpu(), clean[:, :at].cpu()) <= 5e-6
        assert not y[0, at, 0, 3].isfinite() and not y[0, at + 1 :, 0, 3].isfinite().any()
        rest = [i for i in range(64) if i != 3]
        assert max_rel(y[..., rest].cpu(), clean[..., rest].cpu()) <= 5e-6


@pytest.mark.parametrize("reverse", [False, True])
@pytest.mark.parametrize("b,t,h,n,p,r,lengths", [(1, 257, 2, 64, 64, 16, None), (3, 900, 4, 128, 64, 32, [900, 130, 0]),
                                                 (2, 640, 1, 32, 32, 9, [385, 640]), (1, 1600, 3, 16, 32, 8, None)])
def test_segments_match_serial_walk(b, t, h, n, p, r, lengths, reverse):
    """Chunk-parallel (the operator brings scratch) against the serial walk (none given)
    and the oracle: fp32 sums of the same terms, the carried state composed in
    another order and its rotary rows turned once more per segment."""
    args = clip_inputs(b, t, heads=h, head_dim=p, state=n, rotary=r, dtype=torch.float32, seed=t)
    dev = on(args)
    dl = None if lengths is None else torch.tensor(lengths, device=DEV)
    serial = call(dev, torch.full((b, t, h, p), math.nan, device=DEV), dl, reverse)
    out = torch.full((b, t, h, p), math.nan, device=DEV)
    y = fused_mamba(*dev, out=out, lengths=dl, reverse=reverse)
    assert max_rel(y.cpu(), serial.cpu()) <= 5e-6
    hl = None if lengths is None else torch.tensor(lengths)
    ref = (fused_mamba_reversed if reverse else fused_mamba_chunked)(*args, lengths=hl)
    assert max_rel(y.cpu(), ref) <= 1e-5
    if lengths is not None:
        for i, length in enumerate(lengths):
            assert not y[i, length:].any()


@pytest.mark.parametrize("n", [16, 32])
def test_infinite_value_gives_infinities(n):
    """Keys and queries that are all positive and an infinite value: every later
    output of its head dim is infinite, with the sign of the gate, also where the
    state dim is padded to a whole tile. Segments turn the states they hand on,
    which adds infinities of both signs: from the second one on (row 192) the same
    outputs are not finite, and no others. (The decay of a chunk stays above 0: times
    infinity that is not a number.)"""
    q, k, v, adt, dt, trap, qb, kb, angles, d, z = clip_inputs(1, 300, heads=1, head_dim=32, state=n, rotary=n // 4,
                                                               dtype=torch.float32, seed=n)
    v[0, 10, 0, 3] = math.inf
    args = on((q.abs(), k.abs(), v, 0.05 * adt, dt, trap, qb, kb, torch.zeros_like(angles), d, z))
    expect = math.inf * z[0, 10:, 0, 3].sign()
    serial, split = call(args, torch.full((1, 300, 1, 32), math.nan, device=DEV)), fused_mamba(*args)
    assert torch.equal(serial[0, 10:, 0, 3].cpu(), expect)
    assert torch.equal(split[0, 10:192, 0, 3].cpu(), expect[:182]) and not split[0, 192:, 0, 3].isfinite().any()
    for y in (serial, split):
        assert y[..., :3].isfinite().all() and y[..., 4:].isfinite().all() and y[:, :10].isfinite().all()


@pytest.mark.parametrize("at", [10, 300, 630])
@pytest.mark.parametrize("bad", [math.inf, math.nan])
def test_value_that_is_not_finite_in_segments(at, bad):
    """In segments (640 rows of one unit: five of two chunks) a row of v that is not
    finite leaves earlier rows and other head dims as they were, and no later output
    of its own is finite."""
    args = on(clip_inputs(1, 640, heads=1, head_dim=64, state=64, dtype=torch.float32, seed=9))
    clean = fused_mamba(*args)
    v = args[2].clone()
    v[0, at, 0, 3] = bad
    y = fused_mamba(*args[:2], v, *args[3:])
    assert max_rel(y[:, :at].cpu(), clean[:, :at].cpu()) <= 5e-6
    assert not y[0, at:, 0, 3].isfinite().any()
    rest = [i for i in range(64) if i != 3]
    assert max_rel(y[..., rest].cpu(), clean[..., rest].cpu()) <= 5e-6


@pytest.mark.parametrize("reverse", [False, True])
def test_positive_decay_in_segments(reverse):
    """A fifth of the steps grow, in segments, against the fp32 oracle."""
    args = list(clip_inputs(1, 900, heads=4, head_dim=64, state=64, dtype=torch.float32, seed=44))
    flip = torch.rand(args[3].shape, generator=torch.Generator().manual_seed(1)) < 0.2
    args[3] = torch.where(flip, -0.25 * args[3], args[3])
    y = fused_mamba(*on(args), reverse=reverse)
    ref = (fused_mamba_reversed if reverse else fused_mamba_chunked)(*args)
    assert max_rel(y.cpu(), ref) <= 1e-5
