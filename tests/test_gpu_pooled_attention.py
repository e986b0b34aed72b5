"""Pooled attention and the query-read merge at the edges of their tiles: one,
two, four and eight waves per workgroup, ragged and empty key prefixes, both
head dims, values that are not finite, and many-tile query reads, against the
oracle's formulation in float64."""

import math
from types import SimpleNamespace

import pytest
import torch

from trifusion_amd.kernels.block import pooled_attention, query_read

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def attend(q, k, v, mask):
    s = (q.double() @ k.double().transpose(-1, -2)) / math.sqrt(q.shape[-1])
    return s.masked_fill(~mask, -math.inf).softmax(-1) @ v.double()


def rotated(qkv, cos, sin, heads):
    b, t, width = qkv.shape
    d = width // (3 * heads)
    x = qkv.view(b, t, 3, heads, d).permute(2, 0, 3, 1, 4).float()
    a, z = x[:2, ..., 0::2], x[:2, ..., 1::2]
    rot = torch.stack((a * cos - z * sin, a * sin + z * cos), -1).flatten(-2).to(BF)
    return rot[0], rot[1], x[2]


def tables(t, hd):
    phase = torch.arange(t).float()[:, None] * 10000.0 ** (-torch.arange(0, hd, 2).float() / hd)[None, :]
    return phase.cos(), phase.sin()


@pytest.mark.parametrize("heads,hd", [(3, 64), (2, 32)])
@pytest.mark.parametrize("t,low", [(1, [1, 0]), (31, [31, 2]), (32, [32, 1]), (33, [33, 32]), (65, [64, 65]),
                                   (128, [97, 128]), (129, [129, 33]), (451, [451, 257])])
def test_attention_tiles(t, low, heads, hd):
    g = torch.Generator().manual_seed(100 * t + hd)
    low = torch.tensor(low)
    qkv = (2 * torch.randn(2, t, 3 * heads * hd, generator=g)).to(BF)
    cos, sin = tables(t, hd)
    grids = SimpleNamespace(rope_cos=cos.to(DEV), rope_sin=sin.to(DEV), low_lengths=low.to(DEV))
    y = pooled_attention(qkv.to(DEV), grids, heads).cpu().double()
    q, k, v = rotated(qkv, cos, sin, heads)
    mask = (torch.arange(t)[None, :] < low[:, None])[:, None, None, :]
    some = low > 0
    ref = attend(q, k, v, mask).transpose(1, 2).reshape(2, t, heads * hd)
    # half a bf16 step of the result, and fp32 sums of values up to ~8 (scores up
    # to ~50 in magnitude: relative error of a probability below 50 * 2^-22)
    err = (y - ref).abs()[some]
    assert (err <= ref.abs()[some] * 2.0**-8 + 8 * 50 * 2.0**-22).all(), err.max()
    assert not y[~some].any()


def test_attention_infinite_value():
    """A value row that is not finite reaches the queries that attend to it as in
    IEEE arithmetic, and a row past the key prefix reaches none."""
    t, heads, hd = 70, 1, 64
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(2, t, 3 * heads * hd, generator=g).to(BF)
    qkv[0, 3, 2 * hd + 5] = math.inf
    qkv[0, 40, 2 * hd + 7] = math.nan
    qkv[1, 60, 2 * hd :] = math.inf
    low = torch.tensor([t, 60])
    cos, sin = tables(t, hd)
    grids = SimpleNamespace(rope_cos=cos.to(DEV), rope_sin=sin.to(DEV), low_lengths=low.to(DEV))
    y = pooled_attention(qkv.to(DEV), grids, heads).cpu()
    assert torch.isposinf(y[0, :, 5]).all() and y[0, :, 7].isnan().all()
    rest = [i for i in range(hd) if i not in (5, 7)]
    assert y[0][:, rest].isfinite().all() and y[1].isfinite().all()
    clean = qkv.clone()
    clean[0, 3, 2 * hd + 5] = 0
    clean[0, 40, 2 * hd + 7] = 0
    clean[1, 60, 2 * hd :] = 0
    z = pooled_attention(clean.to(DEV), grids, heads).cpu()
    # the other dims run the fp32 product on the affected tiles: equal up to its rounding
    assert (y[0][:, rest].float() - z[0][:, rest].float()).abs().max() <= 2.0**-8 * z[0].abs().max()
    assert torch.equal(y[1], z[1])


@pytest.mark.parametrize("t,lengths", [(64, [64, 0]), (520, [513, 1]), (2049, [2049, 700])])
def test_query_read_merges_many_tiles(t, lengths):
    g = torch.Generator().manual_seed(t)
    q = torch.randn(10, 256, generator=g).to(BF)
    kv = torch.randn(2, t, 512, generator=g).to(BF)
    lengths = torch.tensor(lengths)
    y = query_read(q.to(DEV), kv.to(DEV), lengths.to(DEV), 8).cpu().double()
    k, v = kv.view(2, t, 2, 8, 32).permute(2, 0, 3, 1, 4).unbind(0)
    qq = q.view(10, 8, 32).transpose(0, 1)[None].expand(2, -1, -1, -1)
    mask = (torch.arange(t)[None, :] < lengths[:, None])[:, None, None, :]
    ref = attend(qq, k, v, mask).transpose(1, 2).reshape(2, 10, 256)
    some = lengths > 0
    err = (y - ref).abs()[some]
    # half a bf16 step and fp32 sums of values up to ~5
    assert (err <= ref.abs()[some] * 2.0**-8 + 5 * 64 * 2.0**-23).all(), err.max()
    assert not y[~some].any()


def test_small_probabilities_are_rounded_once():
    """Two keys, scores 0 and -x for x in 40..70, values 0 and 1: the output is
    e^-x / (1 + e^-x), in bf16. The score, the sum and the reciprocal are exact, so
    what stands between it and the correctly rounded value is the exponential. One
    that is off by a unit of 2^-23 everywhere would turn one result in 2^15 (twice the
    error over the least step of a bf16 mantissa, 2^-7): 2 to 3 of 65 536, and 4 are
    allowed. One whose argument is a rounded product turned 16."""
    t, heads, hd = 4096, 16, 64
    g = torch.Generator().manual_seed(8)
    # x = (a b + c) / 8 in multiples of 2^-12
    a, b = (torch.rand(t, heads, generator=g) * 4 + 16).to(BF), (torch.rand(heads, generator=g) * 6 + 21).to(BF)
    c = (torch.rand(t, heads, generator=g) / 2 + 0.5).to(BF)
    qkv = torch.zeros(1, t, 3, heads, hd, dtype=BF)
    qkv[0, :, 0, :, 0], qkv[0, :, 0, :, 2] = a, c
    qkv[0, 1, 1, :, 0], qkv[0, 1, 1, :, 2] = -b, -1
    qkv[0, 1, 2, :, 0] = 1
    cos, sin = torch.ones(t, hd // 2), torch.zeros(t, hd // 2)
    grids = SimpleNamespace(rope_cos=cos.to(DEV), rope_sin=sin.to(DEV), low_lengths=torch.tensor([2], device=DEV))
    y = pooled_attention(qkv.reshape(1, t, -1).to(DEV), grids, heads).cpu().view(t, heads, hd)[..., 0]
    x = (a.double() * b.double() + c.double()) / 8
    ref = (1 / (1 + x.exp())).float().to(BF)
    differ = int((y != ref).sum())
    print(f"{differ} of {y.numel()} results not the correctly rounded ones", flush=True)
    assert differ <= 4


@pytest.mark.parametrize("b,t", [(1, 65), (1, 129), (20, 256), (20, 257), (64, 768), (64, 800)])
def test_query_read_on_both_merges(b, t):
    """Either side of the line between one thread per (query, dim) and eight groups:
    up to 2 tiles of 64 keys, or one tile for every 40 (head, batch row)s."""
    g = torch.Generator().manual_seed(b + t)
    q = torch.randn(10, 256, generator=g).to(BF)
    kv = torch.randn(b, t, 512, generator=g).to(BF)
    lengths = torch.randint(0, t + 1, (b,), generator=g)
    lengths[0] = t
    y = query_read(q.to(DEV), kv.to(DEV), lengths.to(DEV), 8).cpu().double()
    k, v = kv.view(b, t, 2, 8, 32).permute(2, 0, 3, 1, 4).unbind(0)
    qq = q.view(10, 8, 32).transpose(0, 1)[None].expand(b, -1, -1, -1)
    mask = (torch.arange(t)[None, :] < lengths[:, None])[:, None, None, :]
    ref = attend(qq, k, v, mask).transpose(1, 2).reshape(b, 10, 256)
    some = lengths > 0
    err = (y - ref).abs()[some]
    # half a bf16 step and fp32 sums of values up to ~5
    assert (err <= ref.abs()[some] * 2.0**-8 + 5 * 64 * 2.0**-23).all(), err.max()
    assert not y[~some].any()
