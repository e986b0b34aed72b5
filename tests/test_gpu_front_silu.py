"""The front-end stages' SiLU for every bf16 value: a single pixel whose convolution
gives 1 in every channel, so that the norm weights are the values SiLU sees. Its
fp32 error (about one unit) is far below half a bf16 unit, so the result is the
correctly rounded one; below -87, where e^y leaves the normal range, results are
under 2^-119 and only their size is held."""

import math

import pytest
import torch

from trifusion_amd.ops import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("cin,cout,stage", [(1, 32, 1), (64, 128, 1), (64, 128, 2)])
def test_silu_of_every_bf16_value(cin, cout, stage):
    values = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    values = values[values.isfinite()].to(DEV)
    values = torch.cat((values, values.new_zeros(-len(values) % cout)))
    x = torch.zeros(1, cin, 1, 1, device=DEV, dtype=torch.float32 if cin == 1 else torch.bfloat16)
    x[0, 0] = 1
    x = x.contiguous(memory_format=torch.channels_last)
    one = torch.zeros(9, cout, cin, device=DEV, dtype=torch.bfloat16)
    one[4, :, 0] = 1  # the centre tap of the first channel
    lengths = torch.ones(1, device=DEV, dtype=torch.int64)
    got = []
    for nw in values.float().split(cout):
        if stage == 1:
            y = ops.front_conv1(x, one, nw, lengths, 1, 0.0)
        else:
            h = x.new_zeros(1, 1, 1, cout)
            h[..., 0] = 1
            taps = torch.zeros(9, cout, cout, device=DEV, dtype=torch.bfloat16)
            taps[4, :, 0] = 1
            y = ops.front_conv2(h, taps, nw, x, torch.zeros(cout, cin, device=DEV, dtype=torch.bfloat16), lengths, 1, 0.0)
        got.append(y.flatten())
    got, v = torch.cat(got), values.double()
    ref = torch.where(v < -700, -0.0, v / (1 + (-v).exp()))
    differ = got != ref.float().to(torch.bfloat16)
    print(f"{int(differ.sum())} values differ: {values[differ].tolist()[:12]}", flush=True)
    assert not differ[v >= -87].any()
    assert (got[v < -87].double().abs() <= math.ldexp(1, -119)).all()
