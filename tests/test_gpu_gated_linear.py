"""The gated linear layers (product and SwiGLU or GLU in one kernel) against
float64 at the edges of their tiles, on both tile sizes, and the depthwise kernel
on gated rows against the one that gates."""

import pytest
import torch
import torch.nn.functional as F

from trifusion_amd.kernels.block import depthwise_norm_silu, gated_linear, glu_norm_silu

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize(
    "rows,features,depth",
    # 64-row tiles: one to three stages, a partial tile, nine row tiles; then tiles of
    # 160 (2049, 2176, 4223 rows), 192 (1801, 1920) and 128 rows (3969, 4096): exact,
    # one row over, a partial last group
    [(1, 64, 64), (63, 64, 128), (65, 128, 192), (129, 192, 256), (523, 64, 64), (2049, 1024, 128), (2176, 1024, 64),
     (4223, 1024, 192), (1801, 2816, 64), (1920, 1408, 64), (3969, 1024, 64), (4096, 1024, 128)],
)
@pytest.mark.parametrize("kind", ["swiglu", "glu"])
def test_against_float64(rows, features, depth, kind):
    print(f"case gated_linear {rows} x {features} x {depth} {kind}", flush=True)
    g = torch.Generator().manual_seed(rows + depth)
    x = torch.randn(rows, depth, generator=g).to(torch.bfloat16)
    w = (torch.randn(2 * features, depth, generator=g) * depth**-0.5).to(torch.bfloat16)
    x[-1, -1] = float("inf") if rows > 64 else 1.0  # stays in its row
    y = gated_linear(x.to(DEV), w.to(DEV), kind).cpu()
    c = x.double() @ w.double().t()
    a, b = c[:, :features], c[:, features:]
    ref = F.silu(a) * b if kind == "swiglu" else a * b.sigmoid()
    # each sum within depth 2^-24 of its absolute terms and rounded to bf16 (8
    # significant bits: half a unit is up to 2^-8 of the value), through a gate
    # (silu's slope is at most 1.1, sigmoid's 1/4), then rounded to bf16 again
    err = 2.0**-8 * c.abs() + depth * 2.0**-24 * (x.double().abs() @ w.double().abs().t())
    ea, eb = err[:, :features], err[:, features:]
    bound = (1.1 * ea * (b.abs() + eb) + F.silu(a).abs() * eb) if kind == "swiglu" else (ea + (a.abs() + ea) * eb / 4)
    bound = bound + 2.0**-8 * (ref.abs() + bound) + 2.0**-20 * ref.abs()  # the last: the hardware exponential
    fin = slice(None, -1 if rows > 64 else None)
    assert y.shape == ref.shape and ((y.double() - ref).abs() <= bound)[fin].all()
    if rows > 64:
        assert y[:-1].isfinite().all() and not y[-1].isfinite().all()


@pytest.mark.parametrize("d,k,t", [(64, 3, 1), (1024, 7, 13), (520, 7, 4)])
def test_gated_rows_equal_gating_in_the_kernel(d, k, t):
    torch.manual_seed(d)
    up = torch.randn(3, t, 2 * d, device=DEV).to(torch.bfloat16)
    layer = torch.nn.Conv1d(d, d, k, padding=k // 2, groups=d).to(DEV)
    norm = torch.nn.RMSNorm(d, eps=1e-5).to(DEV)
    lengths = torch.tensor([t, t // 2, 0], device=DEV)
    with torch.no_grad():
        y = depthwise_norm_silu(F.glu(up, -1), layer, lengths, norm)
        assert torch.equal(y, glu_norm_silu(up, layer, lengths, norm))
