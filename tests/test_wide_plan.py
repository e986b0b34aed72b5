"""The N = 128, P = 64 recurrence's chunk-parallel plan, as the workspace query tells
it (no GPU: nothing is read or launched)."""

import ctypes

import pytest

from trifusion_amd import _lib

BF16, FP32 = 1, 0


def workspace(batch, heads, time, rotary):
    a = _lib.MambaArgs()
    h, n, p = heads, 128, 64
    shapes = {"q": (time * n, n, n, 1), "k": (time * n, n, n, 1), "v": (time * h * p, h * p, p, 1),
              "z": (time * h * p, h * p, p, 1), "angles": (time * h * rotary, h * rotary, rotary, 1),
              "out": (time * h * p, h * p, p, 1), "adt": (h * time, time, 1), "dt": (h * time, time, 1),
              "trap": (h * time, time, 1)}
    for name, strides in shapes.items():
        setattr(a, name, 1 << 20)
        setattr(a, name + "_dtype", FP32 if name in ("angles", "adt", "dt", "trap") else BF16)
        getattr(a, name + "_stride")[:] = strides
    a.qb = a.kb = a.d = 1 << 20
    a.batch, a.time, a.heads, a.qk_heads, a.state, a.head_dim, a.rotary = batch, time, heads, 1, n, p, rotary
    assert _lib.load().tf_fused_mamba_variant(ctypes.byref(a)) == _lib.VARIANTS["mfma"]
    return _lib.load().tf_fused_mamba_workspace_size(ctypes.byref(a))


def expected(units, segments, pairs):
    def up(x):
        return (x + 255) & ~255

    if segments == 1:
        return 0
    return up(units * (segments - 1) * 32768) + up(units * segments * pairs * 4) + up(units * segments * 4)


# up to 32 rotary pairs two workgroups share a CU, above that one is alone
@pytest.mark.parametrize("units,time,rotary,segments", [
    (32, 1801, 32, 15), (32, 1801, 64, 8), (32, 320, 32, 1), (32, 321, 32, 3), (64, 513, 33, 4), (65, 3600, 64, 7),
    (96, 1801, 64, 5), (128, 1801, 64, 4), (129, 1801, 64, 1), (160, 801, 64, 1), (160, 801, 32, 3), (171, 801, 32, 1)])
def test_segments(units, time, rotary, segments):
    assert workspace(1, units, time, rotary) == expected(units, segments, 32 if rotary <= 32 else 64)


def test_records_fit_the_static_scratch():
    limit = _lib.load().tf_fused_mamba_static_scratch_bytes()
    for rotary in (32, 64):
        for units in range(1, 200):
            assert workspace(1, units, 100000, rotary) <= limit
