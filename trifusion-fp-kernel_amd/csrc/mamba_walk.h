// Pieces shared by the walks that keep the state in registers (mamba_pipe.hip,
// mamba_wide.hip) and their chunk-parallel summaries: work items and segments,
// controls, the fixed-point rotary phase, and the roundings of a key and a
// scaled value. One definition each, so that every kernel forms the same bits.
#pragma once

#include "mfma_tile.h"

namespace tf {
namespace {

// Row (0..7) of an eight-row block held by lanes 8 j .. 8 j + 7: j / 2 + 4 (j % 2),
// so the two rows of each 16 lanes are four apart (conflict-free row writes).
__device__ __forceinline__ int row8_of_lane(int lane) { return (lane >> 4) + 4 * ((lane >> 3) & 1); }

struct PipeCtl {
  float dt, dn, adt, tr, tn;
};

template <bool BF16>
__device__ __forceinline__ float load_elem(const void* base, int i) {
  if constexpr (BF16)
    return bf16_to_f32(static_cast<const uint16_t*>(base)[i]);
  else
    return static_cast<const float*>(base)[i];
}

// Controls of row t and its halo step t + 1 (raw values when P.ctl_raw). Rows
// are clamped to ones that exist and masked where used, so no load sits behind
// a branch and the loads stay in flight until then.
template <bool CTL16, bool TRAP16>
__device__ __forceinline__ PipeCtl load_pipe_ctl(const MfmaParams& P, int dto, int ado, int trb, int t, int L,
                                                 int tlim) {
  const int tc = min(t, L - 1);
  const int tn = min(t + 1, tlim - 1);
  PipeCtl c;
  c.dt = load_elem<CTL16>(P.dt, dto + tc * P.d_st);
  c.dn = load_elem<CTL16>(P.dt, dto + tn * P.d_st);
  c.adt = load_elem<CTL16>(P.adt, ado + tc * P.a_st);
  c.tr = load_elem<TRAP16>(P.trap, trb + tc * P.r_st);
  c.tn = load_elem<TRAP16>(P.trap, trb + tn * P.r_st);
  return c;
}

// First chunk of segment g of a unit's time axis: the ceil(T / 64) chunks
// split as evenly as G segments allow, the first (chunks mod G) segments one
// chunk longer. A later segment's walk first scans the summaries of every
// segment before it, so the segments that scan the most walk the fewest chunks.
__device__ __forceinline__ int seg_start(const MfmaParams& P, int g) {
  const int chunks = (P.T + kChunk - 1) / kChunk;
  const int base = chunks / P.G, extra = chunks % P.G;
  return g * base + min(g, extra);
}

// Work item of workgroup blockIdx.x: (batch row, segment, head). The heads of
// one batch row and segment read the same q/k rows, so they are consecutive
// items, and items are dealt to the 8 XCDs in contiguous ranges so that those
// heads share an L2. A segment's state record is [unit][segment].
struct PipeItem {
  int b, h, seg, unit, rec;
};

__device__ __forceinline__ PipeItem pipe_item(const MfmaParams& P) {
  const int item = P.xcd_per > 0 ? (blockIdx.x & 7) * P.xcd_per + (blockIdx.x >> 3) : static_cast<int>(blockIdx.x);
  const int bseg = item / P.H;
  PipeItem it;
  it.h = item - bseg * P.H;
  it.b = bseg / P.G;
  it.seg = bseg - it.b * P.G;
  it.unit = it.b * P.H + it.h;
  it.rec = it.unit * P.G + it.seg;
  return it;
}

// Fixed-point phase increment of one (row, pair): pi tanh(theta) dt radians
// (mamba_fused.py:102-109) = tanh(theta) dt / 2 revolutions, reduced to
// [-1/2, 1/2] and scaled by 2^32. A row without a step (dt = 0) adds 0. NEAREST
// rounds it to the nearest unit, else towards 0: of increments of one sign that
// loses half a unit per step, 5e-6 rad over 7200 steps.
template <bool NEAREST = false>
__device__ __forceinline__ uint32_t phase_inc(float th, float dt) {
  float om = tanh_fast(th) * dt * 0.5f;
  om -= rintf(om);
  float x = fminf(om * 4294967296.f, 2147483520.f);
  if constexpr (NEAREST) x = rintf(x);
  return static_cast<uint32_t>(static_cast<int>(x));
}

// (cos, sin) of a fixed-point phase (2^-32 revolutions): v_cos/v_sin take revolutions.
__device__ __forceinline__ float2 phase_trig(uint32_t ph) {
  const float rev = static_cast<float>(static_cast<int>(ph)) * 2.3283064365386963e-10f;
  return make_float2(__builtin_amdgcn_cosf(rev), __builtin_amdgcn_sinf(rev));
}

// Rows (2 rp, 2 rp + 1) and (2 rp + 2, 2 rp + 3) of a state record, the rotary
// pairs rp and rp + 1, turned by phases ph (the key rotation of key_pair,
// applied to the rows kr contributes to); pairs >= R are left as they are.
__device__ __forceinline__ float4 turn_rows(const float4& d, uint2 ph, int rp, int R) {
  float4 o = d;
  if (rp < R) {
    const float2 a = phase_trig(ph.x);
    o.x = __builtin_fmaf(d.x, a.x, -(d.y * a.y));
    o.y = __builtin_fmaf(d.x, a.y, d.y * a.x);
  }
  if (rp + 1 < R) {
    const float2 a = phase_trig(ph.y);
    o.z = __builtin_fmaf(d.z, a.x, -(d.w * a.y));
    o.w = __builtin_fmaf(d.z, a.y, d.w * a.x);
  }
  return o;
}

// Controls of one chunk, one wave, lane = row (mamba_fused.py:96-101, 139-142):
// step, key scale, inclusive log2 decay, 2^(tot - cs), dt sigmoid(trap), and
// the chunk's total log2 decay (every lane).
struct RowControls {
  float dt, sc, cs, wv, gam, tot;
};

__device__ __forceinline__ RowControls row_controls(const MfmaParams& P, const PipeCtl& raw, bool valid, bool next,
                                                    float step_bias) {
  float dtv = raw.dt, dnv = raw.dn, adv = raw.adt;
  if (P.ctl_raw) {
    // step and decay from the raw columns (primitives.py:209-214)
    dtv = control_step(dtv, step_bias);
    dnv = control_step(dnv, step_bias);
    adv = control_decay(adv, dtv, P.a_floor);
  }
  // rows without a step keep dt = adt = 0, and a missing halo step loads 0
  dtv = valid ? dtv : 0.f;
  adv = valid ? adv : 0.f;
  dnv = next ? dnv : 0.f;
  const float trv = valid ? raw.tr : 0.f;
  const float tnv = next ? raw.tn : 0.f;
  RowControls r;
  r.dt = dtv;
  r.gam = dtv * sigmoid_fast(trv);
  r.sc = __builtin_fmaf(dnv, 1.f - sigmoid_fast(tnv), r.gam);
  r.cs = wave_scan_dpp(adv * kLog2e);
  r.tot = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, r.cs), 63));
  r.wv = fast_exp2(r.tot - r.cs);
  return r;
}

// bf16 pair of a key rotated by (cv, sv) and scaled by the trapezoid scale
// (mamba_fused.py:126-131), and of a value scaled by 2^(tot - cs) (:151).
// The fused multiply-adds are spelled out, so that every kernel rounds a key
// the same way whatever the compiler would contract in its context.
__device__ __forceinline__ uint32_t key_pair(float k0, float k1, float cv, float sv, float scl) {
  return pack2(__builtin_fmaf(k0, cv, -(k1 * sv)) * scl, __builtin_fmaf(k0, sv, k1 * cv) * scl);
}
__device__ __forceinline__ uint32_t scaled_pair(uint32_t vw, float wvt) {
  return pack2(lo_f(vw) * wvt, hi_f(vw) * wvt);
}

}  // namespace
}  // namespace tf
