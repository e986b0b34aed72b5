// Fused Mamba-3 SISO recurrence on gfx950 bf16 MFMA for N = 128, P = 64.
//
// Same arithmetic and bf16 rounding points as the reference kernel
// (src/trifusion_l4/mamba_fused.py:72-152), the phase summed in 2^-32 revolutions
// (increments rounded to nearest). A workgroup of four waves walks one
// (batch, head) unit, or one time segment of it, in 64-step chunks; up to 32 rotary
// pairs two workgroups share a CU (77 KB of LDS and at most 256 registers each), so
// one's vector work covers the other's latency (above that the cos/sin table takes
// 94 KB and one is alone). Per chunk, between three barriers:
//
//   rotation   16 rows per wave: [B/C norm,] bias, rotation, scale; values and
//              decay-scaled values; all to LDS as bf16 rows
//   products 1 y^T = S^T qr^T (all steps x the wave's 16 head dims), the ten
//              lower 16x16 score tiles shared out; one wave forms the next
//              chunk's controls
//   products 2 scores v, skip, gate, store; state update; the next chunk's
//              rotary phase and cos/sin table
//
// Wave w holds head dims 16 w .. 16 w + 15 of the fp32 state, all 128 channels,
// as eight 16x16 MFMA tiles. Its accumulator registers, packed to bf16, are the
// operand of the next chunk's S qr product: the state never passes through LDS.
//
// MFMA 16x16x32 layout (lane l, r = l & 15, g = l >> 4):
//   A[i][k]: lane i + 16 (k / 8), element k % 8; B[k][j]: lane j + 16 (k / 8)
//   D[i][j]: lane j + 16 (i / 4), element i % 4
// Contraction slots are permuted the same way on both sides: slot j of k-step s
// holds index 32 s + 16 (j / 4) + 4 g + j % 4, which is where a pair of D tiles
// holds its rows.
//
// What bounds it: vector instructions (about 2300 per wave and chunk, rotation and
// controls before all; the matrix cores are busy for a tenth of that) and, on short
// walks, the first chunk's loads and controls (a quarter of the time at 101 rows).
// Measured, bf16 projections, H = 32, one direction, the chunked kernel of
// mamba_mfma.hip against this one (us): 16 x 101 rows 38.6, 21.0; 8 x 201 41.4, 27.6;
// 4 x 401 90.8, 47.2; 1 x 1801 92.3, 49.9.
//
// Chunk-parallel form (few long units): summaries of every segment but the last
// (this kernel, MODE 1: from zero state and phase, only keys and values), a scan
// that turns each summary into the state entering the next segment, and the
// seeded walks. A summary is formed in its segment's own phase frame, and the scan
// turns it by the phase entering the segment (mamba_pipe.hip describes why that is
// the same state). Its keys therefore round to bf16 in that frame, not in the unit's
// as the serial walk's do: as exact, other bits (over 7200 steps 0.9e-4 of the norm
// from an oracle that rounds in the unit's frame, with a model's operands over 1300
// 1.4e-4, against 0.7e-4 and 0.6e-4 for the serial walk and 0.8e-4 to 3e-4 for the
// chunked kernel, whose fp32 increments carry the rounding of pi).
#include <algorithm>

#include "mamba_walk.h"

namespace tf {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
// 16 bytes of a row whose rows are 8-byte aligned
typedef u32x4 u32x4_a8 __attribute__((aligned(8)));

constexpr int kWideThreads = 256;
constexpr int kRecF4 = 2048;  // float4 per state record: [tile][thread]

__device__ __forceinline__ f32x4 mfma16(const u32x4& x, const u32x4& y, const f32x4& acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), acc, 0,
                                                 0, 0);
}

// Rows t0 .. t0 + 15 of a [64][64] row buffer as an operand of k-step s (columns 32 s ..).
__device__ __forceinline__ u32x4 row16(const uint16_t* buf, int t0, int s, int r, int g) {
  const u32x2 lo = rb_read(buf, t0 + r, 8 * s + g), hi = rb_read(buf, t0 + r, 8 * s + 4 + g);
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// Columns 4 u0 .. 4 u0 + 15 of a [64][64] row buffer as an operand of k-step s
// (rows 32 s ..): in each 16-lane group, source lane 4 k + c reads row k, unit c
// of a 4 x 4 block, and output lane j receives column j of the four rows.
template <bool BOTH>
__device__ __forceinline__ u32x4 col16(const uint16_t* buf, int u0, int s, int r, int g) {
  const int row = 32 * s + 4 * g + (r >> 2), u = u0 + (r & 3);
  const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(buf + rb_off(row, u))));
  if constexpr (!BOTH) return u32x4{lo[0], lo[1], 0u, 0u};
  const u32x2 hi =
      __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(buf + rb_off(row + 16, u))));
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// RT: rotary pairs the cos/sin table holds (R <= RT).
template <int RT>
struct WideSmem {
  static constexpr int TS = 2 * RT + 4;  // floats per table row: 16-byte pieces of 8 rows on distinct banks
  uint16_t qr[2][64 * 64];  // bf16(rot(q + qb)), channels 0-63 and 64-127
  uint16_t kr[2][64 * 64];  // bf16(rot(k + kb) * s)
  uint16_t v[64 * 64];      // v
  uint16_t vs[64 * 64];     // bf16(v * 2^(tot - cs))
  uint16_t sc[64 * 64];     // bf16 scores [t][u]
  float trig[64 * TS];      // [row][pair] (cos, sin)
  float qw[128], kw[128];   // fused B/C norm weights
  float qb[128], kb[128];   // biases
  // per-row controls of chunk c (c mod 2)
  float dt[2][64], scl[2][64], cs[2][64], wv[2][64], gam[2][64];
  float tot[2];
  float skip[64];  // (q + qb).(k + kb) of each row
};

// IN: how the controls, trapezoid and angles are read. 0: all fp32, 1: all bf16,
// both with the angles of eight neighbouring pairs in one aligned piece and byte
// offsets below 2^32; 2: any mix, element by element.
template <int IN>
__device__ __forceinline__ float load_in(const void* base, int bf16, uint32_t i) {
  if constexpr (IN == 0)
    return *reinterpret_cast<const float*>(static_cast<const char*>(base) + 4 * i);
  else if constexpr (IN == 1)
    return bf16_to_f32(*reinterpret_cast<const uint16_t*>(static_cast<const char*>(base) + 2 * i));
  else
    return bf16 ? to_f32(static_cast<const bf16_t*>(base)[i]) : static_cast<const float*>(base)[i];
}

// 16 bytes of a bf16 row: the byte offset stays 32-bit (a uniform base plus one register).
__device__ __forceinline__ u32x4 load_piece(const uint16_t* base, uint32_t i) {
  return *reinterpret_cast<const u32x4_a8*>(reinterpret_cast<const char*>(base) + 2 * i);
}

// Raw 16-byte pieces of one row: channels 8 ng .. and 64 + 8 ng .. of q and k,
// head dims 8 ng .. of v.
struct WideRow {
  u32x4 q[2], k[2], v;
};

// acc + the squares of a bf16 pair, summed in fp32 (v_dot2_f32_bf16: up to 1.4 units
// off where two fused multiply-adds are up to 1.0, and as many in root mean square).
// Rows of 128 summed this way, in 16 chains of four, are within 1.7e-7 of the exact
// sum, 0.4e-7 in root mean square; two chains of 64 multiply-adds 4.0e-7 and 0.7e-7.
__device__ __forceinline__ float square_sum(uint32_t x, float acc) {
  const bf16x2 v = __builtin_bit_cast(bf16x2, x);
  return __builtin_amdgcn_fdot2_f32_bf16(v, v, acc, false);
}

// Fused B/C RMSNorm (mamba.py:56-57, kernels/__init__.py:10-12) of a row of 128
// channels, 16 in each of 8 neighbouring lanes: x -> bf16(x rsqrt(mean + eps) w).
__device__ __forceinline__ void norm_row16(u32x4 (&x)[2], const float* w, int ng, float eps) {
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    s0 = square_sum(x[0][j], s0);
    s1 = square_sum(x[1][j], s1);
  }
  const float r = rsqrtf(group8_sum(s0 + s1) / 128.f + eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float4 a = *reinterpret_cast<const float4*>(w + 64 * i + 8 * ng);
    const float4 b = *reinterpret_cast<const float4*>(w + 64 * i + 8 * ng + 4);
    const float ww[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) x[i][j] = pack2(lo_f(x[i][j]) * r * ww[2 * j], hi_f(x[i][j]) * r * ww[2 * j + 1]);
  }
}

// MODE 0: outputs of the unit's (or, P.G > 1, the segment's) chunks. MODE 1: the
// segment's state from zero, its log2 decay and phase sums.
template <int RT, int IN, int MODE>
__global__ __launch_bounds__(kWideThreads, RT == 32 ? 2 : 1) void mamba_wide_kernel(const MfmaParams P) {
  using Sm = WideSmem<RT>;
  constexpr int TS = Sm::TS;
  constexpr int PI = RT / 32;  // phase pairs per lane
  __shared__ __align__(16) Sm sh;
  const PipeItem it = pipe_item(P);
  const int seg = it.seg, h = it.h, b = it.b;
  if (MODE == 1 && seg == P.G - 1) return;  // no walk starts from the last segment's state
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  // lane-derived indices, rebuilt every chunk from an index the compiler cannot
  // see through: hoisted out of the walk, the LDS addresses they feed would
  // hold a register each and spill
  int lane, r16, g, ng, row0;
  auto lane_indices = [&]() {
    lane = static_cast<int>(threadIdx.x & 63);
    asm volatile("" : "+v"(lane));
    r16 = lane & 15, g = lane >> 4;
    // rotation: rows 16 w + 8 i + row8 (i = 0, 1), eight lanes per row
    ng = lane & 7, row0 = 16 * w + row8_of_lane(lane);
  };
  lane_indices();
  const int T = P.T, R = P.R;
  int L = T;
  if (P.lengths != nullptr) {
    const int64_t l = P.lengths[b];
    L = l < 0 ? 0 : (l > T ? T : static_cast<int>(l));
  }
  const int nvalid = (L + kChunk - 1) / kChunk;
  const int c0 = min(seg_start(P, seg), nvalid);
  const int c1 = min(seg_start(P, seg + 1), nvalid);

  if (c1 > c0) {
    const int tlim = P.rev ? L : T;
    const int qh = h / P.group;
    // rows of the unit: step t is row t, or L - 1 - t reversed (the time strides
    // come negated then)
    const uint16_t* qbase = P.q + (b * P.q_sb + qh * P.q_sh);
    const uint16_t* kbase = P.k + (b * P.k_sb + qh * P.k_sh);
    const uint16_t* vbase = P.v + (b * P.v_sb + h * P.v_sh);
    const uint16_t* zbase = P.z + (b * P.z_sb + h * P.z_sh);
    auto in_base = [&](const void* p, bool bf16, int off) -> const void* {
      return static_cast<const char*>(p) + static_cast<int64_t>(off) * (IN == 1 || (IN == 2 && bf16) ? 2 : 4);
    };
    const bool ang16 = P.angles_dtype == TF_BFLOAT16;
    const void* dtp = in_base(P.dt, P.ctl_bf16, b * P.d_sb + h * P.d_sh);
    const void* adp = in_base(P.adt, P.ctl_bf16, b * P.a_sb + h * P.a_sh);
    const void* trp = in_base(P.trap, P.trap_bf16, b * P.r_sb + h * P.r_sh);
    const void* agp = in_base(P.angles, ang16, b * P.g_sb + h * P.g_sh);
    const uint32_t q_st = abs(P.q_st), k_st = abs(P.k_st), v_st = abs(P.v_st), z_st = abs(P.z_st);
    const uint32_t d_st = abs(P.d_st), a_st = abs(P.a_st), r_st = abs(P.r_st), g_st = abs(P.g_st);
    auto row_of = [&](int t) -> uint32_t { return P.rev ? L - 1 - t : t; };
    const int obase = b * P.o_sb + h * P.o_sh - (P.rev ? L - 1 : 0) * P.o_st;
    const float step_bias = P.ctl_raw ? P.dt_bias[h] : 0.f;
    const float skip_d = MODE == 0 ? P.d[h] : 0.f;
    auto load_rows = [&](int c, WideRow (&x)[2]) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t rr = row_of(min(c * kChunk + row0 + 8 * i, L - 1));
        x[i].k[0] = load_piece(kbase, rr * k_st + 8 * ng);
        x[i].k[1] = load_piece(kbase, rr * k_st + 8 * ng + 64);
        x[i].v = load_piece(vbase, rr * v_st + 8 * ng);
        if constexpr (MODE == 0) {
          x[i].q[0] = load_piece(qbase, rr * q_st + 8 * ng);
          x[i].q[1] = load_piece(qbase, rr * q_st + 8 * ng + 64);
        }
      }
    };
    // controls: wave 3, lane = row; rows clamped to ones that exist
    auto load_ctl = [&](int c) {
      const uint32_t rc = row_of(min(c * kChunk + lane, L - 1)), rn = row_of(min(c * kChunk + lane + 1, tlim - 1));
      PipeCtl x;
      x.dt = load_in<IN>(dtp, P.ctl_bf16, rc * d_st);
      x.dn = load_in<IN>(dtp, P.ctl_bf16, rn * d_st);
      x.adt = load_in<IN>(adp, P.ctl_bf16, rc * a_st);
      x.tr = load_in<IN>(trp, P.trap_bf16, rc * r_st);
      x.tn = load_in<IN>(trp, P.trap_bf16, rn * r_st);
      return x;
    };
    float seg_log2 = 0.f;
    auto controls = [&](const PipeCtl& raw, int c) {
      const int t = c * kChunk + lane, cb = c & 1;
      const RowControls rc = row_controls(P, raw, t < L, t + 1 < tlim, step_bias);
      sh.dt[cb][lane] = rc.dt;
      sh.scl[cb][lane] = rc.sc;
      sh.cs[cb][lane] = rc.cs;
      sh.wv[cb][lane] = rc.wv;
      sh.gam[cb][lane] = rc.gam;
      if (lane == 0) sh.tot[cb] = rc.tot;
    };
    // phase: lane = row, pairs 32 i + 8 w + j of wave w (raw angles: eight per row)
    typedef float Angles[PI][8];
    auto load_angles = [&](int c, Angles& th) {
      const uint32_t rr = row_of(min(c * kChunk + lane, L - 1));
#pragma unroll
      for (int i = 0; i < PI; ++i) {
        const int p0 = 32 * i + 8 * w;
        if (p0 < R) {  // wave-uniform
          if constexpr (IN == 0) {
            const char* p = static_cast<const char*>(agp) + 4 * (rr * g_st + p0);
            const float4 x = *reinterpret_cast<const float4*>(p), y = *reinterpret_cast<const float4*>(p + 16);
            th[i][0] = x.x, th[i][1] = x.y, th[i][2] = x.z, th[i][3] = x.w;
            th[i][4] = y.x, th[i][5] = y.y, th[i][6] = y.z, th[i][7] = y.w;
          } else if constexpr (IN == 1) {
            // kept packed until used: four registers
            const u32x4 x = *reinterpret_cast<const u32x4*>(static_cast<const char*>(agp) + 2 * (rr * g_st + p0));
#pragma unroll
            for (int j = 0; j < 4; ++j) th[i][j] = __uint_as_float(x[j]);
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              th[i][j] = load_in<IN>(agp, ang16, rr * g_st + (p0 + j < R ? p0 + j : 0) * P.g_sr);
          }
        }
      }
    };
    uint32_t carry[PI][8];  // phase entering the chunk, 2^-32 revolutions (wave-uniform)
#pragma unroll
    for (int i = 0; i < PI; ++i) {
      uint32_t incl = 0;
      if (MODE == 0 && seg > 0) {
        // the wrapping sum of the preceding segments' phase sums: lane = (pair, eighth)
        const int pair = 32 * i + 8 * w + (lane >> 3);
        uint32_t part = 0;
        if (pair < R)
          for (int s = lane & 7; s < seg; s += 8) part += P.phase_fx[(static_cast<size_t>(it.unit) * P.G + s) * RT + pair];
        incl = group_scan_dpp<8>(part, lane);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        carry[i][j] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), 8 * j + 7));
    }
    auto phase = [&](const Angles& th, int c) {
      const float dt = sh.dt[c & 1][lane];
#pragma unroll
      for (int i = 0; i < PI; ++i) {
        const int p0 = 32 * i + 8 * w;
        if (p0 < R) {
          float* tg = &sh.trig[lane * TS + 2 * p0];
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            float2 x[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              float a;
              if constexpr (IN == 1)
                a = k == 0 ? lo_f(__float_as_uint(th[i][j / 2])) : hi_f(__float_as_uint(th[i][j / 2]));
              else
                a = th[i][j + k];
              const uint32_t incl = wave_scan_u32(phase_inc<true>(a, dt));
              x[k] = phase_trig(carry[i][j + k] + incl);
              // an angle that is not a number makes its row (and with it every
              // later one) not a number; fixed point alone would lose it
              x[k].x = a == a ? x[k].x : a;
              carry[i][j + k] += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
              // pairs that do not rotate turn by the identity
              if (IN == 2 && p0 + j + k >= R) x[k] = make_float2(1.f, 0.f);
            }
            *reinterpret_cast<float4*>(tg + 2 * j) = make_float4(x[0].x, x[0].y, x[1].x, x[1].y);
          }
        }
      }
    };
    // norm, bias, rotation, scale and rounding of the lane's row pieces
    // (mamba_fused.py:112-135, 151; mamba.py:56-57)
    auto rotate = [&](WideRow (&x)[2], int c) {
      const int cb = c & 1;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = row0 + 8 * i;
        // a row past the length repeats the last one with a key scale of 0
        const float scl = sh.scl[cb][row], wvt = sh.wv[cb][row];
        if (P.qk_norm) {
          norm_row16(x[i].k, sh.kw, ng, P.norm_eps);
          if constexpr (MODE == 0) norm_row16(x[i].q, sh.qw, ng, P.norm_eps);
        }
        float part = 0.f;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          u32x4 qo, ko;
          float kbv[8], qbv[8];
#pragma unroll
          for (int j = 0; j < 8; j += 4) {
            const float4 kb4 = *reinterpret_cast<const float4*>(&sh.kb[64 * p + 8 * ng + j]);
            kbv[j] = kb4.x, kbv[j + 1] = kb4.y, kbv[j + 2] = kb4.z, kbv[j + 3] = kb4.w;
            if constexpr (MODE == 0) {
              const float4 qb4 = *reinterpret_cast<const float4*>(&sh.qb[64 * p + 8 * ng + j]);
              qbv[j] = qb4.x, qbv[j + 1] = qb4.y, qbv[j + 2] = qb4.z, qbv[j + 3] = qb4.w;
            }
          }
          if (32 * p < R) {  // wave-uniform: the piece holds rotary pairs
            const float2* tg = reinterpret_cast<const float2*>(&sh.trig[row * TS + 64 * p + 8 * ng]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float2 cs = tg[j];
              const float cv = cs.x, sv = cs.y;  // the identity for pairs >= R
              const float k0 = lo_f(x[i].k[p][j]) + kbv[2 * j], k1 = hi_f(x[i].k[p][j]) + kbv[2 * j + 1];
              ko[j] = key_pair(k0, k1, cv, sv, scl);
              if constexpr (MODE == 0) {
                const float q0 = lo_f(x[i].q[p][j]) + qbv[2 * j], q1 = hi_f(x[i].q[p][j]) + qbv[2 * j + 1];
                part += q0 * k0 + q1 * k1;
                qo[j] = pack2(q0 * cv - q1 * sv, q0 * sv + q1 * cv);
              }
            }
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float k0 = lo_f(x[i].k[p][j]) + kbv[2 * j], k1 = hi_f(x[i].k[p][j]) + kbv[2 * j + 1];
              ko[j] = pack2(k0 * scl, k1 * scl);
              if constexpr (MODE == 0) {
                const float q0 = lo_f(x[i].q[p][j]) + qbv[2 * j], q1 = hi_f(x[i].q[p][j]) + qbv[2 * j + 1];
                part += q0 * k0 + q1 * k1;
                qo[j] = pack2(q0, q1);
              }
            }
          }
          rb_write16(sh.kr[p], row, 2 * ng, ko);
          if constexpr (MODE == 0) rb_write16(sh.qr[p], row, 2 * ng, qo);
        }
        u32x4 vo, vso;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          vo[j] = x[i].v[j];
          vso[j] = scaled_pair(vo[j], wvt);
        }
        rb_write16(sh.vs, row, 2 * ng, vso);
        if constexpr (MODE == 0) {
          rb_write16(sh.v, row, 2 * ng, vo);
          part = group8_sum(part);
          if (ng == 0) sh.skip[row] = part;
        }
      }
    };

    // the start's loads, then chunk c0's controls and phase
    WideRow rows[2];
    PipeCtl ctl = {};
    Angles th;
    if (w == 3) ctl = load_ctl(c0);
    load_angles(c0, th);
    load_rows(c0, rows);
    f32x4 S[8];  // state tiles [2 s + a]: channels 32 s + 16 a + 4 g + e, head dim 16 w + r16
#pragma unroll
    for (int j = 0; j < 8; ++j) S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (MODE == 0 && seg > 0) {
      const float4* rec = P.seg_state + (static_cast<size_t>(it.unit) * (P.G - 1) + seg - 1) * kRecF4 + threadIdx.x;
#pragma unroll
      for (int j = 0; j < 8; ++j) S[j] = __builtin_bit_cast(f32x4, rec[j * kWideThreads]);
    }
    // pairs that no wave forms, up to the end of the last rotating piece
    for (int e = 64 * ((R + 7) & ~7) + static_cast<int>(threadIdx.x); e < 64 * ((R + 31) & ~31); e += kWideThreads)
      *reinterpret_cast<float2*>(&sh.trig[(e & 63) * TS + 2 * (e >> 6)]) = make_float2(1.f, 0.f);
    if (threadIdx.x < 128) {
      sh.kb[threadIdx.x] = P.kb[h * 128 + threadIdx.x];
      if (MODE == 0) sh.qb[threadIdx.x] = P.qb[h * 128 + threadIdx.x];
      if (P.qk_norm) {
        sh.kw[threadIdx.x] = P.kn_w[threadIdx.x];
        if (MODE == 0) sh.qw[threadIdx.x] = P.qn_w[threadIdx.x];
      }
    }
    if (w == 3) controls(ctl, c0);
    lds_barrier();
    phase(th, c0);
    if (c0 + 1 < c1) {
      if (w == 3) ctl = load_ctl(c0 + 1);
      load_angles(c0 + 1, th);
    }
    lds_barrier();

    for (int c = c0; c < c1; ++c) {
      lane_indices();
      const int cb = c & 1;
      const int nrows = L - c * kChunk;  // valid rows of the chunk (may exceed 64)
      const bool more = c + 1 < c1;
      // a wave whose rows all lie past the length has none to rotate
      if (16 * w < nrows) rotate(rows, c);
      u32x2 zr[4];
      if constexpr (MODE == 0) {
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          const uint32_t rr = row_of(min(c * kChunk + 16 * tt + r16, L - 1));
          zr[tt] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const char*>(zbase) +
                                                   2 * (rr * z_st + 16 * w + 4 * g));
        }
      }
      if (more) load_rows(c + 1, rows);
      lds_barrier();

      f32x4 y[4];
      if constexpr (MODE == 0) {
        u32x4 sp[4], kop[4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
          sp[s] = u32x4{pack2(S[2 * s][0], S[2 * s][1]), pack2(S[2 * s][2], S[2 * s][3]),
                        pack2(S[2 * s + 1][0], S[2 * s + 1][1]), pack2(S[2 * s + 1][2], S[2 * s + 1][3])};
        if (w < 3 && 16 * w < nrows) {
#pragma unroll
          for (int s = 0; s < 4; ++s) kop[s] = row16(sh.kr[s >> 1], 16 * w, s & 1, r16, g);
        }
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          y[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (16 * tt < nrows) {
            u32x4 qop[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) qop[s] = row16(sh.qr[s >> 1], 16 * tt, s & 1, r16, g);
#pragma unroll
            for (int s = 0; s < 4; ++s) y[tt] = mfma16(sp[s], qop[s], y[tt]);
            // scores^T tile (u, tt): kr_u . qr_t times 2^min(cs_t - cs_u, 0), strictly
            // causal (mamba_fused.py:144-146). Tiles u = w, wave 2 also (3, 3):
            // wave 3 forms the next chunk's controls meanwhile.
            auto score = [&](const u32x4 (&ko)[4], int u) {
              f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int s = 0; s < 4; ++s) a = mfma16(ko[s], qop[s], a);
              const float cst = sh.cs[cb][16 * tt + r16];
              const float4 cu = *reinterpret_cast<const float4*>(&sh.cs[cb][16 * u + 4 * g]);
              const float csu[4] = {cu.x, cu.y, cu.z, cu.w};
              float x[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                // masked elements may overflow here; the select drops them
                const float v = a[e] * fast_exp2(fminf(cst - csu[e], 0.f));
                x[e] = (u < tt || r16 > 4 * g + e) ? v : 0.f;
              }
              *reinterpret_cast<u32x2*>(sh.sc + rb_off(16 * tt + r16, 4 * u + g)) =
                  u32x2{pack2(x[0], x[1]), pack2(x[2], x[3])};
            };
            if (w < 3 && w <= tt) score(kop, w);
            if (w == 2 && tt == 3) {
              u32x4 k3[4];
#pragma unroll
              for (int s = 0; s < 4; ++s) k3[s] = row16(sh.kr[s >> 1], 48, s & 1, r16, g);
              score(k3, 3);
            }
          }
        }
      }
      if (more && w == 3) controls(ctl, c + 1);
      lds_barrier();

      if constexpr (MODE == 0) {
        u32x4 va[2];
        va[0] = col16<true>(sh.v, 4 * w, 0, r16, g);
        va[1] = col16<true>(sh.v, 4 * w, 1, r16, g);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          if (16 * tt < nrows) {
            const int row = 16 * tt + r16;
            const float decay = fast_exp2(sh.cs[cb][row]);
            const float coef = skip_d + sh.gam[cb][row] * sh.skip[row];
            const u32x2 vv = rb_read(sh.v, row, 4 * w + g);
            const float vf[4] = {lo_f(vv[0]), hi_f(vv[0]), lo_f(vv[1]), hi_f(vv[1])};
            f32x4 a;
            // (D + gamma (q + qb).(k + kb)) v + 2^cs qr . bf16(S)^T (mamba_fused.py:124, 143, 147)
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = coef * vf[e] + y[tt][e] * decay;
            // scores . v: steps u of the score tiles (0 .. tt, tt) alone; the slots
            // past them are 0 on both sides
#pragma unroll
            for (int s = 0; s <= tt / 2; ++s) {
              if (2 * s + 1 <= tt) {
                a = mfma16(va[s], row16(sh.sc, 16 * tt, s, r16, g), a);
              } else {
                const u32x2 lo = rb_read(sh.sc, row, 8 * s + g);
                a = mfma16(u32x4{va[s][0], va[s][1], 0u, 0u}, u32x4{lo[0], lo[1], 0u, 0u}, a);
              }
            }
            const int t = c * kChunk + row;
            const float zf[4] = {lo_f(zr[tt][0]), hi_f(zr[tt][0]), lo_f(zr[tt][1]), hi_f(zr[tt][1])};
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] *= zf[e] * sigmoid_fast(zf[e]);
            if (t < L) {
              const int off = obase + t * P.o_st + 16 * w + 4 * g;
              if (P.out_f32)
                *reinterpret_cast<float4*>(static_cast<float*>(P.out) + off) = make_float4(a[0], a[1], a[2], a[3]);
              else
                *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(P.out) + off) =
                    u32x2{pack2(a[0], a[1]), pack2(a[2], a[3])};
            }
          }
        }
      }
      // S <- S 2^tot + kr^T . vs (mamba_fused.py:150-152); nothing follows the
      // last valid chunk
      if (c + 1 < nvalid) {
        const float tot = sh.tot[cb];
        const float dec = fast_exp2(tot);
        seg_log2 += tot;
        const u32x4 vb0 = col16<true>(sh.vs, 4 * w, 0, r16, g), vb1 = col16<true>(sh.vs, 4 * w, 1, r16, g);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint16_t* buf = sh.kr[j >> 2];
          const int u0 = 4 * (j & 3);
          f32x4 a = S[j];
#pragma unroll
          for (int e = 0; e < 4; ++e) a[e] *= dec;
          a = mfma16(col16<true>(buf, u0, 0, r16, g), vb0, a);
          S[j] = mfma16(col16<true>(buf, u0, 1, r16, g), vb1, a);
        }
      }
      if (more) {
        phase(th, c + 1);
        if (c + 2 < c1) {
          if (w == 3) ctl = load_ctl(c + 2);
          load_angles(c + 2, th);
        }
      }
      lds_barrier();
    }
    if constexpr (MODE == 1) {
      float4* rec = P.seg_state + (static_cast<size_t>(it.unit) * (P.G - 1) + seg) * kRecF4 + threadIdx.x;
#pragma unroll
      for (int j = 0; j < 8; ++j) rec[j * kWideThreads] = __builtin_bit_cast(float4, S[j]);
      if (threadIdx.x == 0) P.seg_decay[it.rec] = seg_log2;
#pragma unroll
      for (int i = 0; i < PI; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (lane == j) P.phase_fx[static_cast<size_t>(it.rec) * RT + 32 * i + 8 * w + j] = carry[i][j];
    }
  }
  if constexpr (MODE == 0) {
    // the segment's rows in [L, T): the same rows in either direction
    const int o_st = P.rev ? -P.o_st : P.o_st;
    const int obase = b * P.o_sb + h * P.o_sh;
    const int row_end = min(seg_start(P, seg + 1) * kChunk, T);
    for (int e = max(seg_start(P, seg) * kChunk, L) * 16 + static_cast<int>(threadIdx.x); e < row_end * 16;
         e += kWideThreads) {
      const int off = obase + (e >> 4) * o_st + 4 * (e & 15);
      if (P.out_f32)
        *reinterpret_cast<float4*>(static_cast<float*>(P.out) + off) = make_float4(0.f, 0.f, 0.f, 0.f);
      else
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(P.out) + off) = u32x2{0u, 0u};
    }
  }
}

// Replaces each unit's summaries by the states entering the next segments:
// S_1 = d_0, S_{g+1} = S_g 2^dec_g + turn_g(d_g), where turn_g rotates the rotary
// row pairs by the phase entering segment g. Workgroup (unit, slice of 64 float4).
template <int RT>
__global__ __launch_bounds__(64) void wide_scan_kernel(const MfmaParams P) {
  constexpr int kSlices = kRecF4 / 64;
  constexpr int kBatch = 8;
  const int unit = blockIdx.x / kSlices;
  const int f = (blockIdx.x - unit * kSlices) * 64 + threadIdx.x;
  const int G = P.G, R = P.R;
  // float4 f: tile f / 256, lane f % 64: channels 16 tile + 4 g + e, rotary pairs rp, rp + 1
  const int rp = 8 * (f >> 8) + 2 * ((f & 63) >> 4);
  float4* st = P.seg_state + static_cast<size_t>(unit) * (G - 1) * kRecF4 + f;
  const float* dec = P.seg_decay + static_cast<size_t>(unit) * G;
  const uint32_t* phs = P.phase_fx + static_cast<size_t>(unit) * G * RT + (rp < RT ? rp : 0);
  const bool turn = rp < R;
  float4 run = make_float4(0.f, 0.f, 0.f, 0.f);
  uint2 ph = make_uint2(0u, 0u);
  for (int g0 = 0; g0 < G - 1; g0 += kBatch) {
    float4 d[kBatch];
    Factor m[kBatch];
    uint2 s[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (g0 + j < G - 1) {
        d[j] = st[static_cast<size_t>(g0 + j) * kRecF4];
        m[j] = factor_of(dec[g0 + j]);
        if (turn) s[j] = *reinterpret_cast<const uint2*>(phs + (g0 + j) * RT);
      }
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (g0 + j < G - 1) {
        if (turn) {
          if (g0 + j > 0) d[j] = turn_rows(d[j], ph, rp, R);
          ph = make_uint2(ph.x + s[j].x, ph.y + s[j].y);
        }
        const int e = m[j].exp;
        run = make_float4(ldexpf(run.x, e), ldexpf(run.y, e), ldexpf(run.z, e), ldexpf(run.w, e));
        run = state_step(run, m[j].mant, d[j]);
        st[static_cast<size_t>(g0 + j) * kRecF4] = run;
      }
    }
  }
}

// Chunk-parallel plan. At most kGroups workgroups (two on each of the 256 CUs, all
// resident) and records that fit the library's static scratch (kMaxRecords of
// 32 KB, and the phases, in 16 MiB); segments as short as that allows, but of two
// chunks. The summaries, the scan and their launches pay from six chunks on, from
// eight above 96 units, and up to 170 units, which leave three segments each (us,
// split against serial): 32 units, 6 chunks 30.6 / 40.9, 29 51.4 / 194;
// 64 units, 4 chunks 29.7 / 26.8, 5 40.3 / 34.4, 6 32.2 / 40.8, 29 70.8 / 193; 128
// units, 7 chunks 46.3 / 47.0, 8 45.8 / 55.6; 160 units, 7 chunks 51.4 / 48.3, 13
// 74.3 / 89.6; 192 units in two segments, 13 chunks 96.5 / 89.6.
// With more than 32 rotary pairs one workgroup fits a CU. One round of them, 256, is
// the better plan up to 64 units (R 64, 32 units, 29 chunks 63 us against 73 in two
// rounds); above, too few segments are left and two rounds are (96 units, 29 chunks
// 162 against 209 serial), up to 128 units (160 units, 13 chunks 124 against 97 serial).
constexpr int64_t kGroups = 512, kMaxRecords = 480, kSegment = 2, kMaxUnits = 170, kMaxUnits64 = 128;

struct WidePlan {
  int G = 1;
  int64_t phase_off = 0, decay_off = 0, bytes = 0;
};

int table_pairs(const tf_mamba_args& a) { return a.rotary <= 32 ? 32 : 64; }

WidePlan wide_plan(const tf_mamba_args& a) {
  WidePlan p;
  const int64_t units = a.batch * a.heads;
  const int64_t chunks = (a.time + kChunk - 1) / kChunk;
  const bool table64 = a.rotary > 32;
  if (units <= 0 || units > (table64 ? kMaxUnits64 : kMaxUnits) || chunks < (units <= 96 ? 6 : 8)) return p;
  const int64_t groups = table64 && units <= 64 ? kGroups / 2 : kGroups;
  const int64_t g = std::min({groups / units, kMaxRecords / units + 1, (chunks + kSegment - 1) / kSegment});
  p.G = static_cast<int>(g);
  auto up = [](int64_t x) { return (x + 255) & ~int64_t(255); };
  p.phase_off = up(units * (g - 1) * kRecF4 * 16);
  p.decay_off = p.phase_off + up(units * g * table_pairs(a) * 4);
  p.bytes = p.decay_off + up(units * g * 4);
  return p;
}

template <int RT, int IN>
int launch_wide_kernel(const MfmaParams& P, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>(P.units) * P.G), block(kWideThreads);
  if (P.G > 1) {
    hipLaunchKernelGGL((mamba_wide_kernel<RT, IN, 1>), grid, block, 0, stream, P);
    if (const int rc = launch_status()) return rc;
    hipLaunchKernelGGL((wide_scan_kernel<RT>), dim3(static_cast<uint32_t>(P.units) * (kRecF4 / 64)), dim3(64), 0,
                       stream, P);
    if (const int rc = launch_status()) return rc;
  }
  hipLaunchKernelGGL((mamba_wide_kernel<RT, IN, 0>), grid, block, 0, stream, P);
  return launch_status();
}

}  // namespace

int64_t wide_workspace_bytes(const tf_mamba_args& a) {
  const WidePlan plan = wide_plan(a);
  return plan.G > 1 ? plan.bytes : 0;
}

int launch_wide(const tf_mamba_args& a, hipStream_t stream) {
  MfmaParams P = make_params(a);
  const WidePlan plan = wide_plan(a);
  if (plan.G > 1 && a.workspace != nullptr && aligned(a.workspace, 256) && a.workspace_bytes >= plan.bytes) {
    char* ws = static_cast<char*>(a.workspace);
    P.G = plan.G;
    P.seg_state = reinterpret_cast<float4*>(ws);
    P.phase_fx = reinterpret_cast<uint32_t*>(ws + plan.phase_off);
    P.seg_decay = reinterpret_cast<float*>(ws + plan.decay_off);
  }
  const int64_t items = static_cast<int64_t>(P.units) * P.G;
  P.xcd_per = (items % 8 == 0 && items >= 64) ? static_cast<int>(items / 8) : 0;
  const bool ang16 = P.angles_dtype == TF_BFLOAT16;
  // angles in aligned pieces of eight pairs, every byte offset of the 32-bit
  // operands below 2^32
  bool pieces = a.rotary % 8 == 0 && P.g_sr == 1 && aligned(a.angles, 16);
  for (int i = 0; i < 3; ++i) pieces = pieces && a.angles_stride[i] % 8 == 0;
  const int64_t span = std::max({a.time * a.angles_stride[1], a.time * a.dt_stride[2], a.time * a.adt_stride[2],
                                 a.time * a.trap_stride[2]});
  pieces = pieces && span < (int64_t(1) << 29);
  const bool all32 = pieces && !P.ctl_bf16 && !P.trap_bf16 && !ang16;
  const bool all16 = pieces && P.ctl_bf16 && P.trap_bf16 && ang16;
  if (a.rotary > 32) {
    if (all32) return launch_wide_kernel<64, 0>(P, stream);
    return all16 ? launch_wide_kernel<64, 1>(P, stream) : launch_wide_kernel<64, 2>(P, stream);
  }
  if (all32) return launch_wide_kernel<32, 0>(P, stream);
  return all16 ? launch_wide_kernel<32, 1>(P, stream) : launch_wide_kernel<32, 2>(P, stream);
}

}  // namespace tf
