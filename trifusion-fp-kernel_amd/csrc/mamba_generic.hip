// Generic fused Mamba-3 SISO recurrence: 32-bit arithmetic on fp32 MFMA, any
// operand dtype (fp32/bf16/fp16) and strides, N <= 128 (even), P <= 64, R <= N/2.
//
// One workgroup of eight waves per (head, batch) walks the sequence in 64-step
// chunks, the way the reference kernel does (src/trifusion_l4/mamba_fused.py:72-152),
// and rounds intermediate values to the operand dtypes at the same points:
// qr -> q dtype, kr -> k dtype (:127-132), the state copy used by qr.S^T -> q
// dtype (:143), the decayed score -> v dtype (:146) and the decay-scaled v ->
// k dtype (:151-152). It is the kernel for shapes and dtypes the bf16 MFMA paths
// do not take (fp32 operands, odd sizes) and an independent second implementation
// those kernels are tested against. Raw controls and the reversed walk follow
// their definitions (computed per step; row L-1-t for step t).
//
// Per chunk:
//   controls     wave 0, lane = row
//   phase        lane = row, a wave per R/8 pairs: fp64 increments and scan
//   rotation     8 lanes per row, each 4 channels of every 32
//   products 1   waves 0-3: qr S of one 32x32 tile of y each; waves 4-6: one
//                32x32 tile of the scores each
//   products 2   waves 0-3: scores v, gate, store; waves 4-7: state tiles
// Contractions run on v_mfma_f32_32x32x2_f32: products and sums of full 32-bit
// operands. N is padded to 32, 64 or 128 and P to 32 or 64 with zeros in LDS.
//
// What bounds it: the chain of one chunk, ~11 us at N = P = 64 of which the
// products take ~4 (a SIMD's two waves share a 32-bit matrix unit), the rest
// being the latency of controls, phase and rotation between barriers. So few long
// fp32 units run chunk-parallel: segment summaries (MODE 1: keys and values only),
// a scan of their states, and walks of the segments. B4 L400 H16 P64 N64, fp32:
// 80 us in one segment per unit, 63 us in three (2,155 us with contractions formed
// element by element from LDS and one thread per phase pair); B1 L1600 H16 N128:
// 446 and 104 us (13.2 ms). 32-bit offsets take the clip from 108 to 80 us against
// 64-bit ones (fewer scalar registers spilled), so they are used wherever they fit.
#include <algorithm>
#include <type_traits>

#include "mfma_tile.h"

// Outside the contractions every product and sum is rounded on its own, as the
// elementwise reference formulation rounds it: a multiply-add fused here or
// not, depending on how the compiler happens to schedule the surrounding code,
// moves the inputs of the bf16 rounding points by an ulp and flips rounded q/k
// elements.
#pragma clang fp contract(off)

namespace tf {
namespace {

constexpr int kThreads = 512;
constexpr int kNMax = 128;
constexpr int kPMax = 64;
constexpr int kRowLanes = 8;                // lanes per row in the rotation

// sigmoid with the correctly rounded-to-1-ulp expf rather than the fast
// hardware exp: the trapezoid weights feed the bf16 rounding of kr.
__device__ __forceinline__ float sigmoid_exact(float x) { return 1.0f / (1.0f + expf(-x)); }

// tanh in fp64, (1 - e) / (1 + e) with e = exp(-2|x|): 2^n times the Taylor sum
// of exp on [-ln2/2, ln2/2] to the 12th power (remainder below 2e-16), and the
// quotient from the hardware reciprocal and two Newton steps. Its absolute
// error, which is what the phase sum carries, is a few 1e-16. NaN stays NaN.
__device__ __forceinline__ double tanh_f64(double x) {
  const double ax = __builtin_fabs(x);
  const double y = ax * -2.8853900817779268;  // -2 log2(e)
  const double n = __builtin_rint(y);
  const double r = (y - n) * 0.6931471805599453;
  constexpr double kInvFact[13] = {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040, 1.0 / 40320,
                                   1.0 / 362880, 1.0 / 3628800, 1.0 / 39916800, 1.0 / 479001600};
  double p = kInvFact[12];
#pragma unroll
  for (int i = 11; i >= 0; --i) p = __builtin_fma(p, r, kInvFact[i]);
  double e = __builtin_ldexp(p, static_cast<int>(n));
  e = ax > 40.0 ? 0.0 : e;
  const double den = 1.0 + e;
  double q = __builtin_amdgcn_rcp(den);
  q = __builtin_fma(q, __builtin_fma(-den, q, 1.0), q);
  q = __builtin_fma(q, __builtin_fma(-den, q, 1.0), q);
  return __builtin_copysign((1.0 - e) * q, x);
}

// Inclusive fp64 prefix sum over the 64 lanes of the wave on DPP.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_f64(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint64_t lo = dpp_u32<CTRL, ROW_MASK>(static_cast<uint32_t>(u));
  const uint64_t hi = dpp_u32<CTRL, ROW_MASK>(static_cast<uint32_t>(u >> 32));
  return __builtin_bit_cast(double, lo | (hi << 32));
}
__device__ __forceinline__ double wave_scan_f64(double x) {
  x += dpp_f64<kDppRowShr + 1>(x);
  x += dpp_f64<kDppRowShr + 2>(x);
  x += dpp_f64<kDppRowShr + 4>(x);
  x += dpp_f64<kDppRowShr + 8>(x);
  x += dpp_f64<kDppRowBcast15, 0xa>(x);
  x += dpp_f64<kDppRowBcast31, 0xc>(x);
  return x;
}
__device__ __forceinline__ double last_lane_f64(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint64_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u), 63));
  const uint64_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u >> 32), 63));
  return __builtin_bit_cast(double, lo | (hi << 32));
}

// Four consecutive elements of a 16- or 32-bit float row at an address that is
// a multiple of four elements.
__device__ __forceinline__ float4 load4_f32(const void* p, int dtype, int64_t i) {
  if (dtype == TF_FLOAT32) return *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
  const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
  if (dtype == TF_BFLOAT16) return make_float4(lo_f(u.x), hi_f(u.x), lo_f(u.y), hi_f(u.y));
  const _Float16* f = reinterpret_cast<const _Float16*>(&u);
  return make_float4(static_cast<float>(f[0]), static_cast<float>(f[1]), static_cast<float>(f[2]),
                     static_cast<float>(f[3]));
}

// Elements n0 .. n0 + 3 of a row (0 past `n`).
template <typename I>
__device__ __forceinline__ float4 load_piece(const void* p, int dtype, I row, I st, int n0, int n, bool vec) {
  if (vec) return n0 < n ? load4_f32(p, dtype, row + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
  float x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = n0 + j < n ? load_f32(p, dtype, row + (n0 + j) * st) : 0.f;
  return make_float4(x[0], x[1], x[2], x[3]);
}

__device__ __forceinline__ f32x16 mfma_f32(float x, float y, const f32x16& acc) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
}

// Operand block with strides and offsets of type I: 32-bit ones where every
// offset fits (address arithmetic in one register), else 64-bit ones. A
// reversed call's time strides are negated; the kernel starts at row L - 1.
template <typename I>
struct GenericParams {
  tf_mamba_args a;
  I q[4], k[4], v[4], z[4], g[4], o[4];  // [batch, time, head, element]
  I ad[3], dt[3], tr[3];                 // [batch, head, time]
  int qvec, kvec, vvec;                  // rows can be read four elements at a time
  // chunk-parallel form: G segments per unit; per (unit, segment but the last) the
  // state in the walk's registers' order, per (unit, segment) log2 decay and phase
  // sums (revolutions, [G][64])
  int G;
  float4* state;
  float* decay;
  double* phase;
};

// First chunk of segment g of `chunks`, split as evenly as G segments allow.
__device__ __forceinline__ int first_chunk(int chunks, int G, int g) {
  return g * (chunks / G) + min(g, chunks % G);
}

template <int NT>
struct GenericShared {
  static constexpr int NP = 32 * NT;   // padded state dim
  static constexpr int NS = NP + 4;    // row stride: 16-byte pieces of 8 rows on distinct banks
  static constexpr int TS = NP + 2;    // trig row stride (NP / 2 pairs of cos, sin)
  static constexpr int VS = kPMax + 4;
  static constexpr int SS = kChunk + 4;
  float qr[kChunk * NS];
  float kr[kChunk * NS];
  float st[kPMax * NS];  // state [p][n] entering the chunk, rounded to q's dtype
  float v[kChunk * VS];
  union {
    float trig[kChunk * TS];  // until the rotation
    float sc[kChunk * SS];    // from the products on
  };
  float qb[NP], kb[NP], qw[NP], kw[NP];  // biases and norm weights, 0 past the state dim
  float cs[kChunk], gamma[kChunk], scale[kChunk], dt[kChunk], wv[kChunk], ecs[kChunk], qk[kChunk];
  int wild;  // the chunk's values hold an infinity or NaN
};

// 16 elements at offsets off(e) of a float array of any dtype (one branch on
// the dtype, not one per element).
template <typename F>
__device__ __forceinline__ void gather16(const void* p, int dtype, F&& off, float (&x)[16]) {
  if (dtype == TF_FLOAT32) {
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = static_cast<const float*>(p)[off(e)];
  } else if (dtype == TF_BFLOAT16) {
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = bf16_to_f32(static_cast<const uint16_t*>(p)[off(e)]);
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = static_cast<float>(static_cast<const _Float16*>(p)[off(e)]);
  }
}

template <typename F>
__device__ __forceinline__ void scatter16(void* p, int dtype, F&& off, const float (&x)[16], int count) {
  if (dtype == TF_FLOAT32) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (e < count) static_cast<float*>(p)[off(e)] = x[e];
  } else if (dtype == TF_BFLOAT16) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (e < count) static_cast<uint16_t*>(p)[off(e)] = f32_to_bf16(x[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (e < count) static_cast<_Float16*>(p)[off(e)] = static_cast<_Float16>(x[e]);
  }
}

// NT: 32-channel tiles of the state dim. RP: phase pairs per wave (8 RP >= R).
// ROUND: some operand is 16-bit, so the rounding points are not the identity.
// MODE 0: outputs of the unit's (or, P.G > 1, the segment's) chunks. MODE 1: the
// segment's state from zero state and phase, its log2 decay and phase sums.
template <int NT, int RP, bool ROUND, typename I, int MODE>
__global__ __launch_bounds__(kThreads) void mamba_generic_kernel(const GenericParams<I> P) {
  using Sm = GenericShared<NT>;
  constexpr int NS = Sm::NS, TS = Sm::TS, VS = Sm::VS, SS = Sm::SS;
  __shared__ __align__(16) Sm sh;
  const tf_mamba_args& a = P.a;
  const int h = blockIdx.x;
  const int b = blockIdx.y;
  const int seg = blockIdx.z;
  if (MODE == 1 && seg == P.G - 1) return;  // no segment starts from the last one's state
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int n_state = static_cast<int>(a.state);
  const int p_dim = static_cast<int>(a.head_dim);
  const int rot = static_cast<int>(a.rotary);
  const int T = static_cast<int>(a.time);
  const int qh = h / static_cast<int>(a.heads / a.qk_heads);
  const int L = valid_length(a, b);
  // reverse: step t < L reads and writes row L-1-t; steps >= L have no row
  const bool rev = a.reverse != 0;
  const int tlim = rev ? L : T;
  const I roff = rev ? max(L - 1, 0) : 0;
  auto rnd = [](float x, int dtype) { return ROUND ? round_to(x, dtype) : x; };
  const bool raw = a.dt_bias != nullptr;
  const bool norm = a.q_norm != nullptr;
  const float step_bias = raw ? a.dt_bias[h] : 0.f;

  const I qo = b * P.q[0] - roff * P.q[1] + qh * P.q[2];
  const I ko = b * P.k[0] - roff * P.k[1] + qh * P.k[2];
  const I vo = b * P.v[0] - roff * P.v[1] + h * P.v[2];
  const I zo = b * P.z[0] - roff * P.z[1] + h * P.z[2];
  const I oo = b * P.o[0] - roff * P.o[1] + h * P.o[2];
  const I go = b * P.g[0] - roff * P.g[1] + h * P.g[2];
  const I ao = b * P.ad[0] + h * P.ad[1] - roff * P.ad[2];
  const I dto = b * P.dt[0] + h * P.dt[1] - roff * P.dt[2];
  const I tro = b * P.tr[0] + h * P.tr[1] - roff * P.tr[2];

  const float skip = a.d[h];
  const int total = (T + kChunk - 1) / kChunk;
  const int nvalid = (L + kChunk - 1) / kChunk;
  const int c0 = min(first_chunk(total, P.G, seg), nvalid);
  const int nchunks = min(first_chunk(total, P.G, seg + 1), nvalid);  // the segment's chunks end here
  const int unit = b * static_cast<int>(a.heads) + h;
  // output waves: rows 32 th .., columns 32 pt ..; state waves: tiles s, s + 4 of (n, p)
  const int PT = p_dim > 32 ? 2 : 1;
  const int th = (w & 3) >> 1, pt = w & 1;
  const bool out_wave = w < 4 && pt < PT;
  const int s_idx = w - 4;

  // raw operands of one chunk, requested one chunk ahead
  float4 xq[NT], xk[NT], xv[2];
  float ang[RP];
  float c_dt = 0.f, c_dn = 0.f, c_ad = 0.f, c_tr = 0.f, c_tn = 0.f;
  auto load_chunk = [&](int c, int tid) {
    const int lane = tid & 63, rrow = tid / kRowLanes, grp = tid % kRowLanes;
    const int t = c * kChunk + rrow;
    const I r = min(t, L - 1);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if (MODE == 0) xq[j] = load_piece(a.q, a.q_dtype, qo + r * P.q[1], P.q[3], 4 * grp + 32 * j, n_state, P.qvec);
      xk[j] = load_piece(a.k, a.k_dtype, ko + r * P.k[1], P.k[3], 4 * grp + 32 * j, n_state, P.kvec);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
      xv[j] = load_piece(a.v, a.v_dtype, vo + r * P.v[1], P.v[3], 4 * grp + 32 * j, p_dim, P.vvec);
    const int tl = c * kChunk + lane;
    const I rl = min(tl, L - 1);
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const int pair = w * RP + i;
      ang[i] = pair < rot ? load_f32(a.angles, a.angles_dtype, go + rl * P.g[1] + pair * P.g[3]) : 0.f;
    }
    if (w == 0) {
      // rows clamped to ones that exist, masked where used
      const I rn = max(min(tl + 1, tlim - 1), 0);
      c_dt = load_f32(a.dt, a.dt_dtype, dto + rl * P.dt[2]);
      c_dn = load_f32(a.dt, a.dt_dtype, dto + rn * P.dt[2]);
      c_ad = load_f32(a.adt, a.adt_dtype, ao + rl * P.ad[2]);
      c_tr = load_f32(a.trap, a.trap_dtype, tro + rl * P.tr[2]);
      c_tn = load_f32(a.trap, a.trap_dtype, tro + rn * P.tr[2]);
    }
  };

  // The state copy the products read, channels n0 .. n0 + 3: 0 past the state dim,
  // where a value that is not finite leaves 0 x infinity, and a query's 0 meets it.
  auto put_state = [&](int row, int n0, float4 x) {
    if (n_state < Sm::NP) {
      x.x = n0 < n_state ? x.x : 0.f, x.y = n0 + 1 < n_state ? x.y : 0.f;
      x.z = n0 + 2 < n_state ? x.z : 0.f, x.w = n0 + 3 < n_state ? x.w : 0.f;
    }
    *reinterpret_cast<float4*>(&sh.st[row * NS + n0]) = x;
  };

  f32x16 state[2] = {zero16(), zero16()};  // state waves
  double carry[RP];             // phase entering the chunk, revolutions
  float seg_log2 = 0.f;
#pragma unroll
  for (int i = 0; i < RP; ++i) carry[i] = 0.0;
  if (MODE == 0 && seg > 0 && nchunks > c0) {
    // the phase and state entering the segment
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const int pair = w * RP + i, ln = static_cast<int>(threadIdx.x & 63);
      double part = 0.0;
      if (pair < rot)
        for (int g = ln; g < seg; g += 64) part += P.phase[(static_cast<int64_t>(unit) * P.G + g) * 64 + pair];
      const double sum = last_lane_f64(wave_scan_f64(part));
      carry[i] = sum - __builtin_rint(sum);
    }
    const float4* rec = P.state + (static_cast<int64_t>(unit) * (P.G - 1) + seg - 1) * (NT * PT * 256);
    if (w >= 4) {
      const int ln = static_cast<int>(threadIdx.x & 63);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int tile = s_idx + 4 * i;
        if (tile < NT * PT) {
          const int sp = PT == 2 ? tile & 1 : 0, sn = PT == 2 ? tile >> 1 : tile;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4 x = rec[(tile * 4 + g) * 64 + ln];
            state[i][4 * g] = x.x, state[i][4 * g + 1] = x.y, state[i][4 * g + 2] = x.z, state[i][4 * g + 3] = x.w;
            put_state(32 * sp + (ln & 31), 32 * sn + 8 * g + 4 * (ln >> 5), x);
          }
        }
      }
    }
  } else if (MODE == 0) {
    for (int e = static_cast<int>(threadIdx.x); e < kPMax * NS; e += kThreads) sh.st[e] = 0.f;
  }
  for (int e = static_cast<int>(threadIdx.x); e < Sm::NP; e += kThreads) {
    const bool on = e < n_state;
    sh.qb[e] = on ? a.qb[h * n_state + e] : 0.f;
    sh.kb[e] = on ? a.kb[h * n_state + e] : 0.f;
    sh.qw[e] = on && norm ? a.q_norm[e] : 0.f;
    sh.kw[e] = on && norm ? a.k_norm[e] : 0.f;
  }
  if (nchunks > c0) load_chunk(c0, static_cast<int>(threadIdx.x));

  for (int c = c0; c < nchunks; ++c) {
    const int t0 = c * kChunk;
    // lane-derived indices from a thread index the compiler cannot see through:
    // hoisted out of the loop, the addresses they feed would live across it
    // and spill
    int tid = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int c32 = lane & 31, hh = lane >> 5;
    const int rrow = tid / kRowLanes, grp = tid % kRowLanes;  // rotation: row and channel group
    if (w == 0) {
      const int t = t0 + lane;
      const bool valid = t < L, next = t + 1 < tlim;
      float dt = c_dt, dn = c_dn, ad = c_ad;
      if (raw) {  // controls from the raw a/ddt columns (primitives.py:209-214)
        dt = control_step(dt, step_bias);
        dn = control_step(dn, step_bias);
        ad = control_decay(ad, dt, a.a_floor);
      }
      dt = valid ? dt : 0.f;
      dn = next ? dn : 0.f;
      ad = valid ? ad : 0.f;
      const float tr = sigmoid_exact(valid ? c_tr : 0.f), tn = sigmoid_exact(next ? c_tn : 0.f);
      const float gamma = dt * tr;
      const float cs = wave_scan_dpp(ad * kLog2e);
      const float tot = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cs), 63));
      sh.cs[lane] = cs;
      sh.wv[lane] = exp2f(tot - cs);
      sh.ecs[lane] = exp2f(cs);
      sh.gamma[lane] = gamma;
      sh.scale[lane] = dn * (1.f - tn) + gamma;
      sh.dt[lane] = dt;
      if (lane == 0) sh.wild = 0;
    }
    // the rotary's tanh does not wait for the controls
    double om[RP];
#pragma unroll
    for (int i = 0; i < RP; ++i) om[i] = tanh_f64(static_cast<double>(ang[i]));
    __syncthreads();
    // phase in revolutions, accumulated in fp64 (mamba_fused.py:102-111): pi tanh dt
    // radians = tanh dt / 2 revolutions; rows past the length add 0
    {
      const double dt = static_cast<double>(sh.dt[lane]);
#pragma unroll
      for (int i = 0; i < RP; ++i) {
        const int pair = w * RP + i;
        if (pair < rot) {
          const double inc = t0 + lane < L ? om[i] * dt * 0.5 : 0.0;
          const double sum = wave_scan_f64(inc) + carry[i];
          const float rev2 = static_cast<float>(2.0 * (sum - __builtin_rint(sum)));
          float si, co;
          sincospif(rev2, &si, &co);
          *reinterpret_cast<float2*>(&sh.trig[lane * TS + 2 * pair]) = make_float2(co, si);
          const double last = last_lane_f64(sum);
          carry[i] = last - __builtin_rint(last);
        }
      }
    }
    __syncthreads();
    // B/C norm, bias, skip term, rotation, scale and rounding (mamba_fused.py:112-135)
    {
      const bool valid = t0 + rrow < L;
      float rq = 1.f, rk = 1.f;
      if (norm) {
        // RMSNorm of the raw rows (mamba.py:56-57, kernels/__init__.py:10-12)
        float sq = 0.f, sk = 0.f;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if (MODE == 0)
            sq += xq[j].x * xq[j].x, sq += xq[j].y * xq[j].y, sq += xq[j].z * xq[j].z, sq += xq[j].w * xq[j].w;
          sk += xk[j].x * xk[j].x, sk += xk[j].y * xk[j].y, sk += xk[j].z * xk[j].z, sk += xk[j].w * xk[j].w;
        }
        if (MODE == 0) rq = rsqrtf(group8_sum(sq) / static_cast<float>(n_state) + a.norm_eps);
        rk = rsqrtf(group8_sum(sk) / static_cast<float>(n_state) + a.norm_eps);
      }
      const float scl = sh.scale[rrow];
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n0 = 4 * grp + 32 * j;
        if (MODE == 1) xq[j] = make_float4(0.f, 0.f, 0.f, 0.f);  // no query is formed
        float q[4] = {xq[j].x, xq[j].y, xq[j].z, xq[j].w}, k[4] = {xk[j].x, xk[j].y, xk[j].z, xk[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (norm) {
            // rounded to the operand dtype as the norm's output is
            q[e] = rnd(q[e] * rq * sh.qw[n0 + e], a.q_dtype);
            k[e] = rnd(k[e] * rk * sh.kw[n0 + e], a.k_dtype);
          }
          q[e] += sh.qb[n0 + e];
          k[e] += sh.kb[n0 + e];
          dot += q[e] * k[e];  // unrotated biased vectors (:124)
        }
        float qv[4], kv[4];
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          float co = 1.f, si = 0.f;
          if ((n0 + e) / 2 < rot) {
            const float2 cs = *reinterpret_cast<const float2*>(&sh.trig[rrow * TS + n0 + e]);
            co = cs.x, si = cs.y;
          }
          qv[e] = rnd(q[e] * co - q[e + 1] * si, a.q_dtype);
          qv[e + 1] = rnd(q[e] * si + q[e + 1] * co, a.q_dtype);
          kv[e] = rnd((k[e] * co - k[e + 1] * si) * scl, a.k_dtype);
          kv[e + 1] = rnd((k[e] * si + k[e + 1] * co) * scl, a.k_dtype);
        }
        const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (MODE == 0) *reinterpret_cast<float4*>(&sh.qr[rrow * NS + n0]) = valid ? make_float4(qv[0], qv[1], qv[2], qv[3]) : z4;
        *reinterpret_cast<float4*>(&sh.kr[rrow * NS + n0]) = valid ? make_float4(kv[0], kv[1], kv[2], kv[3]) : z4;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float4 x = valid ? xv[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(&sh.v[rrow * VS + 4 * grp + 32 * j]) = x;
        if (!isfinite(x.x) || !isfinite(x.y) || !isfinite(x.z) || !isfinite(x.w)) sh.wild = 1;
      }
      dot = group8_sum(dot);
      if (grp == 0) sh.qk[rrow] = dot * sh.gamma[rrow];
    }
    // the gate rows of this chunk and the next chunk's operands, in flight over the products
    float zz[16];
    const bool late = t0 + 32 >= L;  // the chunk's second half has no valid row
    const bool y_on = MODE == 0 && out_wave && !(late && th == 1);
    if (y_on) {
      // rows and columns clamped to ones that exist; masked at the store
      const I zc = zo + min(32 * pt + c32, p_dim - 1) * P.z[3];
      gather16(a.z, a.z_dtype, [&](int e) -> I { return zc + min(t0 + 32 * th + drow(e, hh), L - 1) * P.z[1]; }, zz);
    }
    if (c + 1 < nchunks) load_chunk(c + 1, tid);
    __syncthreads();
    f32x16 inter = zero16();
    if (y_on) {
      const float* x = &sh.qr[(32 * th + c32) * NS + 4 * hh];
      const float* y = &sh.st[(32 * pt + c32) * NS + 4 * hh];
#pragma unroll 4
      for (int s = 0; s < 4 * NT; ++s) {
        const float4 xa = *reinterpret_cast<const float4*>(x + 8 * s), ya = *reinterpret_cast<const float4*>(y + 8 * s);
        inter = mfma_f32(xa.x, ya.x, inter);
        inter = mfma_f32(xa.y, ya.y, inter);
        inter = mfma_f32(xa.z, ya.z, inter);
        inter = mfma_f32(xa.w, ya.w, inter);
      }
    } else if (MODE == 0 && w >= 4 && w < 7 && !(late && w > 4)) {
      // strictly causal decayed scores, rounded to v's dtype (mamba_fused.py:144-146):
      // lane = t, values = u
      const int tt = w > 4 ? 1 : 0, uu = w > 5 ? 1 : 0;
      const float* x = &sh.kr[(32 * uu + c32) * NS + 4 * hh];
      const float* y = &sh.qr[(32 * tt + c32) * NS + 4 * hh];
      f32x16 acc = zero16();
#pragma unroll 4
      for (int s = 0; s < 4 * NT; ++s) {
        const float4 xa = *reinterpret_cast<const float4*>(x + 8 * s), ya = *reinterpret_cast<const float4*>(y + 8 * s);
        acc = mfma_f32(xa.x, ya.x, acc);
        acc = mfma_f32(xa.y, ya.y, acc);
        acc = mfma_f32(xa.z, ya.z, acc);
        acc = mfma_f32(xa.w, ya.w, acc);
      }
      const int t = 32 * tt + c32;
      const float cst = sh.cs[t];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float val[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int u = 32 * uu + drow(4 * g + e, hh);
          const float x2 = rnd(acc[4 * g + e] * exp2f(fminf(cst - sh.cs[u], 0.f)), a.v_dtype);
          val[e] = u < t ? x2 : 0.f;
        }
        *reinterpret_cast<float4*>(&sh.sc[t * SS + 32 * uu + 8 * g + 4 * hh]) =
            make_float4(val[0], val[1], val[2], val[3]);
      }
    }
    __syncthreads();
    if (y_on) {
      // outputs (mamba_fused.py:143-149): lane = p, values = t
      f32x16 intra = zero16();
      const float* x = &sh.sc[(32 * th + c32) * SS + 4 * hh];
      const float* y = &sh.v[4 * hh * VS + 32 * pt + c32];
      const int p = 32 * pt + c32;
      if (!sh.wild) {
#pragma unroll 4
        for (int s = 0; s < 4 * (th + 1); ++s) {
          const float4 xa = *reinterpret_cast<const float4*>(x + 8 * s);
          const float* yr = y + 8 * s * VS;
          intra = mfma_f32(xa.x, yr[0], intra);
          intra = mfma_f32(xa.y, yr[VS], intra);
          intra = mfma_f32(xa.z, yr[2 * VS], intra);
          intra = mfma_f32(xa.w, yr[3 * VS], intra);
        }
      } else {
        // a masked score's 0 times a later row's infinity or NaN would reach
        // earlier rows: sum the preceding rows alone
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = 32 * th + drow(e, hh);
          float sum = 0.f;
          for (int u = 0; u < r; ++u) sum += sh.sc[r * SS + u] * sh.v[u * VS + p];
          intra[e] = sum;
        }
      }
      float y2[16];
      int count = 0;  // the lane's rows below the length: they come in order
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = 32 * th + drow(e, hh);
        count += t0 + r < L ? 1 : 0;
        y2[e] = inter[e] * sh.ecs[r] + intra[e] + (skip + sh.qk[r]) * sh.v[r * VS + p];
        y2[e] *= zz[e] * sigmoidf(zz[e]);
      }
      const I oc = oo + p * P.o[3] + (t0 + 32 * th) * P.o[1];
      if (p < p_dim)
        scatter16(a.out, a.out_dtype, [&](int e) -> I { return oc + drow(e, hh) * P.o[1]; }, y2, count);
    } else if (w >= 4 && (c + 1 < nchunks || (MODE == 1 && c + 1 < nvalid))) {
      // state update S <- S 2^tot + round_k(v 2^(tot-cs))^T kr (mamba_fused.py:150-152):
      // lane = p, values = n
      const float decay = sh.ecs[kChunk - 1];
      seg_log2 += sh.cs[kChunk - 1];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int tile = s_idx + 4 * i;
        if (tile < NT * PT) {
          const int sp = PT == 2 ? tile & 1 : 0, sn = PT == 2 ? tile >> 1 : tile;
          const float* x = &sh.kr[hh * NS + 32 * sn + c32];
          const float* y = &sh.v[hh * VS + 32 * sp + c32];
          f32x16 acc = zero16();
#pragma unroll 8
          for (int u = 0; u < kChunk / 2; ++u)
            acc = mfma_f32(x[2 * u * NS], rnd(y[2 * u * VS] * sh.wv[2 * u + hh], a.k_dtype), acc);
#pragma unroll
          for (int e = 0; e < 16; ++e) state[i][e] = state[i][e] * decay + acc[e];
#pragma unroll
          for (int g = 0; g < 4; ++g)
            put_state(32 * sp + c32, 32 * sn + 8 * g + 4 * hh,
                      make_float4(rnd(state[i][4 * g], a.q_dtype), rnd(state[i][4 * g + 1], a.q_dtype),
                                  rnd(state[i][4 * g + 2], a.q_dtype), rnd(state[i][4 * g + 3], a.q_dtype)));
        }
      }
    }
    __syncthreads();
  }
  if constexpr (MODE == 1) {
    float4* rec = P.state + (static_cast<int64_t>(unit) * (P.G - 1) + seg) * (NT * PT * 256);
    const int ln = static_cast<int>(threadIdx.x & 63);
    if (w >= 4) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int tile = s_idx + 4 * i;
        if (tile < NT * PT) {
#pragma unroll
          for (int g = 0; g < 4; ++g)
            rec[(tile * 4 + g) * 64 + ln] =
                make_float4(state[i][4 * g], state[i][4 * g + 1], state[i][4 * g + 2], state[i][4 * g + 3]);
        }
      }
      if (w == 4 && ln == 0) P.decay[static_cast<int64_t>(unit) * P.G + seg] = seg_log2;
    }
#pragma unroll
    for (int i = 0; i < RP; ++i)
      if (ln == 0 && w * RP + i < rot) P.phase[(static_cast<int64_t>(unit) * P.G + seg) * 64 + w * RP + i] = carry[i];
  } else {
    // rows past the valid prefix (the same rows in either direction)
    const I st = rev ? -P.o[1] : P.o[1];
    const I of = b * P.o[0] + h * P.o[2];
    const int stop = min(first_chunk(total, P.G, seg + 1) * kChunk, T);
    for (int t = max(first_chunk(total, P.G, seg) * kChunk, L) + w; t < stop; t += kThreads / 64) {
      const int p = static_cast<int>(threadIdx.x & 63);
      if (p < p_dim) store_f32(a.out, a.out_dtype, of + t * st + p * P.o[3], 0.f);
    }
  }
}

// Replaces each unit's segment summaries by the states entering the next
// segments: S_1 = d_0, S_{g+1} = S_g 2^dec_g + turn_g(d_g), where turn_g rotates
// the rotary row pairs by the phase entering segment g (a summary is formed from
// phase 0 at its segment's start, and is linear in the keys that phase turns; an
// infinite element turns into one that is not a number).
// Thread f of a unit takes float4 f of its records: channels n .. n + 3.
template <typename I>
__global__ __launch_bounds__(64) void generic_scan_kernel(const GenericParams<I> P, int kf4, int pt) {
  constexpr int kBatch = 4;
  const int slices = kf4 / 64;
  const int unit = blockIdx.x / slices;
  const int f = (blockIdx.x - unit * slices) * 64 + threadIdx.x;
  const int tile = f >> 8, n = 32 * (pt == 2 ? tile >> 1 : tile) + 8 * ((f >> 6) & 3) + 4 * ((f >> 5) & 1);
  const int G = P.G, rot = static_cast<int>(P.a.rotary), pair = n / 2;
  float4* st = P.state + static_cast<int64_t>(unit) * (G - 1) * kf4 + f;
  const float* dec = P.decay + static_cast<int64_t>(unit) * G;
  const double* ph = P.phase + static_cast<int64_t>(unit) * G * 64 + pair;
  float4 run = make_float4(0.f, 0.f, 0.f, 0.f);
  double p0 = 0.0, p1 = 0.0;
  for (int g0 = 0; g0 < G - 1; g0 += kBatch) {
    float4 d[kBatch];
    double s0[kBatch], s1[kBatch];
    Factor m[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const int g = g0 + j;
      if (g < G - 1) {
        d[j] = st[static_cast<int64_t>(g) * kf4];
        m[j] = factor_of(dec[g]);
        s0[j] = pair < rot ? ph[g * 64] : 0.0;
        s1[j] = pair + 1 < rot ? ph[g * 64 + 1] : 0.0;
      }
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      if (g0 + j < G - 1) {
        float4 x = d[j];
        if (pair < rot) {
          float si, co;
          sincospif(static_cast<float>(2.0 * (p0 - __builtin_rint(p0))), &si, &co);
          x.x = d[j].x * co - d[j].y * si;
          x.y = d[j].x * si + d[j].y * co;
        }
        if (pair + 1 < rot) {
          float si, co;
          sincospif(static_cast<float>(2.0 * (p1 - __builtin_rint(p1))), &si, &co);
          x.z = d[j].z * co - d[j].w * si;
          x.w = d[j].z * si + d[j].w * co;
        }
        p0 += s0[j], p1 += s1[j];
        const Factor f2 = m[j];
        run.x = ldexpf(run.x * f2.mant, f2.exp) + x.x, run.y = ldexpf(run.y * f2.mant, f2.exp) + x.y;
        run.z = ldexpf(run.z * f2.mant, f2.exp) + x.z, run.w = ldexpf(run.w * f2.mant, f2.exp) + x.w;
        st[static_cast<int64_t>(g0 + j) * kf4] = run;
      }
    }
  }
}

// Chunk-parallel plan, for fp32 operands (a summary's keys are rounded in its own
// phase frame, which is the same state only while the rounding is the identity):
// segments of at least two chunks, about one workgroup per CU.
struct GenericPlan {
  int G = 1;
  int kf4 = 0, pt = 1;
  int64_t decay_off = 0, phase_off = 0, bytes = 0;
};

bool rounds(const tf_mamba_args& a) {
  return a.q_dtype != TF_FLOAT32 || a.k_dtype != TF_FLOAT32 || a.v_dtype != TF_FLOAT32;
}

GenericPlan generic_plan(const tf_mamba_args& a) {
  GenericPlan p;
  if (rounds(a) || !offsets_fit(a)) return p;
  const int64_t units = a.batch * a.heads, chunks = (a.time + kChunk - 1) / kChunk;
  if (units <= 0 || units > 128) return p;
  const int64_t g = std::min<int64_t>(256 / units, chunks / 2);
  if (g < 2) return p;
  p.G = static_cast<int>(g);
  const int nt = a.state <= 32 ? 1 : (a.state <= 64 ? 2 : 4);
  p.pt = a.head_dim > 32 ? 2 : 1;
  p.kf4 = nt * p.pt * 256;
  auto up = [](int64_t x) { return (x + 255) & ~int64_t(255); };
  p.phase_off = up(units * (g - 1) * p.kf4 * 16);
  p.decay_off = p.phase_off + up(units * g * 64 * 8);
  p.bytes = p.decay_off + up(units * g * 4);
  return p;
}

template <typename I>
GenericParams<I> make_generic(const tf_mamba_args& a);

template <int NT, int RP, typename I>
int launch_pairs(const tf_mamba_args& a, hipStream_t stream) {
  GenericParams<I> P = make_generic<I>(a);
  const GenericPlan plan = generic_plan(a);
  if (std::is_same_v<I, int32_t> && plan.G > 1 && a.workspace != nullptr && aligned(a.workspace, 256) &&
      a.workspace_bytes >= plan.bytes) {
    char* ws = static_cast<char*>(a.workspace);
    P.G = plan.G;
    P.state = reinterpret_cast<float4*>(ws);
    P.phase = reinterpret_cast<double*>(ws + plan.phase_off);
    P.decay = reinterpret_cast<float*>(ws + plan.decay_off);
  }
  const dim3 grid(static_cast<uint32_t>(a.heads), static_cast<uint32_t>(a.batch), static_cast<uint32_t>(P.G));
  if (rounds(a)) {
    hipLaunchKernelGGL((mamba_generic_kernel<NT, RP, true, I, 0>), grid, dim3(kThreads), 0, stream, P);
    return launch_status();
  }
  if constexpr (std::is_same_v<I, int32_t>) {
    if (P.G > 1) {
      hipLaunchKernelGGL((mamba_generic_kernel<NT, RP, false, I, 1>), grid, dim3(kThreads), 0, stream, P);
      if (const int rc = launch_status()) return rc;
      const int64_t units = a.batch * a.heads;
      hipLaunchKernelGGL(generic_scan_kernel<I>, dim3(static_cast<uint32_t>(units * (plan.kf4 / 64))), dim3(64), 0,
                         stream, P, plan.kf4, plan.pt);
      if (const int rc = launch_status()) return rc;
    }
  }
  hipLaunchKernelGGL((mamba_generic_kernel<NT, RP, false, I, 0>), grid, dim3(kThreads), 0, stream, P);
  return launch_status();
}

template <int NT>
int launch_tiles(const tf_mamba_args& a, hipStream_t stream) {
  if (!offsets_fit(a)) return launch_pairs<NT, 2 * NT, int64_t>(a, stream);
  // a quarter of the state dim rotates in the models; a half at most
  if (a.rotary <= 8 * NT) return launch_pairs<NT, NT, int32_t>(a, stream);
  return launch_pairs<NT, 2 * NT, int32_t>(a, stream);
}

// Four elements at a time: whole pieces inside the row, aligned at every row.
int vec4(const void* p, int dtype, const int64_t* st, int64_t n) {
  const int es = dtype_size(dtype);
  return n % 4 == 0 && rows_vectorisable(p, st, es, 4 * es);
}

template <typename I>
GenericParams<I> make_generic(const tf_mamba_args& a) {
  GenericParams<I> P;
  P.a = a;
  const I sign = a.reverse ? -1 : 1;
  auto four = [&](I(&d)[4], const int64_t* s) {
    for (int i = 0; i < 4; ++i) d[i] = static_cast<I>(s[i]);
    d[1] *= sign;
  };
  auto three = [&](I(&d)[3], const int64_t* s) {
    for (int i = 0; i < 3; ++i) d[i] = static_cast<I>(s[i]);
    d[2] *= sign;
  };
  four(P.q, a.q_stride), four(P.k, a.k_stride), four(P.v, a.v_stride), four(P.z, a.z_stride);
  four(P.g, a.angles_stride), four(P.o, a.out_stride);
  three(P.ad, a.adt_stride), three(P.dt, a.dt_stride), three(P.tr, a.trap_stride);
  P.qvec = vec4(a.q, a.q_dtype, a.q_stride, a.state);
  P.kvec = vec4(a.k, a.k_dtype, a.k_stride, a.state);
  P.vvec = vec4(a.v, a.v_dtype, a.v_stride, a.head_dim);
  P.G = 1;
  P.state = nullptr;
  P.decay = nullptr;
  P.phase = nullptr;
  return P;
}

}  // namespace

bool generic_supported(const tf_mamba_args& a) {
  return a.state <= kNMax && a.head_dim <= kPMax;
}

int64_t generic_workspace_bytes(const tf_mamba_args& a) {
  const GenericPlan plan = generic_plan(a);
  return plan.G > 1 ? plan.bytes : 0;
}

int launch_generic(const tf_mamba_args& a, hipStream_t stream) {
  if (a.state <= 32) return launch_tiles<1>(a, stream);
  if (a.state <= 64) return launch_tiles<2>(a, stream);
  return launch_tiles<4>(a, stream);
}

}  // namespace tf
