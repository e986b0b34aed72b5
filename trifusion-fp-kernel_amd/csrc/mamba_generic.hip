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
// operands. N is padded to a multiple of 32 and P to 32 or 64 with zeros in LDS.
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
constexpr int kPairsPerWave = kNMax / 2 / 8;  // phase pairs of one wave, at most

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

// Inclusive fp64 prefix sum over the 64 lanes of the wave.
__device__ __forceinline__ double wave_scan_f64(double v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_up(v, off, 64);
    if (lane >= off) v += o;
  }
  return v;
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
__device__ __forceinline__ float4 load_piece(const void* p, int dtype, int64_t row, int64_t st, int n0, int n, bool vec) {
  if (vec) return n0 < n ? load4_f32(p, dtype, row + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
  float x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = n0 + j < n ? load_f32(p, dtype, row + (n0 + j) * st) : 0.f;
  return make_float4(x[0], x[1], x[2], x[3]);
}

__device__ __forceinline__ f32x16 mfma_f32(float x, float y, const f32x16& acc) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
}

// Rows of q/k (v) can be read four elements at a time.
struct GenericVec {
  int q, k, v;
};

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
  float cs[kChunk], gamma[kChunk], scale[kChunk], dt[kChunk], wv[kChunk], ecs[kChunk], qk[kChunk];
  int wild;  // the chunk's values hold an infinity or NaN
};

// NT: 32-channel tiles of the state dim. ROUND: some operand is 16-bit, so the
// rounding points are not the identity.
template <int NT, bool ROUND>
__global__ __launch_bounds__(kThreads) void mamba_generic_kernel(const tf_mamba_args a, const GenericVec vec) {
  using Sm = GenericShared<NT>;
  constexpr int NS = Sm::NS, TS = Sm::TS, VS = Sm::VS, SS = Sm::SS;
  __shared__ __align__(16) Sm sh;
  const int h = blockIdx.x;
  const int b = blockIdx.y;
  const int tid = static_cast<int>(threadIdx.x);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c32 = lane & 31, hh = lane >> 5;
  const int n_state = static_cast<int>(a.state);
  const int p_dim = static_cast<int>(a.head_dim);
  const int rot = static_cast<int>(a.rotary);
  const int T = static_cast<int>(a.time);
  const int qh = h / static_cast<int>(a.heads / a.qk_heads);
  const int L = valid_length(a, b);
  // reverse: step t < L reads and writes row L-1-t; steps >= L have no row
  const bool rev = a.reverse != 0;
  const int tlim = rev ? L : T;
  auto row = [&](int t) -> int64_t { return rev ? L - 1 - t : t; };
  auto rnd = [](float x, int dtype) { return ROUND ? round_to(x, dtype) : x; };
  const bool raw = a.dt_bias != nullptr;
  const bool norm = a.q_norm != nullptr;
  const float step_bias = raw ? a.dt_bias[h] : 0.f;

  const int64_t qo = b * a.q_stride[0] + qh * a.q_stride[2];
  const int64_t ko = b * a.k_stride[0] + qh * a.k_stride[2];
  const int64_t vo = b * a.v_stride[0] + h * a.v_stride[2];
  const int64_t zo = b * a.z_stride[0] + h * a.z_stride[2];
  const int64_t oo = b * a.out_stride[0] + h * a.out_stride[2];
  const int64_t go = b * a.angles_stride[0] + h * a.angles_stride[2];
  const int64_t ao = b * a.adt_stride[0] + h * a.adt_stride[1];
  const int64_t dto = b * a.dt_stride[0] + h * a.dt_stride[1];
  const int64_t tro = b * a.trap_stride[0] + h * a.trap_stride[1];

  const float skip = a.d[h];
  const int nchunks = (L + kChunk - 1) / kChunk;
  const int rrow = tid / kRowLanes, grp = tid % kRowLanes;  // rotation: row and channel group
  const int rp = (rot + 7) / 8;                             // phase pairs per wave
  // output waves: rows 32 th .., columns 32 pt ..; state waves: tiles s, s + 4 of (n, p)
  const int PT = p_dim > 32 ? 2 : 1;
  const int th = (w & 3) >> 1, pt = w & 1;
  const bool out_wave = w < 4 && pt < PT;
  const int s_idx = w - 4;

  // raw operands of one chunk, requested one chunk ahead
  float4 xq[NT], xk[NT], xv[2];
  float ang[kPairsPerWave];
  float c_dt = 0.f, c_dn = 0.f, c_ad = 0.f, c_tr = 0.f, c_tn = 0.f;
  auto load_chunk = [&](int c) {
    const int t = c * kChunk + rrow;
    const int64_t r = row(min(t, L - 1));
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      xq[j] = load_piece(a.q, a.q_dtype, qo + r * a.q_stride[1], a.q_stride[3], 4 * grp + 32 * j, n_state, vec.q);
      xk[j] = load_piece(a.k, a.k_dtype, ko + r * a.k_stride[1], a.k_stride[3], 4 * grp + 32 * j, n_state, vec.k);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
      xv[j] = load_piece(a.v, a.v_dtype, vo + r * a.v_stride[1], a.v_stride[3], 4 * grp + 32 * j, p_dim, vec.v);
    const int tl = c * kChunk + lane;
    const int64_t rl = row(min(tl, L - 1));
#pragma unroll
    for (int i = 0; i < kPairsPerWave; ++i) {
      const int pair = w * rp + i;
      ang[i] = i < rp && pair < rot
                   ? load_f32(a.angles, a.angles_dtype, go + rl * a.angles_stride[1] + pair * a.angles_stride[3])
                   : 0.f;
    }
    if (w == 0) {
      const bool valid = tl < L, next = tl + 1 < tlim;
      c_dt = valid ? load_f32(a.dt, a.dt_dtype, dto + rl * a.dt_stride[2]) : 0.f;
      c_dn = next ? load_f32(a.dt, a.dt_dtype, dto + row(tl + 1) * a.dt_stride[2]) : 0.f;
      c_ad = valid ? load_f32(a.adt, a.adt_dtype, ao + rl * a.adt_stride[2]) : 0.f;
      c_tr = valid ? load_f32(a.trap, a.trap_dtype, tro + rl * a.trap_stride[2]) : 0.f;
      c_tn = next ? load_f32(a.trap, a.trap_dtype, tro + row(tl + 1) * a.trap_stride[2]) : 0.f;
    }
  };

  f32x16 state[2] = {zero16(), zero16()};  // state waves
  double carry[kPairsPerWave];             // phase entering the chunk, revolutions
#pragma unroll
  for (int i = 0; i < kPairsPerWave; ++i) carry[i] = 0.0;
  for (int e = tid; e < kPMax * NS; e += kThreads) sh.st[e] = 0.f;
  if (nchunks > 0) load_chunk(0);

  for (int c = 0; c < nchunks; ++c) {
    const int t0 = c * kChunk;
    if (w == 0) {
      const int t = t0 + lane;
      const bool valid = t < L, next = t + 1 < tlim;
      float dt = c_dt, dn = c_dn, ad = c_ad;
      if (raw) {  // controls from the raw a/ddt columns (primitives.py:209-214)
        dt = valid ? control_step(dt, step_bias) : 0.f;
        dn = next ? control_step(dn, step_bias) : 0.f;
        ad = valid ? control_decay(ad, dt, a.a_floor) : 0.f;
      }
      const float tr = sigmoid_exact(c_tr), tn = sigmoid_exact(c_tn);
      const float gamma = dt * tr;
      const float cs = wave_inclusive_scan(ad * kLog2e);
      const float tot = __shfl(cs, 63, 64);
      sh.cs[lane] = cs;
      sh.wv[lane] = exp2f(tot - cs);
      sh.ecs[lane] = exp2f(cs);
      sh.gamma[lane] = gamma;
      sh.scale[lane] = dn * (1.f - tn) + gamma;
      sh.dt[lane] = dt;
      if (lane == 0) sh.wild = 0;
    }
    // the rotary's tanh does not wait for the controls
    double om[kPairsPerWave];
#pragma unroll
    for (int i = 0; i < kPairsPerWave; ++i)
      if (i < rp) om[i] = tanh_f64(static_cast<double>(ang[i]));
    __syncthreads();
    // phase in revolutions, accumulated in fp64 (mamba_fused.py:102-111): pi tanh dt
    // radians = tanh dt / 2 revolutions; rows past the length add 0
    {
      const double dt = static_cast<double>(sh.dt[lane]);
#pragma unroll
      for (int i = 0; i < kPairsPerWave; ++i) {
        const int pair = w * rp + i;
        if (i < rp && pair < rot) {
          const double inc = t0 + lane < L ? om[i] * dt * 0.5 : 0.0;
          const double sum = wave_scan_f64(inc, lane) + carry[i];
          const float rev2 = static_cast<float>(2.0 * (sum - __builtin_rint(sum)));
          float si, co;
          sincospif(rev2, &si, &co);
          *reinterpret_cast<float2*>(&sh.trig[lane * TS + 2 * pair]) = make_float2(co, si);
          const double last = __shfl(sum, 63, 64);
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
          sq += xq[j].x * xq[j].x, sq += xq[j].y * xq[j].y, sq += xq[j].z * xq[j].z, sq += xq[j].w * xq[j].w;
          sk += xk[j].x * xk[j].x, sk += xk[j].y * xk[j].y, sk += xk[j].z * xk[j].z, sk += xk[j].w * xk[j].w;
        }
        rq = rsqrtf(group8_sum(sq) / static_cast<float>(n_state) + a.norm_eps);
        rk = rsqrtf(group8_sum(sk) / static_cast<float>(n_state) + a.norm_eps);
      }
      const float scl = sh.scale[rrow];
      float dot = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int n0 = 4 * grp + 32 * j;
        float q[4] = {xq[j].x, xq[j].y, xq[j].z, xq[j].w}, k[4] = {xk[j].x, xk[j].y, xk[j].z, xk[j].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n0 + e;
          if (n < n_state) {
            if (norm) {
              // rounded to the operand dtype as the norm's output is
              q[e] = rnd(q[e] * rq * a.q_norm[n], a.q_dtype);
              k[e] = rnd(k[e] * rk * a.k_norm[n], a.k_dtype);
            }
            q[e] += a.qb[h * n_state + n];
            k[e] += a.kb[h * n_state + n];
          }
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
        *reinterpret_cast<float4*>(&sh.qr[rrow * NS + n0]) = valid ? make_float4(qv[0], qv[1], qv[2], qv[3]) : z4;
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
    const bool y_on = out_wave && !(late && th == 1);
    if (y_on) {
      const int p = 32 * pt + c32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int t = t0 + 32 * th + drow(e, hh);
        zz[e] = t < L && p < p_dim
                    ? load_f32(a.z, a.z_dtype, zo + row(t) * a.z_stride[1] + p * a.z_stride[3])
                    : 0.f;
      }
    }
    if (c + 1 < nchunks) load_chunk(c + 1);
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
    } else if (w >= 4 && w < 7 && !(late && w > 4)) {
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
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = 32 * th + drow(e, hh), t = t0 + r;
        const float y2 = inter[e] * sh.ecs[r] + intra[e] + (skip + sh.qk[r]) * sh.v[r * VS + p];
        if (t < L && p < p_dim)
          store_f32(a.out, a.out_dtype, oo + row(t) * a.out_stride[1] + p * a.out_stride[3],
                    y2 * (zz[e] * sigmoidf(zz[e])));
      }
    } else if (w >= 4 && c + 1 < nchunks) {
      // state update S <- S 2^tot + round_k(v 2^(tot-cs))^T kr (mamba_fused.py:150-152):
      // lane = p, values = n
      const float decay = sh.ecs[kChunk - 1];
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
            *reinterpret_cast<float4*>(&sh.st[(32 * sp + c32) * NS + 32 * sn + 8 * g + 4 * hh]) =
                make_float4(rnd(state[i][4 * g], a.q_dtype), rnd(state[i][4 * g + 1], a.q_dtype),
                            rnd(state[i][4 * g + 2], a.q_dtype), rnd(state[i][4 * g + 3], a.q_dtype));
        }
      }
    }
    __syncthreads();
  }
  // rows past the valid prefix (the same rows in either direction)
  for (int64_t e = static_cast<int64_t>(L) * p_dim + tid; e < static_cast<int64_t>(T) * p_dim; e += kThreads) {
    const int64_t t = e / p_dim, p = e - t * p_dim;
    store_f32(a.out, a.out_dtype, oo + t * a.out_stride[1] + p * a.out_stride[3], 0.f);
  }
}

template <int NT>
int launch_tiles(const tf_mamba_args& a, const GenericVec& vec, bool round, hipStream_t stream) {
  const dim3 grid(static_cast<uint32_t>(a.heads), static_cast<uint32_t>(a.batch));
  if (round)
    hipLaunchKernelGGL((mamba_generic_kernel<NT, true>), grid, dim3(kThreads), 0, stream, a, vec);
  else
    hipLaunchKernelGGL((mamba_generic_kernel<NT, false>), grid, dim3(kThreads), 0, stream, a, vec);
  return launch_status();
}

// Four elements at a time: whole pieces inside the row, aligned at every row.
int vec4(const void* p, int dtype, const int64_t* st, int64_t n) {
  const int es = dtype_size(dtype);
  return n % 4 == 0 && rows_vectorisable(p, st, es, 4 * es);
}

}  // namespace

bool generic_supported(const tf_mamba_args& a) {
  return a.state <= kNMax && a.head_dim <= kPMax;
}

int launch_generic(const tf_mamba_args& a, hipStream_t stream) {
  const GenericVec vec = {vec4(a.q, a.q_dtype, a.q_stride, a.state), vec4(a.k, a.k_dtype, a.k_stride, a.state),
                          vec4(a.v, a.v_dtype, a.v_stride, a.head_dim)};
  const bool round = a.q_dtype != TF_FLOAT32 || a.k_dtype != TF_FLOAT32 || a.v_dtype != TF_FLOAT32;
  if (a.state <= 32) return launch_tiles<1>(a, vec, round, stream);
  if (a.state <= 64) return launch_tiles<2>(a, vec, round, stream);
  if (a.state <= 96) return launch_tiles<3>(a, vec, round, stream);
  return launch_tiles<4>(a, vec, round, stream);
}

}  // namespace tf
