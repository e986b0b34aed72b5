// Rotary + masked softmax attention on the pooled grid of the TriFusion block
// (model.py:84-104, attention.py:8-18): rotary q/k (rounded to bf16), fp32
// softmax over the valid keys j < low_length, [B, T, H D] bf16.
//
// One workgroup takes 32 queries of one (head, batch row); its NW waves share
// the keys, wave w walking the 32-key tiles w, w + NW, ... with its own online
// softmax, and the waves' results meet in LDS at the end. A wave holds
//   scores^T [key][query] = K Q^T     (lane = query, its 16 values = keys)
//   out^T    [dim][query] = V^T P^T   (lane = query, its values = dims)
// so the softmax of a query stays in two lanes (l and l ^ 32), and the scores'
// accumulator registers are the K slots of the second product: P never moves.
// V^T comes from the tile's value rows in LDS by transposing reads.
//
// The second product keeps the probabilities in 32 bits: p is cut into three
// bf16 parts by truncation (8 significant bits each, the remainders exact), so
// p = p1 + p2 + p3 exactly and three bf16 products with fp32 sums stand for
// one 32-bit product. A part that is 0 would turn an infinite value into NaN,
// so a tile that holds a value which is not finite runs the fp32 MFMA instead.
//
// What bounds it: the chain of one key tile (row loads, rotation, four products,
// softmax, six or twelve products), since a bucket of files has few tiles: at
// most 256 workgroups for 16 clips of 26 pooled rows or one file of 451. A kernel
// that formed the dot products on the vector units, four lanes to a query, and
// walked all keys in one wave took 11.8 us at 16 clips of 26 pooled rows, 32.0 at
// 4 of 101 and 123 at one file of 451 (16 heads of 64; calls of a graph, end to
// end); this one takes 5.9, 9.0 and 15.8, with the same distance from a float64
// evaluation. A tenth of that is expf: the hardware exp2 of a rounded product takes
// 5.5, 8.1 and 14.4, and is 20 units of fp32 off where the difference is 50.
#include "mfma_tile.h"

namespace tf {
namespace {

constexpr int kQTile = 32;  // queries per workgroup
constexpr int kKTile = 32;  // keys per step of one wave
constexpr int kMaxWaves = 8;

// Dims 8 c8 .. 8 c8 + 7 of one row rotated (pairs 4 c8 .. 4 c8 + 3): x1 cos -
// x2 sin and x1 sin + x2 cos with separate multiplies and adds, rounded to
// bf16, as the reference's rotary forms them.
__device__ __forceinline__ u32x4 rotate_piece(const u32x4& x, const float4& c, const float4& n) {
#pragma clang fp contract(off)
  const float co[4] = {c.x, c.y, c.z, c.w}, si[4] = {n.x, n.y, n.z, n.w};
  u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = lo_f(x[e]), z = hi_f(x[e]);
    o[e] = pack2(a * co[e] - z * si[e], a * si[e] + z * co[e]);
  }
  return o;
}

// Two probabilities' upper 16 bits as one operand word (the bf16 truncations).
__device__ __forceinline__ uint32_t upper_pair(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
__device__ __forceinline__ float upper(float x) { return __uint_as_float(__float_as_uint(x) & 0xffff0000u); }

// A 16-byte piece of bf16 values holds an infinity or NaN.
__device__ __forceinline__ bool not_finite(const u32x4& x) {
  bool bad = false;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    bad |= (x[e] & 0x7f80u) == 0x7f80u || (x[e] & 0x7f800000u) == 0x7f800000u;
  return bad;
}

template <int D, int NW>
__global__ __launch_bounds__(64 * NW) void attention_kernel(const uint16_t* __restrict__ qkv,
                                                            const float* __restrict__ cs,
                                                            const float* __restrict__ sn,
                                                            const int64_t* __restrict__ low_lengths,
                                                            uint16_t* __restrict__ y, int LT, int H, float scale) {
  constexpr int KS = D / 16;   // k-steps of a score product
  constexpr int DT = D / 32;   // 32-dim tiles of the output
  constexpr int P8 = D / 8;    // 16-byte pieces per row
  constexpr int VL = kKTile * P8 / 64;  // value pieces per lane
  constexpr int OS = D + 4;    // row stride of the merge buffer (16-byte pieces of 8 rows on distinct banks)
  struct Merge {
    float o[NW][kQTile * OS];
    float m[NW][kQTile], l[NW][kQTile];
  };
  struct Tiles {
    uint16_t v[NW][kKTile * 64];
  };
  union Smem {
    Tiles t;
    Merge g;
  };
  __shared__ __align__(16) Smem sh;

  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int c32 = lane & 31, hh = lane >> 5;
  const int h = static_cast<int>(blockIdx.y), b = static_cast<int>(blockIdx.z);
  const int q0 = static_cast<int>(blockIdx.x) * kQTile;
  const int64_t ll = low_lengths[b];
  const int LL = ll < 0 ? 0 : (ll > LT ? LT : static_cast<int>(ll));
  const int64_t width = static_cast<int64_t>(3) * H * D;
  const uint16_t* base = qkv + static_cast<int64_t>(b) * LT * width + static_cast<int64_t>(h) * D;
  const uint16_t* kbase = base + static_cast<int64_t>(H) * D;
  const uint16_t* vbase = base + static_cast<int64_t>(2) * H * D;

  // row `t`, as the MFMA operand whose lane (c32, hh) holds dims 16 s + 8 hh + j
  auto rotated = [&](const uint16_t* rows, int t, u32x4 (&out)[KS]) {
    const uint16_t* row = rows + static_cast<int64_t>(t) * width + 8 * hh;
    const float* ct = cs + static_cast<int64_t>(t) * (D / 2) + 4 * hh;
    const float* st = sn + static_cast<int64_t>(t) * (D / 2) + 4 * hh;
    u32x4 x[KS];
    float4 co[KS], si[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      x[s] = *reinterpret_cast<const u32x4*>(row + 16 * s);
      co[s] = *reinterpret_cast<const float4*>(ct + 8 * s);
      si[s] = *reinterpret_cast<const float4*>(st + 8 * s);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) out[s] = rotate_piece(x[s], co[s], si[s]);
  };

  u32x4 q[KS];
  rotated(base, min(q0 + c32, LT - 1), q);

  f32x16 acc[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) acc[d] = zero16();
  float m = -INFINITY, l = 0.f;
  uint16_t* vt = sh.t.v[w];

  for (int j0 = w * kKTile; j0 < LL; j0 += NW * kKTile) {
    const int nk = min(kKTile, LL - j0);
    // value rows of the tile, whole rows per load; rows past the keys are 0
    u32x4 vv[VL];
    bool bad = false;
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int idx = lane + 64 * i, r = idx / P8, p8 = idx % P8;
      vv[i] = *reinterpret_cast<const u32x4*>(vbase + static_cast<int64_t>(j0 + min(r, nk - 1)) * width + 8 * p8);
      if (r >= nk) vv[i] = u32x4{0u, 0u, 0u, 0u};
    }
    u32x4 k[KS];
    rotated(kbase, j0 + min(c32, nk - 1), k);
    wave_sync();  // the previous tile's values have been read
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int idx = lane + 64 * i, r = idx / P8, p8 = idx % P8;
      bad |= not_finite(vv[i]);
      rb_write16(vt, r, 2 * p8, vv[i]);
    }
    wave_sync();
    f32x16 s = zero16();
#pragma unroll
    for (int i = 0; i < KS; ++i) s = mfma(k[i], q[i], s);
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] *= scale;
    // online softmax of query c32 over keys j0 + drow(e, hh)
    float mx = m;
#pragma unroll
    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, drow(e, hh) < nk ? s[e] : -INFINITY);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float corr = m == mx ? 1.f : expf(m - mx);
    float p[16];
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      p[e] = drow(e, hh) < nk ? expf(s[e] - mx) : 0.f;
      sum += p[e];
    }
    sum += __shfl_xor(sum, 32, 64);
    l = l * corr + sum;
    m = mx;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[d][e] *= corr;
    if (__any(bad)) {
      // fp32 products, keys drow(e, 0) and drow(e, 1) per step
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = drow(e, hh);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          const int col = 32 * d + c32;
          const float x = bf16_to_f32(vt[rb_off(r, col >> 2) + (col & 3)]);
          acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, p[e], acc[d], 0, 0, 0);
        }
      }
    } else {
      u32x4 p1[2], p2[2], p3[2];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float a = p[2 * i], z = p[2 * i + 1];
        const float ra = a - upper(a), rz = z - upper(z);
        p1[i >> 2][i & 3] = upper_pair(a, z);
        p2[i >> 2][i & 3] = upper_pair(ra, rz);
        p3[i >> 2][i & 3] = upper_pair(ra - upper(ra), rz - upper(rz));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          const u32x4 x = tr_operand(vt, d, i, lane);
          acc[d] = mfma(x, p3[i], acc[d]);
          acc[d] = mfma(x, p2[i], acc[d]);
          acc[d] = mfma(x, p1[i], acc[d]);
        }
    }
  }

  if constexpr (NW == 1) {
    const int t = q0 + c32;
    if (t < LT) {
      const float inv = l > 0.f ? 1.0f / l : 0.f;
      uint16_t* dst = y + (static_cast<int64_t>(b) * LT + t) * H * D + static_cast<int64_t>(h) * D;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const u32x2 o = {pack2(acc[d][4 * g] * inv, acc[d][4 * g + 1] * inv),
                           pack2(acc[d][4 * g + 2] * inv, acc[d][4 * g + 3] * inv)};
          *reinterpret_cast<u32x2*>(dst + 32 * d + 8 * g + 4 * hh) = o;
        }
    }
  } else {
    __syncthreads();  // the value tiles are done with: their memory takes the merge
    if (hh == 0) sh.g.m[w][c32] = m, sh.g.l[w][c32] = l;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(&sh.g.o[w][c32 * OS + 32 * d + 8 * g + 4 * hh]) =
            make_float4(acc[d][4 * g], acc[d][4 * g + 1], acc[d][4 * g + 2], acc[d][4 * g + 3]);
    __syncthreads();
    for (int i = static_cast<int>(threadIdx.x); i < kQTile * (D / 4); i += 64 * NW) {
      const int qi = i / (D / 4), d4 = i % (D / 4);
      const int t = q0 + qi;
      if (t >= LT) continue;
      float mm = -INFINITY;
#pragma unroll
      for (int k = 0; k < NW; ++k) mm = fmaxf(mm, sh.g.m[k][qi]);
      float sum = 0.f;
      float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        // a wave without a key has l = 0 and sums of 0
        const float mk = sh.g.m[k][qi], lk = sh.g.l[k][qi];
        const float f = lk == 0.f ? 0.f : (mk == mm ? 1.f : expf(mk - mm));
        const float4 x = *reinterpret_cast<const float4*>(&sh.g.o[k][qi * OS + 4 * d4]);
        sum += f * lk;
        o.x += f * x.x, o.y += f * x.y, o.z += f * x.z, o.w += f * x.w;
      }
      const float inv = sum > 0.f ? 1.0f / sum : 0.f;
      const u32x2 r = {pack2(o.x * inv, o.y * inv), pack2(o.z * inv, o.w * inv)};
      *reinterpret_cast<u32x2*>(y + (static_cast<int64_t>(b) * LT + t) * H * D + static_cast<int64_t>(h) * D + 4 * d4) = r;
    }
  }
}

template <int D>
int launch_attention(const uint16_t* qkv, const float* cs, const float* sn, const int64_t* low, uint16_t* y, int64_t b,
                     int lt, int heads, hipStream_t s) {
  const dim3 grid(static_cast<uint32_t>((lt + kQTile - 1) / kQTile), static_cast<uint32_t>(heads),
                  static_cast<uint32_t>(b));
  const float scale = 1.0f / sqrtf(static_cast<float>(D));
  // a wave per key tile, up to eight
  const int tiles = (lt + kKTile - 1) / kKTile;
#define TF_ATT(NW)                                                                                                \
  hipLaunchKernelGGL((attention_kernel<D, NW>), grid, dim3(64 * NW), 0, s, qkv, cs, sn, low, y, lt, heads, scale); \
  return launch_status();
  if (tiles <= 1) { TF_ATT(1) }
  if (tiles <= 2) { TF_ATT(2) }
  if (tiles <= 4) { TF_ATT(4) }
  TF_ATT(kMaxWaves)
#undef TF_ATT
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace tf

extern "C" int tf_pooled_attention(const void* qkv, const float* cos_t, const float* sin_t,
                                   const int64_t* low_lengths, void* y, int64_t batch, int64_t low_time,
                                   int64_t heads, int64_t head_dim, void* stream) {
  if (!qkv || !cos_t || !sin_t || !low_lengths || !y) return TF_ERR_NULL;
  if (batch < 0 || low_time < 0 || heads < 1 || heads > 65535 || batch > 65535 || batch * low_time > 0x7fffffff)
    return TF_ERR_SHAPE;
  // the tables are read 4 pairs (16 bytes) at a time
  if (!tf::a16(qkv) || !tf::a16(y) || !tf::a16(cos_t) || !tf::a16(sin_t)) return TF_ERR_SHAPE;
  if (batch * low_time == 0) return TF_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t* x = static_cast<const uint16_t*>(qkv);
  uint16_t* out = static_cast<uint16_t*>(y);
  const int lt = static_cast<int>(low_time), nh = static_cast<int>(heads);
  if (head_dim == 32) return tf::launch_attention<32>(x, cos_t, sin_t, low_lengths, out, batch, lt, nh, s);
  if (head_dim == 64) return tf::launch_attention<64>(x, cos_t, sin_t, low_lengths, out, batch, lt, nh, s);
  return TF_ERR_SHAPE;
}
