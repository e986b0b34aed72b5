// Bias-free linear layers whose two output halves gate each other, in one kernel:
//   c = bf16(x w^T)  (x [M, K], w [2 F, K], bf16; fp32 sums)
//   SwiGLU: y = bf16(silu(c[:, :F]) c[:, F:])         (model.py:198, kernels/primitives.py:25-37)
//   GLU:    y = bf16(c[:, :F] sigmoid(c[:, F:]))      (model.py:73)
// The [M, 2 F] product is never written: a workgroup's tile holds 64 columns of
// each half, rounded to bf16 in LDS as the separate product's output is, and the
// gate runs on those values with the separate kernels' arithmetic.
//
// A tile is BM rows by 64 + 64 columns, four waves (WR by 4 / WR) on MFMA 32x32x16.
// Operands go straight from memory into LDS (16 bytes per lane, no registers),
// 64 of K per stage, S stages deep; a stage's rows are 128 bytes and the lane that
// fetches slot p of row r takes piece p ^ (r % 8), so that the operand reads (32
// rows, one piece) fall on distinct banks. Two workgroups share a CU.
//
// What bounds it: the way from L2 into a CU, ~100 KB/us per CU here (26 TB/s over
// the chip), which a tile asks (BM + 128) x 128 bytes of for every 64 of K; so the
// rows of a tile are chosen for the least of that on the busiest CU (see the launch),
// and the 64-row tile (three stages) is for grids that do not fill the chip. SwiGLU
// layer, against the library's product and a gate kernel: 6400 x (2 x 1408) x 512
// 41.2 -> 25.8 us, 1616 x (2 x 2816) x 1024 36.0 -> 27.3, 404 rows 17.5 -> 11.3,
// 28 816 rows 364 -> 334; one row of 64 6.1 -> 2.9. GLU, 1616 x (2 x 1024) x 1024: 13.2
// us against 12.3 for the library's product alone, and the convolution after it 12.4 ->
// 8.0 on rows that are gated once (in the model, beside the attention branch, 20.1
// against 16.5 and 15.8 -> 9.9). Long contractions are not split over workgroups: with
// few tiles and much depth the library is faster, and the callers leave those to it.
#include <algorithm>

#include "mfma_tile.h"

namespace tf {
namespace {

constexpr int kThreads = 256;
constexpr int kHalf = 64;  // columns of each half in a tile
constexpr int kBN = 2 * kHalf;
constexpr int kStep = 64;  // K per stage
constexpr int kCS = kBN + 8;

struct GatedArgs {
  const uint16_t* x;
  const uint16_t* w;
  uint16_t* y;
  int M, F, K;
  int tm, tn;  // tiles
};

// 16 bytes per lane from base + off into LDS at `lds` + 16 lane.
__device__ __forceinline__ void fetch(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(off), "s"(base) : "memory");
}
// Waits until at most N of this wave's fetches are outstanding.
template <int N>
__device__ __forceinline__ void wait_fetches() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Workgroup barrier for LDS filled by fetches: this wave's reads of the stage
// before are done, and what follows stays behind it.
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ float glu(float a, float g) { return a * (1.0f / (1.0f + expf(-g))); }
__device__ __forceinline__ float swiglu(float g, float u) { return g * sigmoidf(g) * u; }

template <int BM, int S, int WR, bool SWIGLU>
__global__ __launch_bounds__(kThreads) void gated_linear_kernel(const GatedArgs P) {
  constexpr int FPW = (BM + kBN) / 8 / 4;  // fetches per wave and stage, 8 rows each
  constexpr int WC = 4 / WR, MT = BM / 32 / WR, NT = 4 / WC;  // 32 x 32 tiles per wave
  constexpr int STAGE = (BM + kBN) * kStep;
  static_assert(S * STAGE >= BM * kCS, "the output tile takes the stages' memory");
  __shared__ __align__(1024) uint16_t lds[S * STAGE];
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int c32 = lane & 31, hh = lane >> 5;
  // Workgroups go to the 8 XCDs in turn; each XCD takes a contiguous range of
  // tiles, ordered down eight row tiles before the next column tile, so the
  // tiles running on it together share rows and columns in its L2.
  const int tiles = P.tm * P.tn, x = static_cast<int>(blockIdx.x & 7), per = tiles / 8, extra = tiles % 8;
  const int id = x * per + min(x, extra) + static_cast<int>(blockIdx.x >> 3);
  const int grp = id / (8 * P.tn), first = 8 * grp, rows = min(P.tm - first, 8), in = id - grp * 8 * P.tn;
  const int m0 = (first + in % rows) * BM, n0 = (in / rows) * kHalf;

  // byte offset of the lane's piece of each fetch: rows m0 .. of x (from row m0,
  // clamped to one that exists), then columns n0 .. of both halves of w
  uint32_t off[FPW];
  const int sub = lane >> 3, piece = 16 * ((lane & 7) ^ sub);
#pragma unroll
  for (int i = 0; i < FPW; ++i) {
    const int r = 8 * (w * FPW + i) + sub;
    const int c = r - BM;
    const uint32_t row = r < BM ? static_cast<uint32_t>(min(r, P.M - 1 - m0))
                                : static_cast<uint32_t>(c < kHalf ? n0 + c : P.F + n0 + c - kHalf);
    off[i] = row * static_cast<uint32_t>(P.K) * 2u + piece;
  }
  const uint32_t lds0 =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint16_t*)lds)) +
      static_cast<uint32_t>(w * FPW * 1024);
  auto issue = [&](int k) {
    const uint32_t to = lds0 + static_cast<uint32_t>((k % S) * (STAGE * 2));
    const uint16_t* xk = P.x + static_cast<int64_t>(m0) * P.K + kStep * k;
    const uint16_t* wk = P.w + kStep * k;
#pragma unroll
    for (int i = 0; i < FPW; ++i) fetch(to + 1024u * i, off[i], 8 * (w * FPW + i) < BM ? xk : wk);
  };
  const int wr = w / WC, wc = w % WC;
  const int xr = (wr * (BM / WR) + c32) * kStep, wro = (BM + wc * (kBN / WC) + c32) * kStep, swz = c32 & 7;
  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = zero16();
  auto multiply = [&](int k) {
    const uint16_t* st = lds + (k % S) * STAGE;
#pragma unroll
    for (int s = 0; s < kStep / 16; ++s) {
      const int p = 8 * ((2 * s + hh) ^ swz);
      u32x4 a[MT], b[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i) a[i] = *reinterpret_cast<const u32x4*>(st + xr + 32 * kStep * i + p);
#pragma unroll
      for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const u32x4*>(st + wro + 32 * kStep * j + p);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma(b[j], a[i], acc[i][j]);
    }
  };
  const int steps = P.K / kStep;
#pragma unroll
  for (int k = 0; k < S - 1; ++k)
    if (k < steps) issue(k);
  int k = 0;
  for (; k + S - 1 < steps; ++k) {
    wait_fetches<(S - 2) * FPW>();  // stage k is here
    stage_barrier();                // ... for every wave, and stage k - 1 has been read
    issue(k + S - 1);
    multiply(k);
  }
  // the last S - 1 stages, nothing left to issue
  if constexpr (S == 3) {
    if (k + 1 < steps) {
      wait_fetches<FPW>();
      stage_barrier();
      multiply(k++);
    }
  }
  wait_fetches<0>();
  stage_barrier();
  multiply(k);
  stage_barrier();  // every wave has read its last stage: its memory takes the output tile

  // acc[i][j]: lane = row, values = columns 8 g + 4 hh + 0..3
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<u32x2*>(lds + (wr * (BM / WR) + 32 * i + c32) * kCS + wc * (kBN / WC) + 32 * j + 8 * g +
                                  4 * hh) =
            u32x2{pack2(acc[i][j][4 * g], acc[i][j][4 * g + 1]), pack2(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3])};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < BM * 8 / kThreads; ++i) {
    const int e = static_cast<int>(threadIdx.x) + kThreads * i, m = e >> 3, n = 8 * (e & 7);
    if (m0 + m < P.M) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(lds + m * kCS + n);
      const u32x4 b = *reinterpret_cast<const u32x4*>(lds + m * kCS + kHalf + n);
      u32x4 o;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        o[q] = SWIGLU ? pack2(swiglu(lo_f(a[q]), lo_f(b[q])), swiglu(hi_f(a[q]), hi_f(b[q])))
                      : pack2(glu(lo_f(a[q]), lo_f(b[q])), glu(hi_f(a[q]), hi_f(b[q])));
      *reinterpret_cast<u32x4*>(P.y + static_cast<int64_t>(m0 + m) * P.F + n0 + n) = o;
    }
  }
}

template <int BM, int S, int WR>
int launch_gated(GatedArgs P, bool swiglu, hipStream_t s) {
  P.tm = (P.M + BM - 1) / BM;
  P.tn = P.F / kHalf;
  const dim3 grid(static_cast<uint32_t>(P.tm) * P.tn), block(kThreads);
  if (swiglu)
    hipLaunchKernelGGL((gated_linear_kernel<BM, S, WR, true>), grid, block, 0, s, P);
  else
    hipLaunchKernelGGL((gated_linear_kernel<BM, S, WR, false>), grid, block, 0, s, P);
  return launch_status();
}

}  // namespace
}  // namespace tf

extern "C" int tf_gated_linear(const void* x, const void* w, void* y, int64_t rows, int64_t features, int64_t depth,
                               int32_t kind, void* stream) {
  if (!x || !w || !y) return TF_ERR_NULL;
  if (kind != 0 && kind != 1) return TF_ERR_VARIANT;
  if (rows < 0 || features < tf::kHalf || features % tf::kHalf || depth < tf::kStep || depth % tf::kStep)
    return TF_ERR_SHAPE;
  // 32-bit byte offsets into w and into a tile's rows of x, 32-bit rows and tiles
  const int64_t most = int64_t(1) << 31;
  if (rows > most - 256 || features >= most || depth >= most / 256 || 2 * features * depth >= most ||
      (rows + 63) / 64 * (features / tf::kHalf) >= most / 8)
    return TF_ERR_SHAPE;
  for (const void* p : {x, w, static_cast<const void*>(y)})
    if (reinterpret_cast<uintptr_t>(p) & 15) return TF_ERR_STRIDE;
  if (rows == 0) return TF_OK;
  tf::GatedArgs P{static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y),
                  static_cast<int>(rows), static_cast<int>(features), static_cast<int>(depth), 0, 0};
  hipStream_t s = static_cast<hipStream_t>(stream);
  // 64-row tiles up to one 128-row tile per CU (256 CUs). K 1024, 1024 features: 128
  // tiles 9.3 us against 12.4 in 128-row tiles, 256 tiles 12.3 against 13.1, 400
  // tiles 21.9 against 18.1; 2816 features: 220 tiles 12.9 against 12.8, 264 tiles
  // 18.6 against 16.7.
  const int64_t cols = features / tf::kHalf;
  const auto tiles = [&](int64_t bm) { return (rows + bm - 1) / bm * cols; };
  if (tiles(128) <= 256) return tf::launch_gated<64, 3, 2>(P, kind == 0, s);
  // Above that the tile whose busiest CU fetches least, which orders what the tiles
  // take (us, 128 / 160 / 192 rows): 1616 x 2816, K 1024 29.5 / 24.9 / 24.7, 1801
  // rows 28.6 / 36.6 / 26.3, 28 816 rows 340 / 356 / 322; 6400 x 1408, K 512 27.6 /
  // 26.8 / 24.7, 1608 rows 11.5 / 10.7 / 11.3.
  const auto cost = [&](int64_t bm) { return (tiles(bm) + 255) / 256 * (bm + tf::kBN); };
  const int64_t best = std::min({cost(128), cost(160), cost(192)});
  if (cost(128) == best) return tf::launch_gated<128, 2, 2>(P, kind == 0, s);
  if (cost(160) == best) return tf::launch_gated<160, 2, 1>(P, kind == 0, s);
  return tf::launch_gated<192, 2, 2>(P, kind == 0, s);
}
