// Native kernels of the trifusion_amd::fused_mamba operators on ROCm devices:
// operand checks, output and scratch allocation and the launch of the C entry,
// what mamba_fused.py's build_args and launch do for callers that need the
// packed arguments. In Python those took ~20 us per call, twice the GPU time of
// a one-second clip (B1 T100 H16: 26.1 us per plain call, 8.8 us from here).
// The schemas, Meta and CPU kernels are registered in ops.py.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include "trifusion_amd.h"

namespace {

using Opt = std::optional<at::Tensor>;

[[noreturn]] void bad_shape(const std::string& message) { TORCH_CHECK_VALUE(false, "fused_mamba: ", message); }

int32_t dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return TF_FLOAT32;
    case at::kBFloat16: return TF_BFLOAT16;
    case at::kHalf: return TF_FLOAT16;
    default: TORCH_CHECK_TYPE(false, "fused_mamba: unsupported dtype ", t.scalar_type());
  }
}

// Status codes of the C entries as Python exceptions (as _lib.check maps them).
void check_status(int64_t status) {
  switch (status) {
    case TF_OK: return;
    case TF_ERR_SHAPE: TORCH_CHECK_VALUE(false, "fused_mamba: unsupported or inconsistent dimensions");
    case TF_ERR_DTYPE: TORCH_CHECK_TYPE(false, "fused_mamba: unsupported dtype");
    case TF_ERR_STRIDE: TORCH_CHECK_VALUE(false, "fused_mamba: unsupported layout (strides)");
    case TF_ERR_VARIANT: TORCH_CHECK_VALUE(false, "fused_mamba: requested kernel variant cannot run these arguments");
    case TF_ERR_WORKSPACE: TORCH_CHECK_VALUE(false, "fused_mamba: needs more scratch than the library's static area holds");
    case TF_ERR_NULL: TORCH_CHECK(false, "fused_mamba: a required pointer is NULL");
    case TF_ERR_LAUNCH: TORCH_CHECK(false, "fused_mamba: the HIP runtime rejected the kernel launch");
    default: TORCH_CHECK(false, "fused_mamba: status ", status);
  }
}

void float_vector(const char* name, const at::Tensor& t, at::IntArrayRef shape) {
  if (t.sizes() != shape || t.scalar_type() != at::kFloat || !t.is_contiguous())
    bad_shape(std::string(name) + " must be a contiguous float32 tensor of shape " + c10::str(shape));
}

at::Tensor& run(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& adt,
                const at::Tensor& dt, const at::Tensor& trap, const at::Tensor& qb, const at::Tensor& kb,
                const at::Tensor& angles, const at::Tensor& d, const at::Tensor& z, const Opt& lengths,
                std::string_view variant, bool reverse, const Opt& dt_bias, double a_floor, const Opt& q_norm,
                const Opt& k_norm, double norm_eps, at::Tensor& out) {
  const std::pair<const char*, const at::Tensor*> four[] = {
      {"q", &q}, {"k", &k}, {"v", &v}, {"z", &z}, {"angles", &angles}};
  for (const auto& [name, t] : four)
    if (t->dim() != 4) bad_shape(std::string(name) + " must be 4-D, got " + c10::str(t->sizes()));
  const std::pair<const char*, const at::Tensor*> three[] = {{"adt", &adt}, {"dt", &dt}, {"trap", &trap}};
  for (const auto& [name, t] : three)
    if (t->dim() != 3) bad_shape(std::string(name) + " must be [B, H, T], got " + c10::str(t->sizes()));
  const int64_t b = v.size(0), t = v.size(1), h = v.size(2), p = v.size(3);
  const int64_t hq = q.size(2), n = q.size(3), r = angles.size(3);
  if (!(n == 16 || n == 32 || n == 64 || n == 128) || !(p == 32 || p == 64) || r > n / 2)
    bad_shape(c10::str("recurrence requires state in (16, 32, 64, 128), head in (32, 64) and rotary <= state/2 (got state=",
                       n, ", head=", p, ", rotary=", r, ")"));
  const int64_t qk[] = {b, t, hq, n}, vz[] = {b, t, h, p}, ctl[] = {b, h, t};
  if (q.sizes() != at::IntArrayRef(qk) || k.sizes() != at::IntArrayRef(qk))
    bad_shape("q/k must be [B, T, Hq, N] = " + c10::str(at::IntArrayRef(qk)));
  if (hq < 1 || h % hq) bad_shape(c10::str("heads ", h, " must be divisible by q/k heads ", hq));
  if (z.sizes() != at::IntArrayRef(vz)) bad_shape("z must match v");
  for (const auto& [name, x] : three)
    if (x->sizes() != at::IntArrayRef(ctl))
      bad_shape(std::string(name) + " must be [B, H, T] = " + c10::str(at::IntArrayRef(ctl)));
  if (angles.size(0) != b || angles.size(1) != t || angles.size(2) != h) bad_shape("angles must be [B, T, H, R]");
  float_vector("qb", qb, {h, n});
  float_vector("kb", kb, {h, n});
  float_vector("d", d, {h});
  if (out.sizes() != at::IntArrayRef(vz)) bad_shape("out must be [B, T, H, P]");
  if (lengths && (lengths->dim() != 1 || lengths->size(0) != b || lengths->scalar_type() != at::kLong ||
                  !lengths->is_contiguous()))
    bad_shape("lengths must be a contiguous int64 tensor of shape [B]");
  if (dt_bias) {
    float_vector("dt_bias", *dt_bias, {h});
    TORCH_CHECK_TYPE(adt.scalar_type() == dt.scalar_type(), "fused_mamba: raw controls a and ddt must share one dtype");
  }
  if (q_norm.has_value() != k_norm.has_value()) bad_shape("q_norm and k_norm must be given together");
  if (q_norm) {
    float_vector("q_norm", *q_norm, {n});
    float_vector("k_norm", *k_norm, {n});
  }
  const at::Device device = q.device();
  const at::Tensor* all[] = {&q, &k, &v, &adt, &dt, &trap, &qb, &kb, &angles, &d, &z, &out,
                             lengths ? &*lengths : nullptr, dt_bias ? &*dt_bias : nullptr,
                             q_norm ? &*q_norm : nullptr, k_norm ? &*k_norm : nullptr};
  for (const at::Tensor* x : all) {
    if (x == nullptr) continue;
    TORCH_CHECK_VALUE(x->is_cuda(), "fused_mamba: tensors must be on a ROCm (cuda) device, got ", x->device());
    TORCH_CHECK_VALUE(x->device() == device, "fused_mamba: tensors must be on one device (", device, " vs ",
                      x->device(), ")");
  }

  tf_mamba_args a = {};
  a.q = q.const_data_ptr(), a.k = k.const_data_ptr(), a.v = v.const_data_ptr(), a.z = z.const_data_ptr();
  a.adt = adt.const_data_ptr(), a.dt = dt.const_data_ptr(), a.trap = trap.const_data_ptr();
  a.angles = angles.const_data_ptr();
  a.qb = qb.const_data_ptr<float>(), a.kb = kb.const_data_ptr<float>(), a.d = d.const_data_ptr<float>();
  a.out = out.data_ptr();
  a.lengths = lengths ? lengths->const_data_ptr<int64_t>() : nullptr;
  a.q_dtype = dtype_code(q), a.k_dtype = dtype_code(k), a.v_dtype = dtype_code(v), a.z_dtype = dtype_code(z);
  a.adt_dtype = dtype_code(adt), a.dt_dtype = dtype_code(dt), a.trap_dtype = dtype_code(trap);
  a.angles_dtype = dtype_code(angles), a.out_dtype = dtype_code(out);
  if (variant == "auto") a.variant = TF_MAMBA_AUTO;
  else if (variant == "generic") a.variant = TF_MAMBA_GENERIC;
  else if (variant == "mfma") a.variant = TF_MAMBA_MFMA;
  else if (variant == "pipe") a.variant = TF_MAMBA_PIPE;
  else TORCH_CHECK_VALUE(false, "fused_mamba: unknown variant '", variant, "'");
  auto strides = [](int64_t* to, const at::Tensor& x) {
    for (int64_t i = 0; i < x.dim(); ++i) to[i] = x.stride(i);
  };
  strides(a.q_stride, q), strides(a.k_stride, k), strides(a.v_stride, v), strides(a.z_stride, z);
  strides(a.angles_stride, angles), strides(a.out_stride, out);
  strides(a.adt_stride, adt), strides(a.dt_stride, dt), strides(a.trap_stride, trap);
  a.batch = b, a.time = t, a.heads = h, a.qk_heads = hq, a.state = n, a.head_dim = p, a.rotary = r;
  a.dt_bias = dt_bias ? dt_bias->const_data_ptr<float>() : nullptr;
  a.a_floor = static_cast<float>(a_floor);
  a.reverse = reverse ? 1 : 0;
  a.q_norm = q_norm ? q_norm->const_data_ptr<float>() : nullptr;
  a.k_norm = k_norm ? k_norm->const_data_ptr<float>() : nullptr;
  a.norm_eps = static_cast<float>(norm_eps);

  const c10::DeviceGuard guard(device);
  // Long sequences over few (batch, head) units run chunk-parallel on scratch
  // the library sizes; it comes from torch's caching allocator on the current
  // stream (the graph's private pool under capture).
  const int64_t need = tf_fused_mamba_split_size(&a);
  if (need < 0) check_status(-need);
  at::Tensor workspace;
  if (need > 0) {
    workspace = at::empty({need}, at::TensorOptions().dtype(at::kByte).device(device));
    a.workspace = workspace.data_ptr();
    a.workspace_bytes = need;
  }
  check_status(tf_fused_mamba_split(&a, c10::hip::getCurrentHIPStream(device.index()).stream()));
  return out;
}

at::Tensor fused_mamba(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& adt,
                       const at::Tensor& dt, const at::Tensor& trap, const at::Tensor& qb, const at::Tensor& kb,
                       const at::Tensor& angles, const at::Tensor& d, const at::Tensor& z, const Opt& lengths,
                       std::string_view variant, bool reverse, const Opt& dt_bias, double a_floor, const Opt& q_norm,
                       const Opt& k_norm, double norm_eps) {
  at::Tensor out = at::empty_like(v, at::MemoryFormat::Contiguous);
  run(q, k, v, adt, dt, trap, qb, kb, angles, d, z, lengths, variant, reverse, dt_bias, a_floor, q_norm, k_norm,
      norm_eps, out);
  return out;
}

at::Tensor& fused_mamba_out(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& adt,
                            const at::Tensor& dt, const at::Tensor& trap, const at::Tensor& qb, const at::Tensor& kb,
                            const at::Tensor& angles, const at::Tensor& d, const at::Tensor& z, const Opt& lengths,
                            std::string_view variant, bool reverse, const Opt& dt_bias, double a_floor,
                            const Opt& q_norm, const Opt& k_norm, double norm_eps, at::Tensor& out) {
  return run(q, k, v, adt, dt, trap, qb, kb, angles, d, z, lengths, variant, reverse, dt_bias, a_floor, q_norm, k_norm,
             norm_eps, out);
}

}  // namespace

TORCH_LIBRARY_IMPL(trifusion_amd, CUDA, m) {
  m.impl("fused_mamba", &fused_mamba);
  m.impl("fused_mamba.out", &fused_mamba_out);
}
