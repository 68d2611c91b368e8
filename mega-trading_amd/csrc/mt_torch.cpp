// GPU kernels and autograd of the mega_trading_amd ops for PyTorch-ROCm.
//
// The op schemas and their fake (shape) implementations are declared from
// Python (mega-trading_amd/attention.py, ops.py, projection.py); this library
// registers what runs for ROCm tensors -- argument preparation, output
// allocation through the caching allocator, the current HIP stream, and one
// call into the C ABI of libmt_attn.so (include/mt_attention.h, mt_ops.h) -- and
// the ops' autograd formulas, whose backwards call the backward ops through the
// dispatcher (so traced graphs hold them too).  In Python both cost more than
// the kernels of a small call: decode attention over 32 caches 27.0 -> 10.5 us a
// call, a prompt of 200 tokens 25.2 -> 18.5, the residual add + norm at 32768 x
// 1024, forward and backward, 210 -> 113 us (its kernels' time).
//
// The layout rules: an attention tensor is used in place when its last stride
// is 1, its outer strides are multiples of 8 elements and its base is 16-byte
// aligned, and is made contiguous otherwise; the row operators take rows in
// place under the same rule.  Errors from the C ABI are raised as RuntimeError with
// mt_last_error()'s message.
#include <ATen/ATen.h>
#include <ATen/FuncTorchTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/library.h>

#include <array>
#include <optional>
#include <tuple>
#include <vector>

#include "../../include/mt_attention.h"
#include "../../include/mt_ops.h"

namespace {

bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

bool kernel_ready(const at::Tensor& t) {
  if (t.dim() == 0 || t.stride(-1) != 1 || !aligned16(t)) return false;
  for (int64_t i = 0; i + 1 < t.dim(); ++i)
    if (t.size(i) > 1 && t.stride(i) % 8) return false;
  return true;
}

at::Tensor ready(const at::Tensor& t) { return kernel_ready(t) ? t : t.contiguous(); }

// (b, h, t, d) element strides; size-1 dims report 0 (their stride is never used)
void put_strides(int64_t* dst, const at::Tensor& t) {
  for (int i = 0; i < 4; ++i) dst[i] = t.size(i) > 1 ? t.stride(i) : 0;
}

int dtype_code(const at::Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return MT_DTYPE_BF16;
  if (t.scalar_type() == at::kHalf) return MT_DTYPE_FP16;
  if (t.scalar_type() == at::kFloat) return MT_DTYPE_FP32;
  TORCH_CHECK(false, "hip attention kernels take bfloat16, float16 or float32 tensors (got ", t.scalar_type(), ")");
}

void check_rc(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", mt_last_error());
}

hipStream_t stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

const void* ptr_or_null(const std::optional<at::Tensor>& t) {
  return t.has_value() && t->defined() ? t->data_ptr() : nullptr;
}

// Forward: (out, lse, q_rot, k_rot).  `out_view`, when defined, is the output
// to write (any kernel-ready strides); q_rot / k_rot are empty without RoPE.
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> forward(
    const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& v_in, const std::optional<at::Tensor>& cos,
    const std::optional<at::Tensor>& sin, double scale, at::Tensor out) {
  TORCH_CHECK(q_in.dim() == 4 && k_in.dim() == 4 && v_in.dim() == 4, "q, k, v must be [B, H, T, D]");
  const c10::DeviceGuard guard(q_in.device());
  const at::Tensor q = ready(q_in), k = ready(k_in), v = ready(v_in);
  const int64_t b = q.size(0), hq = q.size(1), t = q.size(2), d = q.size(3), hkv = k.size(1);
  // the returned output has the query's strides (empty_like of the caller's
  // q, as the reference allocates it); when those are not kernel-ready the
  // kernel writes a contiguous buffer that is copied into it afterwards
  at::Tensor result = out.defined() ? out : at::empty_like(q_in);
  out = ready(result);
  const at::Tensor lse = at::empty({b, hq, t}, q.options().dtype(at::kFloat));
  const bool rope = cos.has_value() && cos->defined();
  at::Tensor q_rot, k_rot;
  if (rope) {
    q_rot = at::empty({b, hq, t, d}, q.options());
    k_rot = at::empty({b, hkv, t, d}, q.options());
  } else {
    q_rot = at::empty({0}, q.options());
    k_rot = at::empty({0}, q.options());
  }
  std::array<int64_t, 16> s{};
  put_strides(s.data(), q);
  put_strides(s.data() + 4, k);
  put_strides(s.data() + 8, v);
  put_strides(s.data() + 12, out);
  check_rc(mt_gqa_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                           rope ? q_rot.data_ptr() : nullptr, rope ? k_rot.data_ptr() : nullptr, int(b), int(hq),
                           int(hkv), int(t), int(d), s.data(), float(scale), dtype_code(q),
                           static_cast<const float*>(ptr_or_null(cos)), static_cast<const float*>(ptr_or_null(sin)),
                           stream_of(q)),
           "mt_gqa_attn_fwd");
  if (!result.is_same(out)) result.copy_(out);
  return {result, lse, q_rot, k_rot};
}

// Backward into the given dq / dk / dv (shapes of q / k / v, kernel-ready strides).
void backward(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& v_in, const at::Tensor& o_in,
              const at::Tensor& lse_in, const at::Tensor& dout_in, const std::optional<at::Tensor>& cos,
              const std::optional<at::Tensor>& sin, double scale, const at::Tensor& dq, const at::Tensor& dk,
              const at::Tensor& dv) {
  const c10::DeviceGuard guard(q_in.device());
  const at::Tensor q = ready(q_in), k = ready(k_in), v = ready(v_in), o = ready(o_in);
  const at::Tensor dout = ready(dout_in.scalar_type() == q.scalar_type() ? dout_in : dout_in.to(q.scalar_type()));
  const at::Tensor lse = lse_in.contiguous();
  const int64_t b = q.size(0), hq = q.size(1), t = q.size(2), d = q.size(3), hkv = k.size(1);
  std::array<int64_t, 32> s{};
  const at::Tensor* ts[8] = {&q, &k, &v, &o, &dout, &dq, &dk, &dv};
  for (int i = 0; i < 8; ++i) put_strides(s.data() + 4 * i, *ts[i]);
  const size_t ws_bytes = mt_gqa_attn_bwd_workspace_size_dtype(int(b), int(hq), int(hkv), int(t), int(d), dtype_code(q));
  const at::Tensor ws = at::empty({int64_t(ws_bytes)}, q.options().dtype(at::kByte));
  check_rc(mt_gqa_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(),
                           dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), ws.data_ptr(), ws_bytes,
                           int(b), int(hq), int(hkv), int(t), int(d), s.data(), float(scale), dtype_code(q),
                           static_cast<const float*>(ptr_or_null(cos)), static_cast<const float*>(ptr_or_null(sin)),
                           stream_of(q)),
           "mt_gqa_attn_bwd");
}

// [B, H, T, D] views of the query, key and value heads of a packed [B, T, (Hq + 2 Hkv) D] tensor
std::array<at::Tensor, 3> packed_views(const at::Tensor& qkv, int64_t hq, int64_t hkv) {
  const int64_t b = qkv.size(0), t = qkv.size(1), d = qkv.size(2) / (hq + 2 * hkv);
  return {qkv.narrow(2, 0, hq * d).view({b, t, hq, d}).transpose(1, 2),
          qkv.narrow(2, hq * d, hkv * d).view({b, t, hkv, d}).transpose(1, 2),
          qkv.narrow(2, (hq + hkv) * d, hkv * d).view({b, t, hkv, d}).transpose(1, 2)};
}

// --- the op kernels (schemas in attention.py) -------------------------------

std::tuple<at::Tensor, at::Tensor> gqa_attn_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                                double scale) {
  auto r = forward(q, k, v, std::nullopt, std::nullopt, scale, at::Tensor());
  return {std::get<0>(r), std::get<1>(r)};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> gqa_rope_attn_fwd(const at::Tensor& q, const at::Tensor& k,
                                                                             const at::Tensor& v, const at::Tensor& cos,
                                                                             const at::Tensor& sin, double scale) {
  return forward(q, k, v, cos, sin, scale, at::Tensor());
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> gqa_attn_bwd(const at::Tensor& q, const at::Tensor& k,
                                                            const at::Tensor& v, const at::Tensor& o,
                                                            const at::Tensor& lse, const at::Tensor& dout,
                                                            const std::optional<at::Tensor>& cos,
                                                            const std::optional<at::Tensor>& sin, double scale) {
  const at::Tensor dq = at::empty(q.sizes(), q.options());
  const at::Tensor dk = at::empty(k.sizes(), k.options());
  const at::Tensor dv = at::empty(v.sizes(), v.options());
  backward(q, k, v, o, lse, dout, cos, sin, scale, dq, dk, dv);
  return {dq, dk, dv};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> gqa_rope_attn_packed_fwd(const at::Tensor& qkv,
                                                                                    const at::Tensor& cos,
                                                                                    const at::Tensor& sin, int64_t hq,
                                                                                    int64_t hkv, double scale) {
  TORCH_CHECK(qkv.dim() == 3, "qkv must be [B, T, (Hq + 2 Hkv) D]");
  const auto views = packed_views(qkv, hq, hkv);
  const int64_t b = qkv.size(0), t = qkv.size(1), d = views[0].size(3);
  const at::Tensor out = at::empty({b, t, hq, d}, qkv.options());
  auto r = forward(views[0], views[1], views[2], cos, sin, scale, out.transpose(1, 2));
  return {out.view({b, t, hq * d}), std::get<1>(r), std::get<2>(r), std::get<3>(r)};
}

at::Tensor gqa_attn_bwd_packed(const at::Tensor& q_rot, const at::Tensor& k_rot, const at::Tensor& qkv,
                               const at::Tensor& out, const at::Tensor& lse, const at::Tensor& dout,
                               const at::Tensor& cos, const at::Tensor& sin, int64_t hq, int64_t hkv, double scale) {
  const auto views = packed_views(qkv, hq, hkv);
  const int64_t b = qkv.size(0), t = qkv.size(1), d = views[2].size(3);
  const at::Tensor dqkv = at::empty(qkv.sizes(), qkv.options());
  const auto grads = packed_views(dqkv, hq, hkv);
  const at::Tensor o = out.view({b, t, hq, d}).transpose(1, 2);
  const at::Tensor dov = dout.reshape({b, t, hq, d}).transpose(1, 2);
  backward(q_rot, k_rot, views[2], o, lse, dov, cos, sin, scale, grads[0], grads[1], grads[2]);
  return dqkv;
}

// --- decode (schemas in attention.py) ----------------------------------------
float* f32_ptr(const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); }
const int* int_ptr_or_null(const std::optional<at::Tensor>& t) { return static_cast<const int*>(ptr_or_null(t)); }

at::Tensor decode_workspace(const at::Tensor& like, int64_t b, int64_t hq, int64_t keys, int64_t d) {
  return at::empty({int64_t(mt_gqa_attn_decode_workspace_size(int(b), int(hq), int(keys), int(d)))},
                   like.options().dtype(at::kByte));
}

// `length` keys, or with length_dev the device's number of them (the launch covers the capacity)
at::Tensor decode(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& v_in, int64_t length,
                  const int* length_dev, double scale) {
  const c10::DeviceGuard guard(q_in.device());
  const at::Tensor q = ready(q_in), k = ready(k_in), v = ready(v_in);
  const int64_t b = q.size(0), hq = q.size(1), d = q.size(3), hkv = k.size(1);
  if (length_dev) length = k.size(2);
  const at::Tensor out = at::empty({b, hq, 1, d}, q.options());
  const at::Tensor ws = decode_workspace(q, b, hq, length, d);
  std::array<int64_t, 16> s{};
  put_strides(s.data(), q);
  put_strides(s.data() + 4, k);
  put_strides(s.data() + 8, v);
  put_strides(s.data() + 12, out);
  if (length_dev)
    check_rc(mt_gqa_attn_decode_dev(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), int(b), int(hq), int(hkv),
                                    int(length), length_dev, int(d), s.data(), float(scale), dtype_code(q),
                                    ws.data_ptr(), size_t(ws.numel()), stream_of(q)),
             "mt_gqa_attn_decode_dev");
  else
    check_rc(mt_gqa_attn_decode(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), int(b), int(hq), int(hkv),
                                int(length), int(d), s.data(), float(scale), dtype_code(q), ws.data_ptr(),
                                size_t(ws.numel()), stream_of(q)),
             "mt_gqa_attn_decode");
  return out;
}

at::Tensor gqa_attn_decode(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t length, double scale) {
  return decode(q, k, v, length, nullptr, scale);
}

at::Tensor gqa_attn_decode_dev(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& length,
                               double scale) {
  return decode(q, k, v, 0, static_cast<const int*>(length.data_ptr()), scale);
}

at::Tensor decode_rope_append(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& cos,
                              const at::Tensor& sin, int64_t pos, const std::optional<at::Tensor>& pos_dev,
                              const at::Tensor& k_cache, const at::Tensor& v_cache) {
  const c10::DeviceGuard guard(q.device());
  const int64_t b = q.size(0), hq = q.size(1), d = q.size(3), hkv = k.size(1);
  const at::Tensor out = at::empty({b, hq, 1, d}, k_cache.options());
  const at::Tensor cs = cos.contiguous(), sn = sin.contiguous();
  const int64_t rows = std::min(cs.numel(), sn.numel()) / (d / 2);
  const int64_t ins[6] = {q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0), v.stride(1)};
  const int64_t cst[6] = {k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
                          v_cache.stride(0), v_cache.stride(1), v_cache.stride(2)};
  check_rc(mt_decode_rope_append(q.data_ptr(), k.data_ptr(), v.data_ptr(), ins, f32_ptr(cs), f32_ptr(sn), int(rows),
                                 int(pos), int_ptr_or_null(pos_dev), out.data_ptr(), k_cache.data_ptr(),
                                 v_cache.data_ptr(), cst, int(k_cache.size(2)), int(b), int(hq), int(hkv), int(d),
                                 dtype_code(q), dtype_code(k_cache), stream_of(q)),
           "mt_decode_rope_append");
  return out;
}

at::Tensor gqa_attn_decode_append(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& cos,
                                  const at::Tensor& sin, int64_t pos, const std::optional<at::Tensor>& pos_dev,
                                  int64_t length, const std::optional<at::Tensor>& length_dev,
                                  const at::Tensor& k_cache, const at::Tensor& v_cache, double scale) {
  const c10::DeviceGuard guard(q.device());
  // rows that cannot be loaded 16 bytes at a time: the two launches it stands for
  for (const at::Tensor* t : {&q, &k, &v, &cos, &sin, &k_cache, &v_cache})
    if (!aligned16(*t)) {
      const at::Tensor q_rot = decode_rope_append(q, k, v, cos, sin, pos, pos_dev, k_cache, v_cache);
      return decode(q_rot, k_cache, v_cache, length, int_ptr_or_null(length_dev), scale);
    }
  const int64_t b = q.size(0), hq = q.size(1), d = q.size(3), hkv = k_cache.size(1), cap = k_cache.size(2);
  const at::Tensor out = at::empty({b, hq, 1, d}, k_cache.options());
  const int* len = int_ptr_or_null(length_dev);
  const at::Tensor ws = decode_workspace(q, b, hq, len ? cap : std::max(length, pos + 1), d);
  const int64_t ins[6] = {q.stride(0), q.stride(1), k.stride(0), k.stride(1), v.stride(0), v.stride(1)};
  const int64_t cst[6] = {k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
                          v_cache.stride(0), v_cache.stride(1), v_cache.stride(2)};
  check_rc(mt_gqa_attn_decode_append(q.data_ptr(), k.data_ptr(), v.data_ptr(), ins, f32_ptr(cos), f32_ptr(sin),
                                     int(cos.numel() / (d / 2)), int(pos), int_ptr_or_null(pos_dev), k_cache.data_ptr(),
                                     v_cache.data_ptr(), cst, int(cap), int(length), len, out.data_ptr(), int(b),
                                     int(hq), int(hkv), int(d), float(scale), dtype_code(q), dtype_code(k_cache),
                                     ws.data_ptr(), size_t(ws.numel()), stream_of(q)),
           "mt_gqa_attn_decode_append");
  return out;
}

// --- row operators (schemas in ops.py, projection.py) ------------------------
at::Tensor flat(const at::Tensor& x) {
  const at::Tensor c = x.contiguous();
  return aligned16(c) ? c : c.clone();
}

// x's rows of the last dim, in place where the kernels can read them
struct Rows {
  at::Tensor t;
  int64_t rows, dim, stride;
};
Rows rows_of(const at::Tensor& x) {
  const int64_t d = x.size(-1), n = d ? x.numel() / d : 0;
  if (x.is_contiguous() && aligned16(x) && d % 8 == 0) return {x, n, d, d};
  at::Tensor r = x.reshape({-1, d});
  if (r.stride(1) != 1 || !aligned16(r) || (r.size(0) > 1 && r.stride(0) % 8)) r = flat(r);
  return {r, r.size(0), d, r.size(0) > 1 ? r.stride(0) : d};
}

// the weight as the kernels take it: x's dtype or fp32, contiguous, aligned
at::Tensor weight_for(const at::Tensor& w, const at::Tensor& x) {
  return flat(w.scalar_type() != x.scalar_type() && w.scalar_type() != at::kFloat ? w.to(at::kFloat) : w);
}

at::ScalarType act_type(int64_t code) {
  TORCH_CHECK(code >= 0 && code <= 2, "dtype code ", code, " unsupported");
  return code == MT_DTYPE_BF16 ? at::kBFloat16 : code == MT_DTYPE_FP16 ? at::kHalf : at::kFloat;
}

std::tuple<at::Tensor, at::Tensor> rms_norm_fwd(const at::Tensor& x, const at::Tensor& weight, double eps) {
  const c10::DeviceGuard guard(x.device());
  const Rows r = rows_of(x);
  const at::Tensor w = weight_for(weight, x);
  const at::Tensor y = at::empty(x.sizes(), x.options());
  const at::Tensor rstd = at::empty({r.rows}, x.options().dtype(at::kFloat));
  check_rc(mt_rms_norm_fwd(r.t.data_ptr(), r.stride, w.data_ptr(), y.data_ptr(), f32_ptr(rstd), r.rows, int(r.dim),
                           float(eps), dtype_code(x), dtype_code(w), stream_of(x)),
           "mt_rms_norm_fwd");
  return {y, rstd};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> add_rms_norm_fwd(const at::Tensor& x, const at::Tensor& residual,
                                                                const at::Tensor& weight, double eps) {
  const c10::DeviceGuard guard(x.device());
  const Rows r = rows_of(x), s = rows_of(residual);
  const at::Tensor w = weight_for(weight, x);
  const at::Tensor sum = at::empty(x.sizes(), x.options()), y = at::empty(x.sizes(), x.options());
  const at::Tensor rstd = at::empty({r.rows}, x.options().dtype(at::kFloat));
  check_rc(mt_add_rms_norm_fwd(r.t.data_ptr(), r.stride, s.t.data_ptr(), s.stride, w.data_ptr(), sum.data_ptr(),
                               y.data_ptr(), f32_ptr(rstd), r.rows, int(r.dim), float(eps), dtype_code(x),
                               dtype_code(w), stream_of(x)),
           "mt_add_rms_norm_fwd");
  return {sum, y, rstd};
}

std::tuple<at::Tensor, at::Tensor> norm_bwd(const at::Tensor& s_in, const at::Tensor& weight, const at::Tensor& rstd,
                                            const at::Tensor& dy_in, const at::Tensor* dres) {
  const c10::DeviceGuard guard(s_in.device());
  const at::Tensor s = flat(s_in), dy = flat(dy_in.to(s.scalar_type())), w = weight_for(weight, s);
  const int64_t d = s.size(-1), rows = s.numel() / std::max<int64_t>(d, 1);
  const at::Tensor dx = at::empty(s.sizes(), s.options());
  const at::Tensor dw = at::empty({d}, w.options());
  const size_t need = std::max<size_t>(mt_rms_norm_bwd_workspace_size(rows, int(d)), 256);
  const at::Tensor ws = at::empty({int64_t(need)}, s.options().dtype(at::kByte));
  if (dres) {
    const at::Tensor dr = flat(dres->to(s.scalar_type()));
    check_rc(mt_add_rms_norm_bwd(s.data_ptr(), w.data_ptr(), f32_ptr(rstd), dr.data_ptr(), dy.data_ptr(), dx.data_ptr(),
                                 dw.data_ptr(), ws.data_ptr(), need, rows, int(d), dtype_code(s), dtype_code(w),
                                 stream_of(s)),
             "mt_add_rms_norm_bwd");
  } else {
    check_rc(mt_rms_norm_bwd(s.data_ptr(), w.data_ptr(), f32_ptr(rstd), dy.data_ptr(), dx.data_ptr(), dw.data_ptr(),
                             ws.data_ptr(), need, rows, int(d), dtype_code(s), dtype_code(w), stream_of(s)),
             "mt_rms_norm_bwd");
  }
  return {dx, dw.to(weight.scalar_type())};
}

std::tuple<at::Tensor, at::Tensor> rms_norm_bwd(const at::Tensor& x, const at::Tensor& weight, const at::Tensor& rstd,
                                                const at::Tensor& dy) {
  return norm_bwd(x, weight, rstd, dy, nullptr);
}

std::tuple<at::Tensor, at::Tensor> add_rms_norm_bwd(const at::Tensor& sum, const at::Tensor& weight,
                                                    const at::Tensor& rstd, const at::Tensor& dsum,
                                                    const at::Tensor& dy) {
  return norm_bwd(sum, weight, rstd, dy, &dsum);
}

std::tuple<at::Tensor, at::Tensor> rms_norm_fwd_mixed(const at::Tensor& x, const at::Tensor& weight, double eps,
                                                      int64_t act) {
  const c10::DeviceGuard guard(x.device());
  const Rows r = rows_of(x);
  const at::Tensor w = flat(weight);
  const at::Tensor y = at::empty(x.sizes(), x.options().dtype(act_type(act)));
  const at::Tensor rstd = at::empty({r.rows}, x.options().dtype(at::kFloat));
  check_rc(mt_rms_norm_fwd_mixed(r.t.data_ptr(), r.stride, w.data_ptr(), y.data_ptr(), f32_ptr(rstd), r.rows,
                                 int(r.dim), float(eps), int(act), dtype_code(w), stream_of(x)),
           "mt_rms_norm_fwd_mixed");
  return {y, rstd};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> add_rms_norm_fwd_mixed(const at::Tensor& x, const at::Tensor& residual,
                                                                      const at::Tensor& weight, double eps) {
  const c10::DeviceGuard guard(x.device());
  const Rows r = rows_of(x), s = rows_of(residual);
  const at::Tensor w = flat(weight);
  const at::Tensor sum = at::empty(x.sizes(), x.options().dtype(at::kFloat)), y = at::empty(x.sizes(), x.options());
  const at::Tensor rstd = at::empty({r.rows}, x.options().dtype(at::kFloat));
  check_rc(mt_add_rms_norm_fwd_mixed(r.t.data_ptr(), r.stride, s.t.data_ptr(), s.stride, w.data_ptr(), sum.data_ptr(),
                                     y.data_ptr(), f32_ptr(rstd), r.rows, int(r.dim), float(eps), dtype_code(x),
                                     dtype_code(w), stream_of(x)),
           "mt_add_rms_norm_fwd_mixed");
  return {sum, y, rstd};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> rms_norm_bwd_mixed(const at::Tensor& s_in, const at::Tensor& weight,
                                                                  const at::Tensor& rstd,
                                                                  const std::optional<at::Tensor>& dsum,
                                                                  const at::Tensor& dy_in, int64_t act, bool want16) {
  const c10::DeviceGuard guard(s_in.device());
  const at::Tensor s = flat(s_in), dy = flat(dy_in.to(act_type(act))), w = flat(weight);
  const at::Tensor dr = dsum.has_value() && dsum->defined() ? flat(dsum->to(at::kFloat)) : at::Tensor();
  const int64_t d = s.size(-1), rows = s.numel() / std::max<int64_t>(d, 1);
  const at::Tensor ds = at::empty(s.sizes(), s.options().dtype(at::kFloat));
  const at::Tensor ds16 = want16 ? at::empty(s.sizes(), s.options().dtype(act_type(act)))
                                 : at::empty({0}, s.options().dtype(act_type(act)));
  const at::Tensor dw = at::empty({d}, s.options().dtype(at::kFloat));
  const size_t need = std::max<size_t>(mt_rms_norm_bwd_workspace_size(rows, int(d)), 256);
  const at::Tensor ws = at::empty({int64_t(need)}, s.options().dtype(at::kByte));
  check_rc(mt_rms_norm_bwd_mixed(s.data_ptr(), w.data_ptr(), f32_ptr(rstd), dr.defined() ? dr.data_ptr() : nullptr,
                                 dy.data_ptr(), ds.data_ptr(), want16 ? ds16.data_ptr() : nullptr, dw.data_ptr(),
                                 ws.data_ptr(), need, rows, int(d), int(act), dtype_code(w), stream_of(s)),
           "mt_rms_norm_bwd_mixed");
  return {ds, ds16, dw};
}

at::Tensor swiglu_fwd(const at::Tensor& gate, const at::Tensor& up) {
  const c10::DeviceGuard guard(gate.device());
  const at::Tensor g = flat(gate), u = flat(up), out = at::empty(gate.sizes(), gate.options());
  check_rc(mt_swiglu_fwd(g.data_ptr(), u.data_ptr(), out.data_ptr(), g.numel(), dtype_code(g), stream_of(gate)),
           "mt_swiglu_fwd");
  return out;
}

std::tuple<at::Tensor, at::Tensor> swiglu_bwd(const at::Tensor& gate, const at::Tensor& up, const at::Tensor& dout) {
  const c10::DeviceGuard guard(gate.device());
  const at::Tensor g = flat(gate), u = flat(up), dy = flat(dout.to(gate.scalar_type()));
  const at::Tensor dg = at::empty(gate.sizes(), gate.options()), du = at::empty(gate.sizes(), gate.options());
  check_rc(mt_swiglu_bwd(g.data_ptr(), u.data_ptr(), dy.data_ptr(), dg.data_ptr(), du.data_ptr(), g.numel(),
                         dtype_code(g), stream_of(gate)),
           "mt_swiglu_bwd");
  return {dg, du};
}

at::Tensor swiglu_packed_fwd(const at::Tensor& gate_up) {
  const c10::DeviceGuard guard(gate_up.device());
  const at::Tensor gu = flat(gate_up);
  const int64_t cols = gu.size(-1) / 2, rows = gu.numel() / std::max<int64_t>(2 * cols, 1);
  std::vector<int64_t> shape = gu.sizes().vec();
  shape.back() = cols;
  const at::Tensor out = at::empty(shape, gu.options());
  check_rc(mt_swiglu_packed_fwd(gu.data_ptr(), out.data_ptr(), rows, cols, dtype_code(gu), stream_of(gu)),
           "mt_swiglu_packed_fwd");
  return out;
}

at::Tensor swiglu_packed_bwd(const at::Tensor& gate_up, const at::Tensor& dout) {
  const c10::DeviceGuard guard(gate_up.device());
  const at::Tensor gu = flat(gate_up), dy = flat(dout.to(gate_up.scalar_type()));
  const int64_t cols = gu.size(-1) / 2, rows = gu.numel() / std::max<int64_t>(2 * cols, 1);
  const at::Tensor dgu = at::empty(gu.sizes(), gu.options());
  check_rc(mt_swiglu_packed_bwd(gu.data_ptr(), dy.data_ptr(), dgu.data_ptr(), rows, cols, dtype_code(gu),
                                stream_of(gu)),
           "mt_swiglu_packed_bwd");
  return dgu;
}

// Outputs take the inputs' layout (empty_like); `inverse` rotates by -theta.
std::tuple<at::Tensor, at::Tensor> rope_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& cos,
                                            const at::Tensor& sin, bool inverse) {
  const c10::DeviceGuard guard(q.device());
  const at::Tensor qo = at::empty_like(q), ko = at::empty_like(k);
  int64_t s[16];
  const at::Tensor* ts[4] = {&q, &qo, &k, &ko};
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) s[4 * i + j] = ts[i]->stride(j);
  check_rc(mt_apply_rope(q.data_ptr(), k.data_ptr(), qo.data_ptr(), ko.data_ptr(), int(q.size(0)), int(q.size(1)),
                         int(k.size(1)), int(q.size(2)), int(q.size(3)), s, f32_ptr(cos), f32_ptr(sin), cos.stride(0),
                         int(cos.size(0)), inverse ? 1 : 0, dtype_code(q), stream_of(q)),
           "mt_apply_rope");
  return {qo, ko};
}

at::Tensor topk_sample(const at::Tensor& logits, const at::Tensor& noise, int64_t k) {
  const c10::DeviceGuard guard(logits.device());
  const at::Tensor x = logits.stride(1) == 1 ? logits : logits.contiguous();
  const at::Tensor e = noise.stride(1) == 1 ? noise : noise.contiguous();
  const at::Tensor out = at::empty({x.size(0), 1}, x.options().dtype(at::kLong));
  check_rc(mt_topk_sample(x.data_ptr(), x.stride(0), e.data_ptr(), e.stride(0), int(x.size(0)), int(x.size(1)), int(k),
                          static_cast<int64_t*>(out.data_ptr()), dtype_code(x), stream_of(x)),
           "mt_topk_sample");
  return out;
}

at::Tensor linear_rows(const at::Tensor& x, at::TensorList weights) {
  const c10::DeviceGuard guard(x.device());
  std::vector<const void*> ptrs;
  std::vector<int> outs;
  std::vector<int64_t> lds;
  int64_t cols = 0;
  for (const at::Tensor& w : weights) {
    ptrs.push_back(w.data_ptr());
    outs.push_back(int(w.size(0)));
    lds.push_back(w.stride(0));
    cols += w.size(0);
  }
  const at::Tensor y = at::empty({x.size(0), cols}, x.options().dtype(at::kFloat));
  check_rc(mt_linear_rows(x.data_ptr(), x.stride(0), ptrs.data(), outs.data(), lds.data(), int(ptrs.size()),
                          y.data_ptr(), y.stride(0), int(x.size(0)), int(x.size(1)), dtype_code(x), stream_of(x)),
           "mt_linear_rows");
  return y;
}

at::Tensor linear_rows_gate(const at::Tensor& x, const at::Tensor& w_gate, const at::Tensor& w_up) {
  const c10::DeviceGuard guard(x.device());
  const at::Tensor y = at::empty({x.size(0), w_gate.size(0)}, x.options().dtype(at::kFloat));
  check_rc(mt_linear_rows_gate(x.data_ptr(), x.stride(0), w_gate.data_ptr(), w_up.data_ptr(), w_gate.stride(0),
                               w_up.stride(0), y.data_ptr(), y.stride(0), int(x.size(0)), int(x.size(1)),
                               int(w_gate.size(0)), dtype_code(x), stream_of(x)),
           "mt_linear_rows_gate");
  return y;
}

// --- loss head (schemas in ops.py; the op itself, which runs library GEMMs, is Python) ---
at::Tensor ce_count(const at::Tensor& labels, int64_t ignore_index) {
  const c10::DeviceGuard guard(labels.device());
  const at::Tensor n = at::empty({}, labels.options());
  check_rc(mt_cross_entropy_count(static_cast<const int64_t*>(labels.data_ptr()), labels.numel(), ignore_index,
                                  static_cast<int64_t*>(n.data_ptr()), stream_of(labels)),
           "mt_cross_entropy_count");
  return n;
}

at::Tensor ce_sum(const at::Tensor& loss_rows) {
  const c10::DeviceGuard guard(loss_rows.device());
  const at::Tensor s = at::empty({}, loss_rows.options());
  check_rc(mt_cross_entropy_sum(f32_ptr(loss_rows), loss_rows.numel(), f32_ptr(s), stream_of(loss_rows)),
           "mt_cross_entropy_sum");
  return s;
}

std::tuple<at::Tensor, at::Tensor> scale_pair(const at::Tensor& a_in, const at::Tensor& b_in, const at::Tensor& scale) {
  const c10::DeviceGuard guard(a_in.device());
  const at::Tensor a = flat(a_in), b = flat(b_in);
  const at::Tensor s = scale.to(at::kFloat).contiguous();
  const at::Tensor ao = at::empty(a.sizes(), a.options()), bo = at::empty(b.sizes(), b.options());
  check_rc(mt_scale_pair(a.data_ptr(), ao.data_ptr(), a.numel(), dtype_code(a), b.data_ptr(), bo.data_ptr(), b.numel(),
                         dtype_code(b), f32_ptr(s), stream_of(a)),
           "mt_scale_pair");
  return {ao, bo};
}

// --- autograd ----------------------------------------------------------------
// Forwards run the op below autograd; backwards call the backward ops through
// the dispatcher.  Gradients that arrive undefined stay undefined except where
// noted.  A forward-mode tangent on a recorded call is refused.
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using Opt = std::optional<at::Tensor>;

template <class Sig>
c10::TypedOperatorHandle<Sig> op_handle(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}
#define MT_OP(name) op_handle<decltype(name)>("mega_trading_amd::" #name)

Opt opt(const at::Tensor& t) { return t.defined() ? Opt(t) : Opt(); }

struct AttnFn : torch::autograd::Function<AttnFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                               double scale) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(gqa_attn_fwd);
    auto [out, lse] = op.call(q, k, v, scale);
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["scale"] = scale;
    ctx->mark_non_differentiable({lse});
    ctx->set_materialize_grads(false);
    return {out, lse};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(4);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(gqa_attn_bwd);
    auto [dq, dk, dv] = op.call(s[0], s[1], s[2], s[3], s[4], g[0], Opt(), Opt(), ctx->saved_data["scale"].toDouble());
    return {dq, dk, dv, at::Tensor()};
  }
};

struct RopeAttnFn : torch::autograd::Function<RopeAttnFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                               const at::Tensor& cos, const at::Tensor& sin, double scale) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(gqa_rope_attn_fwd);
    auto [out, lse, q_rot, k_rot] = op.call(q, k, v, cos, sin, scale);
    ctx->save_for_backward({q_rot, k_rot, v, out, lse, cos, sin});
    ctx->saved_data["scale"] = scale;
    ctx->mark_non_differentiable({lse, q_rot, k_rot});
    ctx->set_materialize_grads(false);
    return {out, lse, q_rot, k_rot};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(6);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(gqa_attn_bwd);
    auto [dq, dk, dv] = op.call(s[0], s[1], s[2], s[3], s[4], g[0], Opt(s[5]), Opt(s[6]),
                                ctx->saved_data["scale"].toDouble());
    return {dq, dk, dv, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

struct PackedAttnFn : torch::autograd::Function<PackedAttnFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& qkv, const at::Tensor& cos,
                               const at::Tensor& sin, int64_t hq, int64_t hkv, double scale) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(gqa_rope_attn_packed_fwd);
    auto [out, lse, q_rot, k_rot] = op.call(qkv, cos, sin, hq, hkv, scale);
    ctx->save_for_backward({q_rot, k_rot, qkv, out, lse, cos, sin});
    ctx->saved_data["hq"] = hq;
    ctx->saved_data["hkv"] = hkv;
    ctx->saved_data["scale"] = scale;
    ctx->mark_non_differentiable({lse, q_rot, k_rot});
    ctx->set_materialize_grads(false);
    return {out, lse, q_rot, k_rot};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(6);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(gqa_attn_bwd_packed);
    variable_list r(6);
    r[0] = op.call(s[0], s[1], s[2], s[3], s[4], g[0], s[5], s[6], ctx->saved_data["hq"].toInt(),
                   ctx->saved_data["hkv"].toInt(), ctx->saved_data["scale"].toDouble());
    return r;
  }
};

struct RmsFn : torch::autograd::Function<RmsFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& w, double eps) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(rms_norm_fwd);
    auto [y, rstd] = op.call(x, w, eps);
    ctx->save_for_backward({x, w, rstd});
    ctx->mark_non_differentiable({rstd});
    ctx->set_materialize_grads(false);
    return {y, rstd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(3);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(rms_norm_bwd);
    auto [dx, dw] = op.call(s[0], s[1], s[2], g[0]);
    return {dx, dw, at::Tensor()};
  }
};

struct AddRmsFn : torch::autograd::Function<AddRmsFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& r, const at::Tensor& w,
                               double eps) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(add_rms_norm_fwd);
    auto [sum, y, rstd] = op.call(x, r, w, eps);
    ctx->save_for_backward({sum, w, rstd});
    ctx->mark_non_differentiable({rstd});
    ctx->set_materialize_grads(false);
    return {sum, y, rstd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined() && !g[1].defined()) return variable_list(4);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(add_rms_norm_bwd);
    auto [dx, dw] = op.call(s[0], s[1], s[2], g[0].defined() ? g[0] : at::zeros_like(s[0]),
                            g[1].defined() ? g[1] : at::zeros_like(s[0]));
    // hidden and residual enter the add symmetrically: the same gradient for both (triton_ops.py:288-291)
    return {dx, dx, dw, at::Tensor()};
  }
};

struct RmsMixedFn : torch::autograd::Function<RmsMixedFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& w, double eps,
                               int64_t act) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(rms_norm_fwd_mixed);
    auto [y, rstd] = op.call(x, w, eps, act);
    ctx->save_for_backward({x, w, rstd});
    ctx->saved_data["act"] = act;
    ctx->set_materialize_grads(false);
    return {y, rstd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(4);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(rms_norm_bwd_mixed);
    auto [dx, ds16, dw] = op.call(s[0], s[1], s[2], Opt(), g[0], ctx->saved_data["act"].toInt(), false);
    return {dx, dw, at::Tensor(), at::Tensor()};
  }
};

struct AddRmsMixedFn : torch::autograd::Function<AddRmsMixedFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& r, const at::Tensor& w,
                               double eps) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(add_rms_norm_fwd_mixed);
    auto [sum, y, rstd] = op.call(x, r, w, eps);
    ctx->save_for_backward({sum, w, rstd});
    ctx->saved_data["act"] = int64_t(dtype_code(x));
    ctx->set_materialize_grads(false);
    return {sum, y, rstd};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const int64_t act = ctx->saved_data["act"].toInt();
    if (!g[1].defined()) {
      if (!g[0].defined()) return variable_list(4);
      // only the sum is used: both inputs get its gradient (in their dtypes)
      return {g[0].to(act_type(act)), g[0], at::Tensor(), at::Tensor()};
    }
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(rms_norm_bwd_mixed);
    auto [ds, ds16, dw] = op.call(s[0], s[1], s[2], opt(g[0]), g[1], act, true);
    return {ds16, ds, dw, at::Tensor()};
  }
};

struct SwigluFn : torch::autograd::Function<SwigluFn> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& gate, const at::Tensor& up) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(swiglu_fwd);
    ctx->save_for_backward({gate, up});
    ctx->set_materialize_grads(false);
    return op.call(gate, up);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(2);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(swiglu_bwd);
    auto [dg, du] = op.call(s[0], s[1], g[0]);
    return {dg, du};
  }
};

struct SwigluPackedFn : torch::autograd::Function<SwigluPackedFn> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& gate_up) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(swiglu_packed_fwd);
    ctx->save_for_backward({gate_up});
    ctx->set_materialize_grads(false);
    return op.call(gate_up);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return variable_list(1);
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(swiglu_packed_bwd);
    return {op.call(s[0], g[0])};
  }
};

// A rotation's gradient is the opposite rotation; an unused output's gradient
// arrives as zeros (gradients are materialized).
struct RopeFn : torch::autograd::Function<RopeFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& cos,
                               const at::Tensor& sin, bool inverse) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = MT_OP(rope_fwd);
    auto [qo, ko] = op.call(q, k, cos, sin, inverse);
    ctx->save_for_backward({cos, sin});
    ctx->saved_data["inverse"] = inverse;
    return {qo, ko};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    static const auto op = MT_OP(rope_fwd);
    auto [gq, gk] = op.call(g[0], g[1], s[0], s[1], !ctx->saved_data["inverse"].toBool());
    return {gq, gk, at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

// The gradients are computed in the forward and scaled here; they are linear in
// the incoming one, and differentiable in it.
using CeSig = std::tuple<at::Tensor, at::Tensor, at::Tensor>(const at::Tensor&, const at::Tensor&, const at::Tensor&,
                                                             int64_t, int64_t, bool);
struct LinearCeFn : torch::autograd::Function<LinearCeFn> {
  static variable_list forward(AutogradContext* ctx, const at::Tensor& hidden, const at::Tensor& weight,
                               const at::Tensor& labels, int64_t ignore_index, int64_t compute, bool need_grad) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = op_handle<CeSig>("mega_trading_amd::fused_linear_ce");
    auto [loss, gh, gw] = op.call(hidden, weight, labels, ignore_index, compute, need_grad);
    ctx->save_for_backward({gh, gw});
    ctx->saved_data["need_grad"] = need_grad;
    ctx->mark_non_differentiable({gh, gw});
    ctx->set_materialize_grads(false);
    return {loss, gh, gw};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined() || !ctx->saved_data["need_grad"].toBool()) return variable_list(6);
    const auto s = ctx->get_saved_variables();
    variable_list r(6);
    if ((c10::GradMode::is_enabled() && g[0].requires_grad()) || g[0]._fw_grad(0).defined()) {
      // products that a derivative with respect to the incoming gradient goes through
      r[0] = s[0] * g[0].to(s[0].scalar_type());
      r[1] = s[1] * g[0].to(s[1].scalar_type());
      return r;
    }
    static const auto op = MT_OP(scale_pair);
    std::tie(r[0], r[1]) = op.call(s[0], s[1], g[0]);
    return r;
  }
};

// Whether a call records a gradient: without one the op runs below autograd
// directly.  RoPE tables that require one record the call too (and get none).
template <class... T>
bool records(const T&... ts) {
  return c10::GradMode::is_enabled() && (ts.requires_grad() || ...);
}
#define MT_BELOW(name, ...)                      \
  do {                                           \
    at::AutoDispatchBelowADInplaceOrView below;  \
    static const auto op = MT_OP(name);          \
    return op.call(__VA_ARGS__);                 \
  } while (0)

std::tuple<at::Tensor, at::Tensor> gqa_attn_fwd_ad(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                                   double scale) {
  if (!records(q, k, v)) MT_BELOW(gqa_attn_fwd, q, k, v, scale);
  auto r = AttnFn::apply(q, k, v, scale);
  return {r[0], r[1]};
}
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> gqa_rope_attn_fwd_ad(const at::Tensor& q,
                                                                                const at::Tensor& k,
                                                                                const at::Tensor& v,
                                                                                const at::Tensor& cos,
                                                                                const at::Tensor& sin, double scale) {
  if (!records(q, k, v, cos, sin)) MT_BELOW(gqa_rope_attn_fwd, q, k, v, cos, sin, scale);
  auto r = RopeAttnFn::apply(q, k, v, cos, sin, scale);
  return {r[0], r[1], r[2], r[3]};
}
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> gqa_rope_attn_packed_fwd_ad(const at::Tensor& qkv,
                                                                                       const at::Tensor& cos,
                                                                                       const at::Tensor& sin,
                                                                                       int64_t hq, int64_t hkv,
                                                                                       double scale) {
  if (!records(qkv, cos, sin)) MT_BELOW(gqa_rope_attn_packed_fwd, qkv, cos, sin, hq, hkv, scale);
  auto r = PackedAttnFn::apply(qkv, cos, sin, hq, hkv, scale);
  return {r[0], r[1], r[2], r[3]};
}
std::tuple<at::Tensor, at::Tensor> rms_norm_fwd_ad(const at::Tensor& x, const at::Tensor& w, double eps) {
  if (!records(x, w)) MT_BELOW(rms_norm_fwd, x, w, eps);
  auto r = RmsFn::apply(x, w, eps);
  return {r[0], r[1]};
}
std::tuple<at::Tensor, at::Tensor, at::Tensor> add_rms_norm_fwd_ad(const at::Tensor& x, const at::Tensor& res,
                                                                   const at::Tensor& w, double eps) {
  if (!records(x, res, w)) MT_BELOW(add_rms_norm_fwd, x, res, w, eps);
  auto r = AddRmsFn::apply(x, res, w, eps);
  return {r[0], r[1], r[2]};
}
std::tuple<at::Tensor, at::Tensor> rms_norm_fwd_mixed_ad(const at::Tensor& x, const at::Tensor& w, double eps,
                                                         int64_t act) {
  if (!records(x, w)) MT_BELOW(rms_norm_fwd_mixed, x, w, eps, act);
  auto r = RmsMixedFn::apply(x, w, eps, act);
  return {r[0], r[1]};
}
std::tuple<at::Tensor, at::Tensor, at::Tensor> add_rms_norm_fwd_mixed_ad(const at::Tensor& x, const at::Tensor& res,
                                                                         const at::Tensor& w, double eps) {
  if (!records(x, res, w)) MT_BELOW(add_rms_norm_fwd_mixed, x, res, w, eps);
  auto r = AddRmsMixedFn::apply(x, res, w, eps);
  return {r[0], r[1], r[2]};
}
at::Tensor swiglu_fwd_ad(const at::Tensor& gate, const at::Tensor& up) {
  if (!records(gate, up)) MT_BELOW(swiglu_fwd, gate, up);
  return SwigluFn::apply(gate, up);
}
at::Tensor swiglu_packed_fwd_ad(const at::Tensor& gate_up) {
  if (!records(gate_up)) MT_BELOW(swiglu_packed_fwd, gate_up);
  return SwigluPackedFn::apply(gate_up);
}
std::tuple<at::Tensor, at::Tensor> rope_fwd_ad(const at::Tensor& q, const at::Tensor& k, const at::Tensor& cos,
                                               const at::Tensor& sin, bool inverse) {
  if (!records(q, k, cos, sin)) MT_BELOW(rope_fwd, q, k, cos, sin, inverse);
  auto r = RopeFn::apply(q, k, cos, sin, inverse);
  return {r[0], r[1]};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> fused_linear_ce_ad(const at::Tensor& hidden, const at::Tensor& weight,
                                                                  const at::Tensor& labels, int64_t ignore_index,
                                                                  int64_t compute, bool need_grad) {
  if (!records(hidden, weight)) {
    at::AutoDispatchBelowADInplaceOrView below;
    static const auto op = op_handle<CeSig>("mega_trading_amd::fused_linear_ce");
    return op.call(hidden, weight, labels, ignore_index, compute, need_grad);
  }
  auto r = LinearCeFn::apply(hidden, weight, labels, ignore_index, compute, need_grad);
  return {r[0], r[1], r[2]};
}

// An op without a formula (the backward ops among them: no double backward)
// refuses a gradient instead of dropping it: its outputs' node raises.  torch's
// own fallback for such ops only warns and passes no gradient on.  Caches that an
// op writes keep their own autograd state.
void no_formula(const c10::OperatorHandle& op, c10::DispatchKeySet ks, torch::jit::Stack* stack) {
  variable_list recorded;
  bool tangent = false;
  if (c10::GradMode::is_enabled()) {
    auto look = [&](const at::Tensor& t) {
      if (!t.defined()) return;
      if (t.requires_grad()) recorded.push_back(t);
      tangent |= t._fw_grad(0).defined();
    };
    for (const c10::IValue& a : torch::jit::last(*stack, op.schema().arguments().size())) {
      if (a.isTensor()) look(a.toTensor());
      else if (a.isTensorList())
        for (const at::Tensor& t : a.toTensorList()) look(t);
    }
  }
  if (!recorded.empty()) {
    if (const auto& f = at::functorch::functorchTLSAccessor()) f->checkSupportsCppAutogradFunction();
    TORCH_CHECK(!tangent, op.schema().name(), " has no forward-mode derivative");
  }
  {
    at::AutoDispatchBelowAutograd below;
    op.redispatchBoxed(ks & c10::after_autograd_keyset, stack);
  }
  if (recorded.empty()) return;
  const std::shared_ptr<torch::autograd::Node> node(
      new torch::autograd::Error(
          "Trying to backward through " + op.schema().name() + " but no autograd formula was registered",
          torch::autograd::collect_next_edges(recorded)),
      torch::autograd::deleteNode);
  for (const c10::IValue& r : torch::jit::last(*stack, op.schema().returns().size()))
    if (r.isTensor() && torch::autograd::isDifferentiableType(r.toTensor().scalar_type()))
      torch::autograd::set_history(r.toTensor(), node);
}

// An op that writes caches counts it in their versions, so that a backward over
// a cache saved before the write raises.  (torch's own fallback for this key only
// looks at arguments that are returned.)
void count_writes(const c10::OperatorHandle& op, c10::DispatchKeySet ks, torch::jit::Stack* stack) {
  const auto& params = op.schema().arguments();
  variable_list written;
  for (size_t i = 0; i < params.size(); ++i) {
    const c10::IValue& a = torch::jit::peek(*stack, i, params.size());
    if (params[i].alias_info() && params[i].alias_info()->isWrite() && a.isTensor()) written.push_back(a.toTensor());
  }
  {
    at::AutoDispatchBelowADInplaceOrView below;
    op.redispatchBoxed(ks & c10::after_ADInplaceOrView_keyset, stack);
  }
  for (const at::Tensor& t : written)
    if (!t.is_inference()) torch::autograd::impl::bump_version(t);
}

}  // namespace

TORCH_LIBRARY_IMPL(mega_trading_amd, Autograd, m) {
  // gqa_attn_bwd_packed keeps torch's fallback, a warning, which it has always had
  for (const char* op : {"gqa_attn_bwd", "gqa_attn_decode", "gqa_attn_decode_dev", "decode_rope_append",
                         "gqa_attn_decode_append", "rms_norm_bwd", "add_rms_norm_bwd", "rms_norm_bwd_mixed", "swiglu_bwd",
                         "swiglu_packed_bwd", "topk_sample", "linear_rows", "linear_rows_gate", "ce_sum", "scale_pair"})
    m.impl(op, torch::CppFunction::makeFromBoxedFunction<&no_formula>());
  m.impl("fused_linear_ce", &fused_linear_ce_ad);
  m.impl("gqa_attn_fwd", &gqa_attn_fwd_ad);
  m.impl("gqa_rope_attn_fwd", &gqa_rope_attn_fwd_ad);
  m.impl("gqa_rope_attn_packed_fwd", &gqa_rope_attn_packed_fwd_ad);
  m.impl("rms_norm_fwd", &rms_norm_fwd_ad);
  m.impl("add_rms_norm_fwd", &add_rms_norm_fwd_ad);
  m.impl("rms_norm_fwd_mixed", &rms_norm_fwd_mixed_ad);
  m.impl("add_rms_norm_fwd_mixed", &add_rms_norm_fwd_mixed_ad);
  m.impl("swiglu_fwd", &swiglu_fwd_ad);
  m.impl("swiglu_packed_fwd", &swiglu_packed_fwd_ad);
  m.impl("rope_fwd", &rope_fwd_ad);
}

TORCH_LIBRARY_IMPL(mega_trading_amd, ADInplaceOrView, m) {
  for (const char* op : {"decode_rope_append", "gqa_attn_decode_append"})
    m.impl(op, torch::CppFunction::makeFromBoxedFunction<&count_writes>());
}

TORCH_LIBRARY_IMPL(mega_trading_amd, CUDA, m) {
  m.impl("gqa_attn_fwd", &gqa_attn_fwd);
  m.impl("gqa_rope_attn_fwd", &gqa_rope_attn_fwd);
  m.impl("gqa_attn_bwd", &gqa_attn_bwd);
  m.impl("gqa_rope_attn_packed_fwd", &gqa_rope_attn_packed_fwd);
  m.impl("gqa_attn_bwd_packed", &gqa_attn_bwd_packed);
  m.impl("gqa_attn_decode", &gqa_attn_decode);
  m.impl("gqa_attn_decode_dev", &gqa_attn_decode_dev);
  m.impl("decode_rope_append", &decode_rope_append);
  m.impl("gqa_attn_decode_append", &gqa_attn_decode_append);
  m.impl("rms_norm_fwd", &rms_norm_fwd);
  m.impl("rms_norm_bwd", &rms_norm_bwd);
  m.impl("add_rms_norm_fwd", &add_rms_norm_fwd);
  m.impl("add_rms_norm_bwd", &add_rms_norm_bwd);
  m.impl("rms_norm_fwd_mixed", &rms_norm_fwd_mixed);
  m.impl("add_rms_norm_fwd_mixed", &add_rms_norm_fwd_mixed);
  m.impl("rms_norm_bwd_mixed", &rms_norm_bwd_mixed);
  m.impl("swiglu_fwd", &swiglu_fwd);
  m.impl("swiglu_bwd", &swiglu_bwd);
  m.impl("swiglu_packed_fwd", &swiglu_packed_fwd);
  m.impl("swiglu_packed_bwd", &swiglu_packed_bwd);
  m.impl("rope_fwd", &rope_fwd);
  m.impl("topk_sample", &topk_sample);
  m.impl("linear_rows", &linear_rows);
  m.impl("linear_rows_gate", &linear_rows_gate);
  m.impl("ce_count", &ce_count);
  m.impl("ce_sum", &ce_sum);
  m.impl("scale_pair", &scale_pair);
}
