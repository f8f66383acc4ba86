// Host path of the Python entry points: argument checks, output allocation, autograd and the calls into libqfa.so, as
// one CPython module (_qfa_host).  A call costs a few microseconds here against 60 to 250 when the same steps run as
// Python (a dozen torch.empty, three torch.autograd.Function round trips through the interpreter, ctypes calls of up to
// 45 arguments): at B1 H4 N256 D64 the kernels of a training step take about 50 us, so the host was the bound.
//
// The module does not link against libqfa.so: the binding that loads the library hands over the addresses of its entry
// points (init), so there is one place that decides which library file is used, and none of this works without it.
// Nothing is kept between calls.
#include <algorithm>
#include <cmath>
#include <ATen/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <array>
#include <string>
#include <utility>

#include "../../include/qfa.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------------ the library's entry points
struct Api {
#define QFA_ENTRY(name) decltype(&::name) name = nullptr
  QFA_ENTRY(qfa_last_error);
  QFA_ENTRY(qfa_quant_per_token);
  QFA_ENTRY(qfa_quant_per_token_pair);
  QFA_ENTRY(qfa_quant_qkv_f32);
  QFA_ENTRY(qfa_dequant_per_token);
  QFA_ENTRY(qfa_code_rowsum);
  QFA_ENTRY(qfa_cache_stage_q);
  QFA_ENTRY(qfa_attn_fwd);
  QFA_ENTRY(qfa_attn_fwd_split_workspace_bytes);
  QFA_ENTRY(qfa_attn_fwd_split);
  QFA_ENTRY(qfa_bench_qk_stage);
  QFA_ENTRY(qfa_attn_bwd_workspace_bytes);
  QFA_ENTRY(qfa_attn_bwd);
  QFA_ENTRY(qfa_attn_bwd_split_workspace_bytes);
  QFA_ENTRY(qfa_attn_bwd_f32);
  QFA_ENTRY(qfa_attn_bwd_f32_workspace_bytes);
  QFA_ENTRY(qfa_sum_grads);
  QFA_ENTRY(qfa_attn_fwd_shared_kv_workspace_bytes);
  QFA_ENTRY(qfa_attn_fwd_shared_kv);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_workspace_bytes);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_split);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_is_direct);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_direct);
  QFA_ENTRY(qfa_attn_fwd_cache_workspace_bytes);
  QFA_ENTRY(qfa_attn_fwd_cache_lse);
  QFA_ENTRY(qfa_dout_normalise_workspace_bytes);
  QFA_ENTRY(qfa_dout_normalise_cast);
#undef QFA_ENTRY
};
Api api;

void init(const py::dict &address) {
  auto get = [&](auto &fn, const char *name) {
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(address[name].cast<uintptr_t>());
  };
#define QFA_ENTRY(name) get(api.name, #name)
  QFA_ENTRY(qfa_last_error);
  QFA_ENTRY(qfa_quant_per_token);
  QFA_ENTRY(qfa_quant_per_token_pair);
  QFA_ENTRY(qfa_quant_qkv_f32);
  QFA_ENTRY(qfa_dequant_per_token);
  QFA_ENTRY(qfa_code_rowsum);
  QFA_ENTRY(qfa_cache_stage_q);
  QFA_ENTRY(qfa_attn_fwd);
  QFA_ENTRY(qfa_attn_fwd_split_workspace_bytes);
  QFA_ENTRY(qfa_attn_fwd_split);
  QFA_ENTRY(qfa_bench_qk_stage);
  QFA_ENTRY(qfa_attn_bwd_workspace_bytes);
  QFA_ENTRY(qfa_attn_bwd);
  QFA_ENTRY(qfa_attn_bwd_split_workspace_bytes);
  QFA_ENTRY(qfa_attn_bwd_f32);
  QFA_ENTRY(qfa_attn_bwd_f32_workspace_bytes);
  QFA_ENTRY(qfa_sum_grads);
  QFA_ENTRY(qfa_attn_fwd_shared_kv_workspace_bytes);
  QFA_ENTRY(qfa_attn_fwd_shared_kv);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_workspace_bytes);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_split);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_is_direct);
  QFA_ENTRY(qfa_attn_bwd_shared_kv_direct);
  QFA_ENTRY(qfa_attn_fwd_cache_workspace_bytes);
  QFA_ENTRY(qfa_attn_fwd_cache_lse);
  QFA_ENTRY(qfa_dout_normalise_workspace_bytes);
  QFA_ENTRY(qfa_dout_normalise_cast);
#undef QFA_ENTRY
}

void check(int code, const char *what) {
  if (code != 0) TORCH_CHECK(false, what, " failed (code ", code, "): ", api.qfa_last_error());
}

// ------------------------------------------------------------------------------------------------------ checks
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return QFA_F32;
    case at::kHalf: return QFA_F16;
    case at::kBFloat16: return QFA_BF16;
    default: return -1;
  }
}
bool is_io(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }

template <typename... T> void require_gpu(const Tensor &first, const T &...rest) {
  auto one = [&](const Tensor &t) {
    TORCH_CHECK(t.is_cuda(), "quant_flash_attn_amd runs on the GPU only: got a tensor on '", t.device().str(),
                "'. There is no CPU implementation in this package.");
    TORCH_CHECK(t.device() == first.device(), "all tensors must be on the same device, got ", first.device().str(), " and ",
                t.device().str());
  };
  one(first);
  (one(rest), ...);
}
void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// [B,H,N,D] tensor whose rows are contiguous and whose strides and base are multiples of `align` bytes
Tensor rows_aligned(const Tensor &t, int64_t align) {
  const int64_t es = t.element_size();
  bool ok = t.stride(3) == 1 && t.stride(2) >= t.size(3) && reinterpret_cast<uintptr_t>(t.data_ptr()) % align == 0;
  for (int i = 0; i < 3; ++i) ok = ok && t.stride(i) > 0 && (t.stride(i) * es) % align == 0;
  return ok ? t : t.contiguous();
}
Tensor rows16(const Tensor &t) { return rows_aligned(t, 16); }
// the n values of a per-token vector, dense
Tensor flat(const Tensor &t, at::ScalarType dtype, int64_t n, const char *name) {
  TORCH_CHECK_VALUE(t.scalar_type() == dtype && t.numel() == n, name, ": expected ", n, " values of ", dtype, ", got ",
                    t.numel(), " of ", t.scalar_type());
  return t.is_contiguous() ? t : t.contiguous();
}
void check_codes(const Tensor &t, const char *name) {
  TORCH_CHECK_VALUE(t.dim() == 4 && t.scalar_type() == at::kChar, name, " must be a 4-D int8 tensor");
}
Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor &like) {
  return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}
Tensor to(const Tensor &t, at::ScalarType dtype) { return t.scalar_type() == dtype ? t : t.to(dtype); }
#define QFA_STRIDES(t) (t).stride(0), (t).stride(1), (t).stride(2)

// -------------------------------------------------------------------------------------- quantized operands
// A quantized tensor as the attention entry points take it
struct Quantized {
  const int8_t *codes;
  const float *scale;
  const int8_t *zp;
  const int32_t *rowsum;
  int64_t B, H, N, D;
  int64_t sb, sh, sn;   // strides of the codes
};

// The outputs of quantizing two tensors, and the log-sum-exp of the attention on them, in ONE allocation: one block for
// autograd to keep, one call of the allocator instead of nine
struct PairBuffer {
  int64_t B, H, N[2], D;
  int64_t codes[2], scale[2], rowsum[2], zp[2], lse, bytes;
  PairBuffer(int64_t B_, int64_t H_, int64_t Nq, int64_t Nk, int64_t D_) : B(B_), H(H_), N{Nq, Nk}, D(D_) {
    int64_t at = 0;
    auto take = [&](int64_t n) {
      const int64_t here = at;
      at += (n + 255) / 256 * 256;
      return here;
    };
    for (int i = 0; i < 2; ++i) codes[i] = take(B * H * N[i] * D);
    for (int i = 0; i < 2; ++i) scale[i] = take(B * H * N[i] * 4);
    for (int i = 0; i < 2; ++i) rowsum[i] = take(B * H * N[i] * 4);
    for (int i = 0; i < 2; ++i) zp[i] = take(B * H * N[i]);
    lse = take(B * H * N[0] * 4);
    bytes = at;
  }
  Quantized view(const Tensor &buf, int i) const {
    uint8_t *p = buf.data_ptr<uint8_t>();
    return {reinterpret_cast<int8_t *>(p + codes[i]), reinterpret_cast<float *>(p + scale[i]),
            reinterpret_cast<int8_t *>(p + zp[i]), reinterpret_cast<int32_t *>(p + rowsum[i]), B, H, N[i], D,
            H * N[i] * D, N[i] * D, D};
  }
  float *lse_of(const Tensor &buf) const { return reinterpret_cast<float *>(buf.data_ptr<uint8_t>() + lse); }
};

Tensor check_input(const Tensor &x) {
  TORCH_CHECK_VALUE(x.dim() == 4, "expected a 4-D (Batch, Heads, Seq, Head_Dim) tensor, got shape ", x.sizes());
  TORCH_CHECK_TYPE(dtype_code(x.scalar_type()) >= 0, "unsupported dtype ", x.scalar_type(),
                   ": expected float16, bfloat16 or float32");
  require_gpu(x);
  return rows16(x);
}

// x -> the memory of `out`
void quantize_into(const Tensor &x, const Quantized &out) {
  check(api.qfa_quant_per_token(x.data_ptr(), dtype_code(x.scalar_type()), const_cast<int8_t *>(out.codes),
                                const_cast<float *>(out.scale), nullptr, 0, const_cast<int8_t *>(out.zp),
                                const_cast<int32_t *>(out.rowsum), out.B, out.H, out.N, (int)out.D, QFA_STRIDES(x), out.sb,
                                out.sh, out.sn, stream_of(x)),
        "qfa_quant_per_token");
}
void quantize_pair_into(const Tensor &x0, const Tensor &x1, const Quantized &a, const Quantized &b) {
  if (x0.scalar_type() != x1.scalar_type()) {
    quantize_into(x0, a);
    quantize_into(x1, b);
    return;
  }
  auto w = [](auto *p) { return const_cast<std::remove_const_t<std::remove_pointer_t<decltype(p)>> *>(p); };
  check(api.qfa_quant_per_token_pair(x0.data_ptr(), x1.data_ptr(), dtype_code(x0.scalar_type()), w(a.codes), w(b.codes),
                                     w(a.scale), w(b.scale), w(a.zp), w(b.zp), w(a.rowsum), w(b.rowsum), a.B, a.H, a.N,
                                     b.N, (int)a.D, QFA_STRIDES(x0), QFA_STRIDES(x1), a.sb, a.sh, a.sn, b.sb, b.sh, b.sn,
                                     stream_of(x0)),
        "qfa_quant_per_token_pair");
}

using QuantTensors = std::tuple<Tensor, Tensor, Tensor, Tensor>;   // codes, scale fp32, zero point, row sum

// The fp32 scale is an output only where it is asked for (scale_dtype fp32)
std::tuple<Tensor, Tensor, Tensor> quant(const Tensor &x_in, at::ScalarType scale_dtype) {
  TORCH_CHECK_TYPE(dtype_code(scale_dtype) >= 0, "scale_dtype must be float16, bfloat16 or float32, got ", scale_dtype);
  const Tensor x = check_input(x_in);
  const c10::DeviceGuard guard(x.device());
  const int64_t B = x.size(0), H = x.size(1), N = x.size(2), D = x.size(3);
  Tensor codes = empty({B, H, N, D}, at::kChar, x), scale = empty({B, H, N, 1}, scale_dtype, x),
         zp = empty({B, H, N, 1}, at::kChar, x);
  const bool lp = scale_dtype != at::kFloat;
  check(api.qfa_quant_per_token(x.data_ptr(), dtype_code(x.scalar_type()), codes.data_ptr<int8_t>(),
                                lp ? nullptr : scale.data_ptr<float>(), lp ? scale.data_ptr() : nullptr,
                                lp ? dtype_code(scale_dtype) : 0, zp.data_ptr<int8_t>(), nullptr, B, H, N, (int)D,
                                QFA_STRIDES(x), QFA_STRIDES(codes), stream_of(x)),
        "qfa_quant_per_token");
  return {codes, scale, zp};
}

QuantTensors alloc_quantized(const Tensor &x) {
  const int64_t B = x.size(0), H = x.size(1), N = x.size(2), D = x.size(3);
  return {empty({B, H, N, D}, at::kChar, x), empty({B, H, N, 1}, at::kFloat, x), empty({B, H, N, 1}, at::kChar, x),
          empty({B, H, N, 1}, at::kInt, x)};
}
Quantized view_of(const QuantTensors &t) {
  const Tensor &c = std::get<0>(t);
  return {c.data_ptr<int8_t>(), std::get<1>(t).data_ptr<float>(), std::get<2>(t).data_ptr<int8_t>(),
          std::get<3>(t).data_ptr<int32_t>(), c.size(0), c.size(1), c.size(2), c.size(3), QFA_STRIDES(c)};
}
QuantTensors quant_attn(const Tensor &x_in) {
  const Tensor x = check_input(x_in);
  const c10::DeviceGuard guard(x.device());
  QuantTensors out = alloc_quantized(x);
  quantize_into(x, view_of(out));
  return out;
}
std::pair<QuantTensors, QuantTensors> quant_attn_pair(const Tensor &x0_in, const Tensor &x1_in) {
  const Tensor x0 = check_input(x0_in), x1 = check_input(x1_in);
  if (x0.size(0) != x1.size(0) || x0.size(1) != x1.size(1) || x0.size(3) != x1.size(3) || x0.device() != x1.device())
    return {quant_attn(x0), quant_attn(x1)};
  const c10::DeviceGuard guard(x0.device());
  QuantTensors a = alloc_quantized(x0), b = alloc_quantized(x1);
  quantize_pair_into(x0, x1, view_of(a), view_of(b));
  return {a, b};
}

Tensor dequant(const Tensor &codes_in, const Tensor &scale_in, const Tensor &zp_in, at::ScalarType dtype) {
  require_gpu(codes_in, scale_in, zp_in);
  check_codes(codes_in, "codes");
  TORCH_CHECK_TYPE(dtype_code(dtype) >= 0 && dtype_code(scale_in.scalar_type()) >= 0,
                   "dtype and scale.dtype must be float16, bfloat16 or float32");
  const c10::DeviceGuard guard(codes_in.device());
  const Tensor codes = rows_aligned(codes_in, 8), scale = scale_in.contiguous(), zp = zp_in.contiguous();
  const int64_t B = codes.size(0), H = codes.size(1), N = codes.size(2), D = codes.size(3);
  TORCH_CHECK_VALUE(scale.numel() == B * H * N && zp.numel() == B * H * N && zp.scalar_type() == at::kChar,
                    "scale / zero_point must hold one value per token (zero_point int8)");
  Tensor out = empty({B, H, N, D}, dtype, codes);
  check(api.qfa_dequant_per_token(codes.data_ptr<int8_t>(), scale.data_ptr(), dtype_code(scale.scalar_type()),
                                  zp.data_ptr<int8_t>(), out.data_ptr(), dtype_code(dtype), B, H, N, (int)D,
                                  QFA_STRIDES(codes), QFA_STRIDES(out), stream_of(codes)),
        "qfa_dequant_per_token");
  return out;
}

Tensor rowsum(const Tensor &codes_in) {
  require_gpu(codes_in);
  check_codes(codes_in, "codes");
  const c10::DeviceGuard guard(codes_in.device());
  const Tensor codes = rows_aligned(codes_in, 8);
  const int64_t B = codes.size(0), H = codes.size(1), N = codes.size(2), D = codes.size(3);
  Tensor out = empty({B, H, N, 1}, at::kInt, codes);
  check(api.qfa_code_rowsum(codes.data_ptr<int8_t>(), out.data_ptr<int32_t>(), B, H, N, (int)D, QFA_STRIDES(codes),
                            stream_of(codes)),
        "qfa_code_rowsum");
  return out;
}

// ------------------------------------------------------------------------------------- INT8-score attention
// o and lse are written; v and o have rows of 16-byte alignment
void fwd_into(const Quantized &q, const Quantized &k, const Tensor &v, const Tensor &o, float *lse, bool causal, double sm,
              bool qk_only = false) {
  auto *entry = qk_only ? api.qfa_bench_qk_stage : api.qfa_attn_fwd;
  check(entry(q.codes, q.scale, q.zp, q.rowsum, k.codes, k.scale, k.zp, k.rowsum, v.data_ptr(), o.data_ptr(), lse,
              dtype_code(v.scalar_type()), q.B, q.H, q.N, k.N, (int)q.D, q.sb, q.sh, q.sn, k.sb, k.sh, k.sn,
              QFA_STRIDES(v), QFA_STRIDES(o), (float)sm, causal, stream_of(v)),
        qk_only ? "qfa_bench_qk_stage" : "qfa_attn_fwd");
}

// Scratch that a call can do without: undefined for none, and where the memory is not there (the call is not split then, and runs
// wherever it runs without a scratch)
Tensor optional_scratch(int64_t bytes, const Tensor &like) {
  if (bytes <= 0) return Tensor();
  try {
    return empty({bytes}, at::kByte, like);
  } catch (const c10::OutOfMemoryError &) {
    return Tensor();
  }
}
void *data_of(const Tensor &scratch) { return scratch.defined() ? scratch.data_ptr() : nullptr; }
int64_t bytes_of(const Tensor &scratch) { return scratch.defined() ? scratch.numel() : 0; }

// the same with the keys split over workgroups where there are few queries; o32 dense, o or o32 may be undefined
void fwd_split_into(const Quantized &q, const Quantized &k, const Tensor &v, const Tensor &o, const Tensor &o32, float *lse,
                    bool causal, double sm) {
  const Tensor ws = optional_scratch(api.qfa_attn_fwd_split_workspace_bytes(q.B, q.H, q.N, k.N, (int)q.D, causal), v);
  const Tensor &like = o.defined() ? o : o32;
  check(api.qfa_attn_fwd_split(q.codes, q.scale, q.zp, q.rowsum, k.codes, k.scale, k.zp, k.rowsum, v.data_ptr(),
                               o.defined() ? o.data_ptr() : nullptr, o32.defined() ? o32.data_ptr<float>() : nullptr, lse,
                               dtype_code(v.scalar_type()), q.B, q.H, q.N, k.N, (int)q.D, q.sb, q.sh, q.sn, k.sb, k.sh, k.sn,
                               QFA_STRIDES(v), QFA_STRIDES(like), (float)sm, causal, data_of(ws), bytes_of(ws), stream_of(v)),
        "qfa_attn_fwd_split");
}

using Grads = std::array<Tensor, 3>;
// split: the streamed rows may be dealt to several workgroups (autograd; the public call's bits do not depend on the batch);
// f32: dO comes and the gradients leave in fp32
Grads bwd_of(const Quantized &q, const Quantized &k, const Tensor &v_in, const Tensor &o_in, const Tensor &do_in,
             const float *lse, bool causal, double sm, bool split, bool f32 = false) {
  const at::ScalarType gt = f32 ? at::kFloat : v_in.scalar_type();
  const Tensor v = rows16(v_in), o = rows16(o_in), dout = rows16(to(do_in, gt));
  const int64_t plain = f32 ? api.qfa_attn_bwd_f32_workspace_bytes(q.B, q.H, q.N, k.N, (int)q.D)
                            : api.qfa_attn_bwd_workspace_bytes(q.B, q.H, q.N, k.N, (int)q.D),
                most = split || f32 ? api.qfa_attn_bwd_split_workspace_bytes(q.B, q.H, q.N, k.N, (int)q.D, causal, f32) : plain;
  TORCH_CHECK_VALUE(plain > 0, "unsupported backward shape B=", q.B, " H=", q.H, " Nq=", q.N, " Nk=", k.N, " D=", q.D);
  Tensor dq = empty({q.B, q.H, q.N, q.D}, gt, v), dk = empty({q.B, q.H, k.N, q.D}, gt, v), dv = empty({q.B, q.H, k.N, q.D}, gt, v);
  Tensor ws;   // (last: what is left is for the parts)
  if (most > plain) ws = optional_scratch(most, v);
  if (!ws.defined()) ws = empty({plain}, at::kByte, v);
  const int64_t ws_bytes = ws.numel();
  if (f32) {
    check(api.qfa_attn_bwd_f32(q.codes, q.scale, q.zp, q.rowsum, k.codes, k.scale, k.zp, k.rowsum, v.data_ptr(), o.data_ptr(),
                               dout.data_ptr<float>(), lse, ws.data_ptr(), ws_bytes, dq.data_ptr<float>(), dk.data_ptr<float>(),
                               dv.data_ptr<float>(), dtype_code(v.scalar_type()), q.B, q.H, q.N, k.N, (int)q.D, q.sb, q.sh, q.sn,
                               k.sb, k.sh, k.sn, QFA_STRIDES(v), QFA_STRIDES(o), QFA_STRIDES(dout), QFA_STRIDES(dq),
                               QFA_STRIDES(dk), QFA_STRIDES(dv), (float)sm, causal, stream_of(v)),
          "qfa_attn_bwd_f32");
    return {dq, dk, dv};
  }
  check(api.qfa_attn_bwd(q.codes, q.scale, q.zp, q.rowsum, k.codes, k.scale, k.zp, k.rowsum, v.data_ptr(), o.data_ptr(),
                         dout.data_ptr(), lse, ws.data_ptr(), ws_bytes, dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                         dtype_code(v.scalar_type()), q.B, q.H, q.N, k.N, (int)q.D, q.sb, q.sh, q.sn, k.sb, k.sh, k.sn,
                         QFA_STRIDES(v), QFA_STRIDES(o), QFA_STRIDES(dout), QFA_STRIDES(dq), QFA_STRIDES(dk),
                         QFA_STRIDES(dv), (float)sm, causal, stream_of(v)),
        "qfa_attn_bwd");
  return {dq, dk, dv};
}

// a caller's (codes, scale fp32, zero point, row sum), checked; the tensors that had to be copied are kept in `hold`
struct Unpacked : Quantized {
  std::array<Tensor, 4> hold;
};
Unpacked unpack(const QuantTensors &t, const char *name) {
  const Tensor &c = std::get<0>(t);
  TORCH_CHECK_VALUE(c.dim() == 4 && c.scalar_type() == at::kChar, name, ".codes must be a 4-D int8 tensor");
  const int64_t n = c.size(0) * c.size(1) * c.size(2);
  const std::string s(name);
  Unpacked u;
  u.hold = {rows16(c), flat(std::get<1>(t), at::kFloat, n, (s + ".scale").c_str()),
            flat(std::get<2>(t), at::kChar, n, (s + ".zero_point").c_str()),
            flat(std::get<3>(t), at::kInt, n, (s + ".rowsum").c_str())};
  static_cast<Quantized &>(u) = view_of({u.hold[0], u.hold[1], u.hold[2], u.hold[3]});
  return u;
}

std::tuple<Tensor, Tensor> attn_fwd(const QuantTensors &qq, const QuantTensors &kq, const Tensor &v_in, bool causal,
                                    double sm, bool qk_only) {
  TORCH_CHECK_TYPE(is_io(v_in.scalar_type()), "v must be bfloat16 or float16, got ", v_in.scalar_type());
  const Unpacked q = unpack(qq, "q"), k = unpack(kq, "k");
  require_gpu(q.hold[0], q.hold[1], q.hold[2], q.hold[3], k.hold[0], k.hold[1], k.hold[2], k.hold[3], v_in);
  TORCH_CHECK_VALUE(k.B == q.B && k.H == q.H && k.D == q.D && v_in.sizes() == k.hold[0].sizes(), "shape mismatch: q ",
                    q.hold[0].sizes(), ", k ", k.hold[0].sizes(), ", v ", v_in.sizes());
  const c10::DeviceGuard guard(v_in.device());
  const Tensor v = rows16(v_in);
  Tensor o = empty({q.B, q.H, q.N, q.D}, v.scalar_type(), v), lse = empty({q.B, q.H, q.N}, at::kFloat, v);
  fwd_into(q, k, v, o, lse.data_ptr<float>(), causal, sm, qk_only);
  return {o, lse};
}

Grads attn_bwd(const QuantTensors &qq, const QuantTensors &kq, const Tensor &v, const Tensor &o, const Tensor &dout,
               const Tensor &lse, bool causal, double sm) {
  TORCH_CHECK_TYPE(is_io(v.scalar_type()), "v must be bfloat16 or float16, got ", v.scalar_type());
  const Unpacked q = unpack(qq, "q"), k = unpack(kq, "k");
  const std::array<int64_t, 4> qs{q.B, q.H, q.N, q.D}, ks{q.B, q.H, k.N, q.D};
  TORCH_CHECK_VALUE(o.sizes() == at::IntArrayRef(qs) && dout.sizes() == at::IntArrayRef(qs) && v.sizes() == at::IntArrayRef(ks),
                    "shape mismatch between o / do / v and the quantized tensors");
  TORCH_CHECK_TYPE(o.scalar_type() == v.scalar_type(), "o and v must have the same dtype");
  require_gpu(q.hold[0], k.hold[0], v, o, dout, lse);
  const c10::DeviceGuard guard(v.device());
  return bwd_of(q, k, v, o, dout, flat(lse, at::kFloat, q.B * q.H * q.N, "lse").data_ptr<float>(), causal, sm,
                false);
}

at::ScalarType io_dtype(const Tensor &t) { return is_io(t.scalar_type()) ? t.scalar_type() : at::kBFloat16; }
bool wants_grad(std::initializer_list<const Tensor *> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor *t : ts)
    if (t->requires_grad()) return true;
  return false;
}

// The operators have no forward-mode derivative: a tangent is refused, with or without a backward gradient beside it (an
// input that needs none does not reach the autograd node, which would refuse it).
void refuse_tangents(std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(0).defined(),
                                "quant_flash_attn_amd: forward-mode differentiation (jvp) is not implemented for this operator");
}
// A call that is being traced goes through the dispatcher, which records the operator as one node of the graph (what the
// function below does by itself is invisible there but for its allocations); others save themselves that round trip.
template <typename F> struct Traced;
template <typename... A> struct Traced<Tensor(A...)> {
  static Tensor call(const char *name, A... args) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Tensor(A...)>().call(args...);
  }
};

// forward results that the backward needs: the pair buffer (codes, scales, zero points, row sums, LSE), v and o in 16 bit
struct Kept {
  Tensor buf, v16, o16, o;
};
// backward from them
Grads bwd_from(AutogradContext *ctx, const variable_list &saved, const Tensor &grad, bool f32) {
  const Tensor &buf = saved[0], &v16 = saved[1], &o16 = saved[2];
  const int64_t Nk = v16.size(2);
  const PairBuffer pb(o16.size(0), o16.size(1), o16.size(2), Nk, o16.size(3));
  const c10::DeviceGuard guard(v16.device());
  return bwd_of(pb.view(buf, 0), pb.view(buf, 1), v16, o16, grad, pb.lse_of(buf),
                ctx->saved_data["causal"].toBool(), ctx->saved_data["sm"].toDouble(), true, f32);
}

// ---- q, k, v
bool all_f32(const Tensor &q, const Tensor &k, const Tensor &v) {
  return q.scalar_type() == at::kFloat && k.scalar_type() == at::kFloat && v.scalar_type() == at::kFloat;
}
// keep: what a backward takes is made too
Kept qkv_forward(const Tensor &q_in, const Tensor &k_in, const Tensor &v_in, bool causal, double sm, bool keep) {
  const c10::DeviceGuard guard(q_in.device());
  const Tensor q = check_input(q_in), k = check_input(k_in);
  const PairBuffer pb(q.size(0), q.size(1), q.size(2), k.size(2), q.size(3));
  Kept r;
  r.buf = empty({pb.bytes}, at::kByte, q);
  if (all_f32(q, k, v_in) && (pb.D == 64 || pb.D == 128 || pb.D == 256)) {
    // fp32 in and out without launches of their own for the conversions: the quantizer's launch takes V along, the forward
    // writes O in both types, the staging pass rounds dO, and the gradients leave in fp32 (B1 H4 N256 D64, forward and backward:
    // 5 launches instead of 11, 103 -> 75 us, of which the kernels are 37)
    const Tensor v = rows16(v_in);
    const Quantized a = pb.view(r.buf, 0), b = pb.view(r.buf, 1);
    auto w = [](auto *p) { return const_cast<std::remove_const_t<std::remove_pointer_t<decltype(p)>> *>(p); };
    r.v16 = empty({pb.B, pb.H, pb.N[1], pb.D}, at::kBFloat16, q);
    check(api.qfa_quant_qkv_f32(q.data_ptr<float>(), k.data_ptr<float>(), v.data_ptr<float>(), w(a.codes), w(b.codes), w(a.scale),
                                w(b.scale), w(a.zp), w(b.zp), w(a.rowsum), w(b.rowsum), r.v16.data_ptr(), a.B, a.H, a.N, b.N,
                                (int)a.D, QFA_STRIDES(q), QFA_STRIDES(k), QFA_STRIDES(v), a.sb, a.sh, a.sn, b.sb, b.sh, b.sn,
                                stream_of(q)),
          "qfa_quant_qkv_f32");
    r.o = empty({pb.B, pb.H, pb.N[0], pb.D}, at::kFloat, q);
    if (keep) r.o16 = empty({pb.B, pb.H, pb.N[0], pb.D}, at::kBFloat16, q);
    fwd_split_into(a, b, r.v16, r.o16, r.o, pb.lse_of(r.buf), causal, sm);
    return r;
  }
  quantize_pair_into(q, k, pb.view(r.buf, 0), pb.view(r.buf, 1));
  r.v16 = rows16(to(v_in, io_dtype(v_in)));
  r.o16 = empty({pb.B, pb.H, pb.N[0], pb.D}, r.v16.scalar_type(), q);
  fwd_split_into(pb.view(r.buf, 0), pb.view(r.buf, 1), r.v16, r.o16, Tensor(), pb.lse_of(r.buf), causal, sm);
  r.o = to(r.o16, q.scalar_type());
  return r;
}
struct QkvFn : torch::autograd::Function<QkvFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, bool causal, double sm) {
    const at::AutoDispatchBelowADInplaceOrView below;
    Kept r = qkv_forward(q, k, v, causal, sm, true);
    ctx->save_for_backward({r.buf, r.v16, r.o16});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["sm"] = sm;
    ctx->saved_data["dt"] = (int64_t)q.scalar_type() | (int64_t)k.scalar_type() << 8 | (int64_t)v.scalar_type() << 16;
    return r.o;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const int64_t dt = ctx->saved_data["dt"].toInt();
    const int64_t f = (int64_t)at::kFloat, all = f | f << 8 | f << 16;
    const Grads g = bwd_from(ctx, ctx->get_saved_variables(), grads[0], dt == all);
    return {to(g[0], (at::ScalarType)(dt & 255)), to(g[1], (at::ScalarType)(dt >> 8 & 255)),
            to(g[2], (at::ScalarType)(dt >> 16)), Tensor(), Tensor()};
  }
};
Tensor qkv_op(const Tensor &q, const Tensor &k, const Tensor &v, bool causal, double sm) {
  refuse_tangents({&q, &k, &v});
  require_gpu(q, k, v);
  TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k, v must be 4-D (Batch, Heads, Seq, Head_Dim)");
  TORCH_CHECK_VALUE(q.size(3) == k.size(3) && k.sizes() == v.sizes() && q.size(0) == k.size(0) && q.size(1) == k.size(1),
                    "shape mismatch: q ", q.sizes(), ", k ", k.sizes(), ", v ", v.sizes());
  if (wants_grad({&q, &k, &v})) return QkvFn::apply(q, k, v, causal, sm);
  return qkv_forward(q, k, v, causal, sm, false).o;
}
Tensor qkv(const Tensor &q, const Tensor &k, const Tensor &v, bool causal, double sm) {
  if (torch::jit::tracer::isTracing()) return Traced<decltype(qkv_op)>::call("quant_flash_attn_amd::qkv", q, k, v, causal, sm);
  return qkv_op(q, k, v, causal, sm);
}

// ---- q and an INT8 cache of keys and values
struct CacheKept : Kept {
  Tensor kc, ks, kz, kr;   // the keys as the kernels take them
};
Quantized keys_of(const Tensor &kc, const Tensor &ks, const Tensor &kz, const Tensor &kr) {
  return view_of({kc, ks, kz, kr});
}
// what the long-query kernels take of q and the cache: everything but O and the LSE
CacheKept cache_stage(const Tensor &q_in, const Tensor &kc, const Tensor &ks, const Tensor &kz, const Tensor &vc,
                      const Tensor &vs, const Tensor &vz) {
  const c10::DeviceGuard guard(q_in.device());
  const Tensor q = check_input(q_in);
  check_codes(kc, "k.codes");
  TORCH_CHECK_VALUE(kc.size(0) == q.size(0) && kc.size(1) == q.size(1) && kc.size(3) == q.size(3) && vc.sizes() == kc.sizes(),
                    "shape mismatch: q ", q.sizes(), ", k codes ", kc.sizes(), ", v codes ", vc.sizes());
  const int64_t nk = kc.size(0) * kc.size(1) * kc.size(2);
  const PairBuffer pb(q.size(0), q.size(1), q.size(2), 0, q.size(3));   // (no room for keys: they are the caller's)
  CacheKept r;
  r.buf = empty({pb.bytes}, at::kByte, q);
  r.kc = rows16(kc);
  r.kz = flat(kz, at::kChar, nk, "k.zero_point");
  require_gpu(q, kc, ks, kz, vc, vs, vz);
  check_codes(vc, "v.codes");
  // q quantized, K's row sums and fp32 scales and V dequantized, in one launch
  const Tensor v = rows16(vc), vzf = flat(vz, at::kChar, nk, "v.zero_point");
  TORCH_CHECK_TYPE(dtype_code(vs.scalar_type()) >= 0, "dtype and scale.dtype must be float16, bfloat16 or float32");
  const Tensor vsf = flat(vs, vs.scalar_type(), nk, "v.scale");
  const bool widen = is_io(ks.scalar_type());
  const Tensor ksf = widen ? flat(ks, ks.scalar_type(), nk, "k.scale") : flat(to(ks, at::kFloat), at::kFloat, nk, "k.scale");
  r.ks = widen ? empty({nk}, at::kFloat, q) : ksf;
  r.kr = empty({nk}, at::kInt, q);
  r.v16 = empty({kc.size(0), kc.size(1), kc.size(2), kc.size(3)}, io_dtype(q), q);
  const Quantized qq = pb.view(r.buf, 0);
  check(api.qfa_cache_stage_q(q.data_ptr(), dtype_code(q.scalar_type()), const_cast<int8_t *>(qq.codes), const_cast<float *>(qq.scale),
                              const_cast<int8_t *>(qq.zp), const_cast<int32_t *>(qq.rowsum), qq.N, QFA_STRIDES(q), qq.sb, qq.sh, qq.sn,
                              r.kc.data_ptr<int8_t>(), ksf.data_ptr(), dtype_code(ksf.scalar_type()), widen ? r.ks.data_ptr<float>() : nullptr,
                              r.kr.data_ptr<int32_t>(), v.data_ptr<int8_t>(), vsf.data_ptr(), dtype_code(vsf.scalar_type()),
                              vzf.data_ptr<int8_t>(), r.v16.data_ptr(), dtype_code(r.v16.scalar_type()), pb.B, pb.H, kc.size(2), (int)pb.D,
                              QFA_STRIDES(r.kc), QFA_STRIDES(v), stream_of(q)),
        "qfa_cache_stage_q");
  return r;
}
CacheKept cache_forward(const Tensor &q, const Tensor &kc, const Tensor &ks, const Tensor &kz, const Tensor &vc, const Tensor &vs,
                        const Tensor &vz, bool causal, double sm) {
  CacheKept r = cache_stage(q, kc, ks, kz, vc, vs, vz);
  const c10::DeviceGuard guard(q.device());
  const PairBuffer pb(q.size(0), q.size(1), q.size(2), 0, q.size(3));
  r.o16 = empty({pb.B, pb.H, pb.N[0], pb.D}, r.v16.scalar_type(), q);
  fwd_split_into(pb.view(r.buf, 0), keys_of(r.kc, r.ks, r.kz, r.kr), r.v16, r.o16, Tensor(), pb.lse_of(r.buf), causal, sm);
  r.o = to(r.o16, q.scalar_type());
  return r;
}
// Longest query block for qfa_attn_fwd_cache, which reads the cache once per 16 queries and leaves nothing for a backward;
// what it saves is a pass over V, the row sums of K and the casts, so the line depends on the keys per head_dim.  Measured
// against these passes and qfa_attn_fwd with the chip full (256 to 1024 heads), the queries at which both take as long:
//     keys / head_dim      1     2        4        8          16
//     head_dim 64                         100      115        130
//     head_dim 128               78       88       100-128    130
//     head_dim 256         49    66       95       118        135
// (at the old line of 128: 256 heads, 256 keys of 256: 95 against 51 us).  While one round of workgroups covers the call it
// wins up to 128 queries at any of these sizes (64 heads, 1024 keys of 256, 128 queries: 44 against 59 us; 32 heads: 25
// against 57).
int64_t cache_max_q(int64_t BH, int64_t Nq, int64_t Nk, int64_t D) {
  if (BH * ((Nq + 15) / 16) <= 512 || Nk >= 16 * D) return 128;
  return Nk >= 8 * D ? 112 : Nk >= 4 * D ? 80 : Nk >= 2 * D ? 64 : 48;
}
// Beyond that line the few launches of qfa_attn_fwd_cache still win where the work is small or the other path fills the chip badly
// (4 heads, 200 queries, 1000 keys of 64: 9 against 20 us).  Both paths' times in us as fitted to 6500 calls of 2 to 1024 heads, 8
// to 512 queries, 300 to 20000 keys (within 8 % in the mean): the short one takes what its memory or its blocks of 16 queries
// take, and loses by a last round of workgroups that is not full; the other one the pass over the cache and blocks of 128
// queries.  Calls are taken from the other path where that should gain 12 %: over all shapes the choice costs 0.4 - 1 % against
// the better path each time, where the line alone cost 3 - 6 %; the moved calls gain 1.4 times in the mean.  920 of them timed on
// both once more: 1.6 times, three lost more than 3 % (7 heads, 149 queries, 19668 keys of 256: 4.6 %).
bool cache_short_cheaper(int64_t BH, int64_t Nq, int64_t Nk, int64_t D) {
  struct Cost { double s0, s_byte, s_block, s_start, s_fill, l0, l_byte, l_block, l_idle, l_query; };
  static const Cost c64 = {9.8, 0.48, 11.4, 2.0, 0.37, 18.6, 0.84, 33.7, 0.1, 0.69}, c128 = {11.6, 0.56, 22.4, 6.1, 0.22, 20.4, 0.88, 51.9, 0.095, 0.42},
                    c256 = {15.3, 0.59, 41.9, 30.8, 0.22, 23.0, 0.88, 127.0, 0.0, 0.6};
  const Cost &c = D == 64 ? c64 : D == 128 ? c128 : c256;
  const int64_t nb = (Nq + 15) / 16, mb = (Nq + 127) / 128, wgs = BH * nb;
  const double n = (double)BH * (double)Nk * 1e-6, fill = wgs <= 512 ? (double)(wgs * (512 / wgs)) / 512.0 : (double)wgs / (double)((wgs + 511) / 512 * 512);
  const double blocks = (double)nb / std::pow(fill, c.s_fill), work = c.s_block * n * blocks + c.s_start * (double)BH * blocks * 1e-3;
  const double s = c.s0 + std::pow(std::pow(c.s_byte * n * (double)D, 4.0) + std::pow(work, 4.0), 0.25);
  const double idle = std::max(0.0, 1.0 - (double)(BH * mb) / 256.0);
  const double l = c.l0 + c.l_byte * n * (double)D + c.l_block * n * (double)mb * (1.0 + c.l_idle * idle) + c.l_query * (double)(BH * Nq * D) * 1e-6;
  return s < 0.88 * l;
}
enum class CachePath { Short, ShortBeyondLine, Long };
CachePath cache_path(const Tensor &q, const Tensor &kc) {
  const int64_t BH = q.size(0) * q.size(1), Nq = q.size(2), Nk = kc.size(2), D = q.size(3);
  if (Nq <= cache_max_q(BH, Nq, Nk, D)) return CachePath::Short;
  const bool cheaper = Nq <= 512 && BH > 0 && Nk > 0 && cache_short_cheaper(BH, Nq, Nk, D);   // (as far as was measured)
  return cheaper ? CachePath::ShortBeyondLine : CachePath::Long;
}
Tensor cache_short(const Tensor &q_in, const Tensor &kc_in, const Tensor &ks_in, const Tensor &kz, const Tensor &vc_in,
                   const Tensor &vs_in, const Tensor &vz, bool causal, double sm, float *lse = nullptr) {
  const c10::DeviceGuard guard(q_in.device());
  const Tensor q = check_input(q_in);
  check_codes(kc_in, "k.codes");
  check_codes(vc_in, "v.codes");
  const Tensor kc = rows16(kc_in), vc = rows16(vc_in);
  const int64_t B = q.size(0), H = q.size(1), Nq = q.size(2), D = q.size(3), Nk = kc.size(2), n = B * H * Nk;
  const bool as_is = ks_in.scalar_type() == vs_in.scalar_type() && dtype_code(ks_in.scalar_type()) >= 0;
  const at::ScalarType sdt = as_is ? ks_in.scalar_type() : at::kFloat;
  const Tensor ks = flat(to(ks_in, sdt), sdt, n, "k.scale"), vs = flat(to(vs_in, sdt), sdt, n, "v.scale"),
               kzf = flat(kz, at::kChar, n, "k.zero_point"), vzf = flat(vz, at::kChar, n, "v.zero_point");
  Tensor o = empty({B, H, Nq, D}, q.scalar_type(), q), ws;
  const int64_t ws_bytes = api.qfa_attn_fwd_cache_workspace_bytes(B, H, Nq, Nk, (int)D);
  if (ws_bytes > 0) ws = empty({ws_bytes}, at::kByte, q);
  check(api.qfa_attn_fwd_cache_lse(q.data_ptr(), dtype_code(q.scalar_type()), kc.data_ptr<int8_t>(), ks.data_ptr(),
                                   kzf.data_ptr<int8_t>(), vc.data_ptr<int8_t>(), vs.data_ptr(), vzf.data_ptr<int8_t>(),
                                   dtype_code(sdt), o.data_ptr(), lse, B, H, Nq, Nk, (int)D, QFA_STRIDES(q), QFA_STRIDES(kc),
                                   QFA_STRIDES(vc), QFA_STRIDES(o), (float)sm, causal, ws_bytes > 0 ? ws.data_ptr() : nullptr,
                                   ws_bytes, stream_of(q)),
        "qfa_attn_fwd_cache");
  return o;
}

struct CacheFn : torch::autograd::Function<CacheFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k_fp16, const Tensor &v_fp16, const Tensor &kc,
                        const Tensor &ks, const Tensor &kz, const Tensor &vc, const Tensor &vs, const Tensor &vz, bool causal,
                        double sm) {
    const at::AutoDispatchBelowADInplaceOrView below;
    // what a call without a gradient returns, bit for bit (a forward that is computed again for its gradient, as activation
    // checkpointing does)
    const CachePath path = cache_path(q, kc);
    CacheKept r;
    if (path == CachePath::ShortBeyondLine) {
      // O and the LSE of the short kernel serve the backward too, which wants the staged keys and values beside them
      r = cache_stage(q, kc, ks, kz, vc, vs, vz);
      const PairBuffer pb(q.size(0), q.size(1), q.size(2), 0, q.size(3));
      r.o = cache_short(q, kc, ks, kz, vc, vs, vz, causal, sm, pb.lse_of(r.buf));
      r.o16 = to(r.o, io_dtype(q));
    } else {
      r = cache_forward(q, kc, ks, kz, vc, vs, vz, causal, sm);
      // (the backward takes O, LSE and V of the long-query path here)
      if (path == CachePath::Short) r.o = cache_short(q, kc, ks, kz, vc, vs, vz, causal, sm);
    }
    ctx->save_for_backward({r.buf, r.v16, r.o16, r.kc, r.ks, r.kz, r.kr});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["sm"] = sm;
    ctx->saved_data["dt"] =
        (int64_t)q.scalar_type() | (int64_t)k_fp16.scalar_type() << 8 | (int64_t)v_fp16.scalar_type() << 16;
    return r.o;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const variable_list s = ctx->get_saved_variables();
    const Quantized k = keys_of(s[3], s[4], s[5], s[6]);
    const Tensor &buf = s[0], &v16 = s[1], &o16 = s[2];
    const PairBuffer pb(o16.size(0), o16.size(1), o16.size(2), 0, o16.size(3));
    const c10::DeviceGuard guard(v16.device());
    const Grads g = bwd_of(pb.view(buf, 0), k, v16, o16, grads[0], pb.lse_of(buf), ctx->saved_data["causal"].toBool(),
                           ctx->saved_data["sm"].toDouble(), true);
    const int64_t dt = ctx->saved_data["dt"].toInt();
    variable_list out(11);
    for (int i = 0; i < 3; ++i) out[i] = to(g[i], (at::ScalarType)(dt >> (8 * i) & 255));
    return out;
  }
};
Tensor cache_op(const Tensor &q, const Tensor &k_fp16, const Tensor &v_fp16, const Tensor &kc, const Tensor &ks,
                const Tensor &kz, const Tensor &vc, const Tensor &vs, const Tensor &vz, bool causal, double sm) {
  refuse_tangents({&q, &k_fp16, &v_fp16});
  require_gpu(q, kc, ks, kz, vc, vs, vz);
  TORCH_CHECK_VALUE(q.dim() == 4 && kc.dim() == 4 && kc.sizes() == vc.sizes() && q.size(3) == kc.size(3) &&
                        q.size(0) == kc.size(0) && q.size(1) == kc.size(1),
                    "shape mismatch: q ", q.sizes(), ", k codes ", kc.sizes(), ", v codes ", vc.sizes());
  if (wants_grad({&q, &k_fp16, &v_fp16})) return CacheFn::apply(q, k_fp16, v_fp16, kc, ks, kz, vc, vs, vz, causal, sm);
  if (cache_path(q, kc) != CachePath::Long) return cache_short(q, kc, ks, kz, vc, vs, vz, causal, sm);
  return cache_forward(q, kc, ks, kz, vc, vs, vz, causal, sm).o;
}
Tensor cache(const Tensor &q, const Tensor &k_fp16, const Tensor &v_fp16, const Tensor &kc, const Tensor &ks,
             const Tensor &kz, const Tensor &vc, const Tensor &vs, const Tensor &vz, bool causal, double sm) {
  if (torch::jit::tracer::isTracing())
    return Traced<decltype(cache_op)>::call("quant_flash_attn_amd::quantized_kv", q, k_fp16, v_fp16, kc, ks, kz, vc, vs, vz,
                                            causal, sm);
  return cache_op(q, k_fp16, v_fp16, kc, ks, kz, vc, vs, vz, causal, sm);
}

// ------------------------------------------------------------------------------------------- shared K = V
std::tuple<Tensor, Tensor> skv_fwd(const Tensor &q_in, const Tensor &codes_in, const Tensor &scale_in, const Tensor &zp_in,
                                   double sm) {
  TORCH_CHECK_TYPE(is_io(q_in.scalar_type()), "q must be bfloat16 or float16, got ", q_in.scalar_type());
  check_codes(codes_in, "codes");
  require_gpu(q_in, codes_in, scale_in, zp_in);
  TORCH_CHECK_VALUE(q_in.dim() == 4 && codes_in.size(0) == q_in.size(0) && codes_in.size(1) == q_in.size(1) &&
                        codes_in.size(3) == q_in.size(3),
                    "shape mismatch: q ", q_in.sizes(), ", codes ", codes_in.sizes());
  const c10::DeviceGuard guard(q_in.device());
  const int64_t B = q_in.size(0), H = q_in.size(1), Nq = q_in.size(2), D = q_in.size(3), Nk = codes_in.size(2);
  const bool as_is = scale_in.scalar_type() == at::kFloat || scale_in.scalar_type() == at::kHalf ||
                     scale_in.scalar_type() == q_in.scalar_type();
  const Tensor s = as_is ? scale_in : scale_in.to(at::kFloat);
  const Tensor scale = flat(s, s.scalar_type(), B * H * Nk, "scale"), zp = flat(zp_in, at::kChar, B * H * Nk, "zero_point");
  const Tensor q = rows16(q_in), codes = rows16(codes_in);
  Tensor o = empty({B, H, Nq, D}, q.scalar_type(), q), lse = empty({B, H, Nq}, at::kFloat, q);
  // scratch for the split over keys the library uses when B*H alone cannot fill the GPU (0: no split)
  const int64_t ws_bytes = api.qfa_attn_fwd_shared_kv_workspace_bytes(B, H, Nq, Nk, (int)D);
  Tensor ws;
  if (ws_bytes > 0) ws = empty({ws_bytes}, at::kByte, q);
  check(api.qfa_attn_fwd_shared_kv(q.data_ptr(), codes.data_ptr<int8_t>(), scale.data_ptr(), dtype_code(scale.scalar_type()),
                                   zp.data_ptr<int8_t>(), o.data_ptr(), lse.data_ptr<float>(), dtype_code(q.scalar_type()), B,
                                   H, Nq, Nk, (int)D, QFA_STRIDES(q), QFA_STRIDES(codes), QFA_STRIDES(o), (float)sm,
                                   ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes, stream_of(q)),
        "qfa_attn_fwd_shared_kv");
  return {o, lse};
}

std::tuple<Tensor, Tensor> skv_bwd(const Tensor &q_in, const Tensor &codes_in, const Tensor &scale_in, const Tensor &zp_in,
                                   const Tensor &o_in, const Tensor &do_in, const Tensor &lse_in, double sm,
                                   at::ScalarType grad_dtype, const std::optional<Tensor> &grad_scale_in, bool split,
                                   bool direct = false) {
  TORCH_CHECK_TYPE(direct || (q_in.scalar_type() == at::kHalf && o_in.scalar_type() == at::kHalf),
                   "the shared-KV backward kernel computes in float16: q and o must be float16");
  TORCH_CHECK_TYPE(is_io(grad_dtype), "grad_dtype must be float16 or bfloat16, got ", grad_dtype);
  check_codes(codes_in, "codes");
  TORCH_CHECK_VALUE(q_in.dim() == 4 && codes_in.size(0) == q_in.size(0) && codes_in.size(1) == q_in.size(1) &&
                        codes_in.size(3) == q_in.size(3) && o_in.sizes() == q_in.sizes() && do_in.sizes() == q_in.sizes(),
                    "shape mismatch between q / o / do and the codes");
  require_gpu(q_in, codes_in, scale_in, zp_in, o_in, do_in, lse_in);
  const c10::DeviceGuard guard(q_in.device());
  const int64_t B = q_in.size(0), H = q_in.size(1), Nq = q_in.size(2), D = q_in.size(3), Nk = codes_in.size(2);
  Tensor grad_scale;
  if (grad_scale_in) {
    require_gpu(q_in, *grad_scale_in);
    grad_scale = flat(*grad_scale_in, at::kFloat, 1, "grad_scale");
  }
  const bool as_is = scale_in.scalar_type() == at::kFloat || scale_in.scalar_type() == at::kHalf;
  const Tensor s = as_is ? scale_in : scale_in.to(at::kFloat);
  const Tensor scale = flat(s, s.scalar_type(), B * H * Nk, "scale"), zp = flat(zp_in, at::kChar, B * H * Nk, "zero_point"),
               lse = flat(lse_in, at::kFloat, B * H * Nq, "lse");
  const Tensor q = rows16(q_in), codes = rows16(codes_in), o = rows16(o_in), dout = rows16(to(do_in, direct ? io_dtype(do_in) : at::kHalf));
  Tensor dq = empty({B, H, Nq, D}, grad_dtype, q), dkv = empty({B, H, Nk, D}, grad_dtype, q);
  // scratch for the split over keys where B*H alone cannot fill the GPU (0: no split)
  const Tensor ws = optional_scratch(split ? api.qfa_attn_bwd_shared_kv_workspace_bytes(B, H, Nq, Nk, D) : 0, q);
  if (direct) {
    check(api.qfa_attn_bwd_shared_kv_direct(q.data_ptr(), codes.data_ptr<int8_t>(), scale.data_ptr(), dtype_code(scale.scalar_type()),
                                            zp.data_ptr<int8_t>(), o.data_ptr(), dout.data_ptr(), lse.data_ptr<float>(),
                                            dq.data_ptr(), dkv.data_ptr(), dtype_code(q.scalar_type()),
                                            dtype_code(dout.scalar_type()), dtype_code(grad_dtype), B, H, Nq, Nk, (int)D,
                                            QFA_STRIDES(q), QFA_STRIDES(codes), QFA_STRIDES(o), QFA_STRIDES(dout),
                                            QFA_STRIDES(dq), QFA_STRIDES(dkv), (float)sm, data_of(ws), bytes_of(ws),
                                            stream_of(q)),
          "qfa_attn_bwd_shared_kv_direct");
    return {dq, dkv};
  }
  check(api.qfa_attn_bwd_shared_kv_split(q.data_ptr(), codes.data_ptr<int8_t>(), scale.data_ptr(), dtype_code(scale.scalar_type()),
                                   zp.data_ptr<int8_t>(), o.data_ptr(), dout.data_ptr(), lse.data_ptr<float>(),
                                   dq.data_ptr(), dkv.data_ptr(), QFA_F16, dtype_code(grad_dtype),
                                   grad_scale.defined() ? grad_scale.data_ptr<float>() : nullptr, B, H, Nq, Nk, (int)D,
                                   QFA_STRIDES(q), QFA_STRIDES(codes), QFA_STRIDES(o), QFA_STRIDES(dout), QFA_STRIDES(dq),
                                   QFA_STRIDES(dkv), (float)sm, data_of(ws), bytes_of(ws), stream_of(q)),
        "qfa_attn_bwd_shared_kv_split");
  return {dq, dkv};
}

// (dO * 2^k as float16, 2^-k as a one-element float32 tensor) for the binary16 backward kernels: two launches, nothing
// synchronises
// and q and o (undefined or) in float16: bf16 ones are cast by the second of these launches, which takes dense tensors
struct Normalised { Tensor dout, back, q, o; };
Normalised normalise(const Tensor &grad_in, const Tensor &scale_in, const Tensor &q, const Tensor &o) {
  require_gpu(grad_in, scale_in);
  const c10::DeviceGuard guard(grad_in.device());
  // (a gradient that is not 16-bit is not what autograd hands over for a 16-bit output; bf16 keeps the range)
  const Tensor grad = to(grad_in, io_dtype(grad_in)).contiguous();
  const bool as_is = scale_in.scalar_type() == at::kFloat || scale_in.scalar_type() == at::kHalf;
  Tensor scale = (as_is ? scale_in : scale_in.to(at::kFloat)).contiguous();
  if (reinterpret_cast<uintptr_t>(scale.data_ptr()) % 16) scale = scale.clone();   // a view that starts inside an allocation
  Tensor do16 = empty(grad.sizes(), at::kHalf, grad), back = empty({1}, at::kFloat, grad);
  const Tensor ws = empty({api.qfa_dout_normalise_workspace_bytes()}, at::kByte, grad);
  const void *x[2] = {nullptr, nullptr};
  void *y[2] = {nullptr, nullptr};
  int casts = 0;
  auto half = [&](const Tensor &t) -> Tensor {
    if (!t.defined()) return t;
    if (t.scalar_type() != at::kBFloat16 || !t.is_contiguous() || t.numel() != grad.numel() || t.device() != grad.device() ||
        reinterpret_cast<uintptr_t>(t.data_ptr()) % 16)
      return to(t, at::kHalf);
    const Tensor h = empty(t.sizes(), at::kHalf, t);
    x[casts] = t.data_ptr();
    y[casts++] = h.data_ptr();
    return h;
  };
  const Tensor q16 = half(q), o16 = half(o);
  check(api.qfa_dout_normalise_cast(grad.data_ptr(), dtype_code(grad.scalar_type()), grad.numel(), scale.data_ptr(),
                                    dtype_code(scale.scalar_type()), scale.numel(), ws.data_ptr(), do16.data_ptr(),
                                    back.data_ptr<float>(), x[0], y[0], x[1], y[1], stream_of(grad)),
        "qfa_dout_normalise");
  return {do16, back, q16, o16};
}
std::tuple<Tensor, Tensor> normalised_dout(const Tensor &grad, const Tensor &scale) {
  const Normalised n = normalise(grad, scale, Tensor(), Tensor());
  return {n.dout, n.back};
}

// The reference's operator with the shared-KV kernels (short query blocks, Q as it comes)
struct SharedFn : torch::autograd::Function<SharedFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &kv_fp16, const Tensor &codes, const Tensor &scale,
                        const Tensor &zp, double sm) {
    const at::AutoDispatchBelowADInplaceOrView below;
    auto [o, lse] = skv_fwd(q, codes, scale, zp, sm);
    ctx->save_for_backward({q, codes, scale, zp, o, lse});
    ctx->saved_data["sm"] = sm;
    ctx->saved_data["kv_dtype"] = (int64_t)kv_fp16.scalar_type();
    return o;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const variable_list s = ctx->get_saved_variables();
    const Tensor &q = s[0], &o = s[4];
    // The backward kernels compute in binary16, and what they feed the matrix pipe is not dO but
    // sm_scale * p * (dP - delta) and that times the key's scale: with dO as it comes, ordinary small
    // gradients land in binary16's subnormals (or flush to zero) there.  dQ and dKV are linear in dO,
    // so dO is handed over scaled by a power of two chosen on the device (no synchronisation) from
    // its largest magnitude and from the largest key scale, and the kernels scale dQ and dKV back
    // while they round them.  q and o convert exactly from bf16 (more mantissa, values of order one).
    // Kernels whose workgroups hold all rows that they need do that themselves.
    const double sm = ctx->saved_data["sm"].toDouble();
    Tensor dq, dkv;
    if (is_io(o.scalar_type()) && o.scalar_type() == q.scalar_type() && api.qfa_attn_bwd_shared_kv_is_direct(q.size(2), (int)q.size(3))) {
      std::tie(dq, dkv) = skv_bwd(q, s[1], s[2], s[3], o, grads[0], s[5], sm, q.scalar_type(), std::nullopt, true, true);
    } else {
      const Normalised n = normalise(grads[0], s[2], q, o);
      std::tie(dq, dkv) = skv_bwd(n.q, s[1], s[2], s[3], n.o, n.dout, s[5], sm, q.scalar_type(), n.back, true);
    }
    return {dq, to(dkv, (at::ScalarType)ctx->saved_data["kv_dtype"].toInt()), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
// ... and with the INT8-score kernels (long query blocks): Q quantized per token, K = the caller's codes with the scale
// exactly as stored, V = dequant(kv) (quant_flash_attn.py:65)
struct SharedLongFn : torch::autograd::Function<SharedLongFn> {
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &kv_fp16, const Tensor &codes, const Tensor &scale,
                        const Tensor &zp, double sm) {
    const at::AutoDispatchBelowADInplaceOrView below;
    CacheKept r = cache_forward(q, codes, scale, zp, codes, scale, zp, false, sm);
    ctx->save_for_backward({r.buf, r.v16, r.o16, r.kc, r.ks, r.kz, r.kr});
    ctx->saved_data["sm"] = sm;
    ctx->saved_data["q_dtype"] = (int64_t)q.scalar_type();
    ctx->saved_data["kv_dtype"] = (int64_t)kv_fp16.scalar_type();
    return r.o;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const at::AutoDispatchBelowADInplaceOrView below;
    const variable_list s = ctx->get_saved_variables();
    const Tensor &buf = s[0], &v16 = s[1], &o16 = s[2];
    const PairBuffer pb(o16.size(0), o16.size(1), o16.size(2), 0, o16.size(3));
    const c10::DeviceGuard guard(v16.device());
    const Grads g = bwd_of(pb.view(buf, 0), keys_of(s[3], s[4], s[5], s[6]), v16, o16, grads[0], pb.lse_of(buf), false,
                           ctx->saved_data["sm"].toDouble(), true);
    // quant_flash_attn.py:161 (dk already carries sm_scale): one pass, added in fp32 and rounded once
    check(api.qfa_sum_grads(g[1].data_ptr(), g[2].data_ptr(), g[1].data_ptr(), dtype_code(g[1].scalar_type()), g[1].numel(),
                            stream_of(g[1])),
          "qfa_sum_grads");
    return {to(g[0], (at::ScalarType)ctx->saved_data["q_dtype"].toInt()),
            to(g[1], (at::ScalarType)ctx->saved_data["kv_dtype"].toInt()), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
// max_q: longest query block for the shared-KV kernels at this head dimension
Tensor shared_op(const Tensor &q, const Tensor &kv_fp16, const Tensor &codes, const Tensor &scale, const Tensor &zp, double sm,
                 int64_t max_q) {
  refuse_tangents({&q, &kv_fp16});
  require_gpu(q, codes, scale, zp);
  TORCH_CHECK_VALUE(q.dim() == 4 && codes.sizes() == kv_fp16.sizes() && codes.dim() == 4 && q.size(3) == codes.size(3),
                    "shape mismatch: q ", q.sizes(), ", kv ", kv_fp16.sizes(), ", codes ", codes.sizes());
  const bool short_q = q.size(2) <= max_q && is_io(q.scalar_type()), grad = wants_grad({&q, &kv_fp16});
  if (short_q) return grad ? SharedFn::apply(q, kv_fp16, codes, scale, zp, sm) : std::get<0>(skv_fwd(q, codes, scale, zp, sm));
  return grad ? SharedLongFn::apply(q, kv_fp16, codes, scale, zp, sm)
              : cache_forward(q, codes, scale, zp, codes, scale, zp, false, sm).o;
}
Tensor shared(const Tensor &q, const Tensor &kv_fp16, const Tensor &codes, const Tensor &scale, const Tensor &zp, double sm,
              int64_t max_q) {
  if (torch::jit::tracer::isTracing())
    return Traced<decltype(shared_op)>::call("quant_flash_attn_amd::shared_kv", q, kv_fp16, codes, scale, zp, sm, max_q);
  return shared_op(q, kv_fp16, codes, scale, zp, sm, max_q);
}

}  // namespace

// (no backend key: the operators attach their autograd nodes themselves)
TORCH_LIBRARY(quant_flash_attn_amd, m) {
  m.def("qkv(Tensor q, Tensor k, Tensor v, bool causal, float sm_scale) -> Tensor", &qkv_op);
  m.def("quantized_kv(Tensor q, Tensor k_fp16, Tensor v_fp16, Tensor k_codes, Tensor k_scale, Tensor k_zero_point, "
        "Tensor v_codes, Tensor v_scale, Tensor v_zero_point, bool causal, float sm_scale) -> Tensor", &cache_op);
  m.def("shared_kv(Tensor q, Tensor kv_fp16, Tensor codes, Tensor scale, Tensor zero_point, float sm_scale, int max_q) -> Tensor",
        &shared_op);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  typedef py::call_guard<py::gil_scoped_release> nogil;
  m.def("init", &init);
  m.def("quant", &quant, nogil());
  m.def("quant_attn", &quant_attn, nogil());
  m.def("quant_attn_pair", &quant_attn_pair, nogil());
  m.def("dequant", &dequant, nogil());
  m.def("rowsum", &rowsum, nogil());
  m.def("attn_fwd", &attn_fwd, nogil());
  m.def("attn_bwd", &attn_bwd, nogil());
  m.def("qkv", &qkv, nogil());
  m.def("cache", &cache, nogil());
  m.def("skv_fwd", &skv_fwd, nogil());
  // (what qfa_attn_bwd_shared_kv returns, bit for bit: not split)
  m.def("skv_bwd", [](const Tensor &q, const Tensor &codes, const Tensor &scale, const Tensor &zp, const Tensor &o, const Tensor &dout,
                      const Tensor &lse, double sm, at::ScalarType grad_dtype, const std::optional<Tensor> &grad_scale) {
    return skv_bwd(q, codes, scale, zp, o, dout, lse, sm, grad_dtype, grad_scale, false);
  }, nogil());
  m.def("normalised_dout", &normalised_dout, nogil());
  m.def("shared", &shared, nogil());
}
