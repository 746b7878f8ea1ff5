// Autograd functions of the LoRA projections and of packed-row attention over the artk C-ABI, for PyTorch-ROCm.
//
// Everything around the kernels of one projection or attention call (layout checks, output and workspace
// allocation, argument tables, the autograd node) used to be Python: 300 us per step for q|k|v of a short row whose
// kernels take 60.  Here it is a few microseconds of C++ each way, without the interpreter lock.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include "../../include/artk.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ValueError for an argument error, art_amd._lib.ArtkError for a hipError_t, as art_amd._lib.check raises them.
void check(int32_t rc) {
  if (rc == 0) return;
  const std::string text = artk_last_error();  // (of this thread)
  TORCH_CHECK_VALUE(rc > 0, "artk error ", rc, ": ", text);
  py::gil_scoped_acquire gil;
  const py::object type = py::module_::import("art_amd._lib").attr("ArtkError");
  const py::object error = type(rc, py::bytes(text).attr("decode")("utf-8", "replace"));
  PyErr_SetObject(type.ptr(), error.ptr());
  python_error e;
  e.persist();
  throw e;
}

void need(const Tensor& t, const char* name, at::ScalarType dtype, at::IntArrayRef shape) {
  TORCH_CHECK_VALUE(t.defined() && t.is_cuda(), name, " must live on the GPU; there is no CPU path");
  TORCH_CHECK_TYPE(t.scalar_type() == dtype, name, " must be ", dtype, ", got ", t.scalar_type());
  TORCH_CHECK_VALUE(t.sizes() == shape, name, " must have shape ", shape, ", got ", t.sizes());
  TORCH_CHECK_VALUE(t.is_contiguous(), name, " must be contiguous");
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

Tensor make(const Tensor& like, at::IntArrayRef shape, at::ScalarType dtype) {
  return at::empty(shape, like.options().dtype(dtype));
}
Tensor workspace(const Tensor& like, size_t bytes) {
  return make(like, {(int64_t)(bytes > 256 ? bytes : 256)}, at::kByte);
}

// `t` as contiguous bf16 rows [-1, last dimension].
Tensor rows_bf16(const Tensor& t) { return t.reshape({-1, t.size(-1)}).to(at::kBFloat16).contiguous(); }

// NF4 weight: the tensors behind artk_nf4_t, owned by the caller's module.
struct Nf4 {
  Tensor packed, absmax, absmax_q, code2, absmax2;
  double offset = 0;
  int64_t blocksize = 64, out = 0, in = 0;
  artk_nf4_t view() const {
    auto p = [](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
    artk_nf4_t v{};
    v.packed = p(packed);
    v.absmax = (const float*)p(absmax);
    v.absmax_q = p(absmax_q);
    v.code2 = (const float*)p(code2);
    v.absmax2 = (const float*)p(absmax2);
    v.offset = (float)offset;
    v.blocksize = (int32_t)blocksize;
    return v;
  }
  void dequantise(bool transposed, const Tensor& into) const {
    const artk_nf4_t v = view();
    if (transposed)
      check(artk_nf4_dequant_t(v.packed, v.absmax, v.absmax_q, v.code2, v.absmax2, v.offset, out, in, v.blocksize,
                               into.data_ptr(), stream_of(into)));
    else
      check(artk_nf4_dequant(v.packed, v.absmax, v.absmax_q, v.code2, v.absmax2, v.offset, out * in, v.blocksize,
                             into.data_ptr(), stream_of(into)));
  }
};

// The transposed copies of frozen weights as art_amd.ops.transposed_weight keeps them (made there if need be).
std::vector<Tensor> transposed_weights(const std::vector<Tensor>& W) {
  py::gil_scoped_acquire gil;
  std::vector<Tensor> out;
  try {
    const py::object find = py::module_::import("art_amd.ops").attr("transposed_weight");
    for (const Tensor& w : W) out.push_back(find(w).cast<Tensor>());
  } catch (py::error_already_set& e) {  // on to the caller as the Python exception that it is
    e.restore();
    python_error error;
    error.persist();
    throw error;
  }
  return out;
}

// What a call of n projections over one input brings besides the differentiable tensors.
struct LoraArgs {
  std::vector<Tensor> W, W_t;               // frozen weights and their transposed copies (W_t: empty where not all exist)
  std::vector<std::optional<Tensor>> bias;  // frozen
  std::shared_ptr<Nf4> nf4;                 // one projection on 4-bit codes instead of W
  double scale = 1;
};

// y_i = x W_i^T + bias_i + scale (x A_i^T) B_i^T with gradients for x, A_i, B_i.
struct LoraFunction : torch::autograd::Function<LoraFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, at::TensorList A, at::TensorList B,
                               const LoraArgs& a) {
    const int n = (int)A.size();
    TORCH_CHECK_VALUE(n >= 1 && n <= ARTK_LORA_MULTI_MAX && B.size() == A.size() && a.bias.size() == A.size() &&
                          (a.nf4 ? n == 1 : a.W.size() == A.size()),
                      "1 to ", ARTK_LORA_MULTI_MAX, " projections, one weight, A, B and bias each");
    TORCH_CHECK_VALUE(x.is_cuda(), "x must live on the GPU; there is no CPU path");
    c10::OptionalDeviceGuard guard(x.device());
    const Tensor x2 = rows_bf16(x);
    const int64_t T = x2.size(0), in = x2.size(1);
    artk_lora_proj_t proj[ARTK_LORA_MULTI_MAX] = {};
    variable_list saved{x2}, ys;
    std::vector<Tensor> A16, B16, xa;
    Tensor W_nf4;
    if (a.nf4) {
      TORCH_CHECK_VALUE(a.nf4->in == in && a.nf4->out == B[0].size(0), "NF4 weight has shape [", a.nf4->out, ", ",
                        a.nf4->in, "], expected [", B[0].size(0), ", ", in, "]");
      TORCH_CHECK_VALUE(in % a.nf4->blocksize == 0, "the input size must be a multiple of the quantisation block size");
      W_nf4 = make(x2, {a.nf4->out, in}, at::kBFloat16);   // exists for this call only
      a.nf4->dequantise(false, W_nf4);
    }
    std::vector<int64_t> lead(x.sizes().begin(), x.sizes().end());
    for (int i = 0; i < n; ++i) {
      A16.push_back(A[i].to(at::kBFloat16).contiguous());
      B16.push_back(B[i].to(at::kBFloat16).contiguous());
      const Tensor& W = a.nf4 ? W_nf4 : a.W[i];
      const int64_t out = B16[i].size(0), r = B16[i].size(1);
      need(W, "W", at::kBFloat16, {out, in});
      need(A16[i], "A", at::kBFloat16, {r, in});
      need(B16[i], "B", at::kBFloat16, {out, r});
      const Tensor y = make(x2, {T, out}, at::kBFloat16);
      xa.push_back(make(x2, {T, r}, at::kFloat));
      artk_lora_proj_t& p = proj[i];
      p.W = W.data_ptr();
      p.A = A16[i].data_ptr();
      p.B = B16[i].data_ptr();
      if (a.bias[i]) {
        need(*a.bias[i], "bias", at::kBFloat16, {out});
        p.bias = a.bias[i]->data_ptr();
      }
      p.y = y.data_ptr();
      p.xa = xa[i].data_ptr<float>();
      p.out = out;
      p.r = (int32_t)r;
      lead.back() = out;
      ys.push_back(y.view(lead));
    }
    const Tensor ws = workspace(x2, artk_lora_linear_multi_fwd_workspace_bytes(T, in, proj, n));
    check(artk_lora_linear_multi_fwd(x2.data_ptr(), proj, n, (float)a.scale, T, in, ws.data_ptr(), ws.numel(),
                                     stream_of(x2)));
    saved.insert(saved.end(), A16.begin(), A16.end());
    saved.insert(saved.end(), B16.begin(), B16.end());
    saved.insert(saved.end(), xa.begin(), xa.end());
    // Frozen storage that outlives the call (codes, transposed copies) rides on the node itself: as saved tensors,
    // hooks that move activations to the host would copy it for every projection.
    if (a.nf4) {
      ctx->saved_data["frozen"] =
          variable_list{a.nf4->packed, a.nf4->absmax, a.nf4->absmax_q, a.nf4->code2, a.nf4->absmax2};
      ctx->saved_data["offset"] = a.nf4->offset;
      ctx->saved_data["blocksize"] = a.nf4->blocksize;
    } else {
      ctx->saved_data["frozen"] = a.W_t;
      if (a.W_t.empty()) ctx->saved_data["W"] = a.W;  // the backward asks for the copies
      saved.insert(saved.end(), a.W.begin(), a.W.end());  // (their versions are checked with the rest)
    }
    ctx->save_for_backward(saved);
    ctx->saved_data["n"] = (int64_t)n;
    ctx->saved_data["nf4"] = a.nf4 != nullptr;
    ctx->saved_data["scale"] = a.scale;
    ctx->saved_data["x_shape"] = x.sizes();
    ctx->saved_data["x_type"] = (int64_t)x.scalar_type();
    std::vector<int64_t> types;
    for (const auto& list : {A, B})
      for (const Tensor& t : list) types.push_back((int64_t)t.scalar_type());
    ctx->saved_data["types"] = types;
    return ys;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const int n = (int)ctx->saved_data["n"].toInt();
    const auto types = ctx->saved_data["types"].toIntVector();
    const bool on_codes = ctx->saved_data["nf4"].toBool();
    const Tensor& x2 = saved[0];
    c10::OptionalDeviceGuard guard(x2.device());
    const int64_t T = x2.size(0), in = x2.size(1);
    auto t = ctx->saved_data["frozen"].toTensorVector();
    Tensor W_t;
    if (on_codes) {
      const Nf4 w{t[0], t[1], t[2], t[3], t[4], ctx->saved_data["offset"].toDouble(),
                  ctx->saved_data["blocksize"].toInt(), saved[1 + n].size(0), in};
      W_t = make(x2, {in, w.out}, at::kBFloat16);
      w.dequantise(true, W_t);
    } else {
      if (t.empty()) t = transposed_weights(ctx->saved_data["W"].toTensorVector());
      TORCH_CHECK((int)t.size() == n, "a transposed copy for each weight is needed");
    }
    artk_lora_proj_t proj[ARTK_LORA_MULTI_MAX] = {};
    std::vector<Tensor> g2, dA, dB;
    bool all_bf16 = true;
    for (int64_t t : types) all_bf16 = all_bf16 && t == (int64_t)at::kBFloat16;
    const at::ScalarType gt = all_bf16 ? at::kBFloat16 : at::kFloat;
    for (int i = 0; i < n; ++i) {
      const Tensor &A = saved[1 + i], &B = saved[1 + n + i], &xa = saved[1 + 2 * n + i];
      const Tensor& Wt = on_codes ? W_t : t[i];
      const int64_t out = B.size(0), r = B.size(1);
      g2.push_back(rows_bf16(grads[i]));
      need(Wt, "W_t", at::kBFloat16, {in, out});
      dA.push_back(make(x2, {r, in}, gt));
      dB.push_back(make(x2, {out, r}, gt));
      artk_lora_proj_t& p = proj[i];
      p.W_t = Wt.data_ptr();
      p.A = A.data_ptr();
      p.B = B.data_ptr();
      p.g = g2[i].data_ptr();
      p.xa = xa.data_ptr<float>();
      p.dA = (float*)dA[i].data_ptr();
      p.dB = (float*)dB[i].data_ptr();
      p.out = out;
      p.r = (int32_t)r;
    }
    const Tensor dx = make(x2, {T, in}, at::kBFloat16);
    const Tensor ws = workspace(x2, artk_lora_linear_multi_bwd_workspace_bytes(T, in, proj, n));
    check(artk_lora_linear_multi_bwd_typed(x2.data_ptr(), proj, n, (float)ctx->saved_data["scale"].toDouble(), T, in,
                                           all_bf16, dx.data_ptr(), ws.data_ptr(), ws.numel(), stream_of(x2)));
    variable_list out{dx.view(ctx->saved_data["x_shape"].toIntVector())
                          .to((at::ScalarType)ctx->saved_data["x_type"].toInt())};
    for (int i = 0; i < n; ++i) out.push_back(dA[i].to((at::ScalarType)types[i]));
    for (int i = 0; i < n; ++i) out.push_back(dB[i].to((at::ScalarType)types[n + i]));
    out.emplace_back();
    return out;
  }
};

std::vector<Tensor> lora_multi(const Tensor& x, std::vector<Tensor> W, std::vector<Tensor> W_t, std::vector<Tensor> A,
                               std::vector<Tensor> B, std::vector<std::optional<Tensor>> bias, double scale) {
  LoraArgs a;
  a.W = std::move(W);
  a.W_t = std::move(W_t);
  a.bias = std::move(bias);
  a.scale = scale;
  return LoraFunction::apply(x, at::TensorList(A), at::TensorList(B), a);
}

Tensor lora_nf4(const Tensor& x, const Tensor& packed, std::optional<Tensor> absmax, std::optional<Tensor> absmax_q,
                std::optional<Tensor> code2, std::optional<Tensor> absmax2, double offset, int64_t blocksize,
                int64_t out, int64_t in, const Tensor& A, const Tensor& B, std::optional<Tensor> bias, double scale) {
  auto w = std::make_shared<Nf4>();
  auto set = [](std::optional<Tensor>& t) { return t ? *t : Tensor(); };
  TORCH_CHECK_VALUE(blocksize >= 32, "the quantisation block size must be at least 32, got ", blocksize);
  need(packed, "packed", at::kByte, {out * in / 2});
  const int64_t blocks = out * in / blocksize;
  if (absmax) {
    need(*absmax, "absmax", at::kFloat, {blocks});
  } else {
    TORCH_CHECK_VALUE(absmax_q && code2 && absmax2, "block maxima or their quantised form are needed");
    need(*absmax_q, "absmax_q", at::kByte, {blocks});
    need(*code2, "code2", at::kFloat, {256});
    need(*absmax2, "absmax2", at::kFloat, absmax2->sizes());
  }
  *w = Nf4{packed, set(absmax), set(absmax_q), set(code2), set(absmax2), offset, blocksize, out, in};
  LoraArgs a;
  a.nf4 = std::move(w);
  a.bias = {std::move(bias)};
  a.scale = scale;
  const Tensor As[1] = {A}, Bs[1] = {B};
  return LoraFunction::apply(x, at::TensorList(As), at::TensorList(Bs), a)[0];
}

// ---- attention over packed rows -------------------------------------------------------------------------------
void need_heads(const Tensor& t, const char* name) {
  TORCH_CHECK_VALUE(t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == 4, name,
                    ": expected a bf16 device tensor [B, S, H, D]");
}

// (batch, position, head) strides of a [B, S, H, D] view whose last dimension is contiguous.
void strides_of(const Tensor& t, const char* name, int64_t* out) {
  TORCH_CHECK_VALUE(t.stride(3) == 1, name, ": expected a bf16 device tensor [B, S, H, D] with contiguous D");
  out[0] = t.size(0) > 1 ? t.stride(0) : 0;
  out[1] = t.stride(1);
  out[2] = t.stride(2);
}

// `t` [B, S, H, D], or a copy of it where its layout is none that the kernels address.
Tensor addressable(const Tensor& t) {
  const int64_t rows = (t.size(1) + 255) / 256 * 256;  // a row's tiles cover this many positions
  bool ok = t.stride(3) == 1 && ((uintptr_t)t.data_ptr() & 15) == 0 && rows * t.stride(1) * 2 < (1ll << 31);
  for (int i = t.size(0) > 1 ? 0 : 1; i < 3; ++i) ok = ok && t.stride(i) > 0 && t.stride(i) % 8 == 0;
  // (not contiguous(): it returns t itself where only a pointer or the stride of a dimension of size 1 is odd)
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

struct AttentionFunction : torch::autograd::Function<AttentionFunction> {
  static Tensor forward(AutogradContext* ctx, Tensor q, Tensor k, Tensor v, const Tensor& plan, double scale) {
    need_heads(q, "q");
    need_heads(k, "k");
    need_heads(v, "v");
    const int64_t B = q.size(0), S = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
    TORCH_CHECK_VALUE(k.sizes() == at::IntArrayRef({B, S, Hkv, D}) && v.sizes() == k.sizes(),
                      "attention: inconsistent shapes");
    TORCH_CHECK_VALUE((size_t)plan.numel() >= (size_t)B * artk_attn_plan_row_stride(S), "the plan is for other rows");
    c10::OptionalDeviceGuard guard(q.device());
    if (S % 256 != 0) {  // rows that end inside a block may have any layout; whole blocks are taken as they are
      q = addressable(q);
      k = addressable(k);
      v = addressable(v);
    }
    int64_t st[12];
    strides_of(q, "q", st);
    strides_of(k, "k", st + 3);
    strides_of(v, "v", st + 6);
    const Tensor out = make(q, {B, S, Hq, D}, at::kBFloat16), lse = make(q, {B, Hq, S}, at::kFloat);
    strides_of(out, "out", st + 9);
    check(artk_attn_fwd_rows(q.data_ptr(), k.data_ptr(), v.data_ptr(), plan.data_ptr(), B, S, (int32_t)Hq, (int32_t)Hkv,
                             (int32_t)D, st, (float)scale, out.data_ptr(), lse.data_ptr<float>(), stream_of(q)));
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["plan"] = plan;  // shared by all layers: hooks on saved tensors need not see it
    ctx->saved_data["scale"] = scale;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &out = saved[3], &lse = saved[4];
    const Tensor plan = ctx->saved_data["plan"].toTensor();
    c10::OptionalDeviceGuard guard(q.device());
    const int64_t B = q.size(0), S = q.size(1), Hq = q.size(2), D = q.size(3), Hkv = k.size(2);
    const Tensor g = addressable(grads[0].to(at::kBFloat16));
    const Tensor dq = make(q, {B, S, Hq, D}, at::kBFloat16), dk = make(q, {B, S, Hkv, D}, at::kBFloat16),
                 dv = make(q, {B, S, Hkv, D}, at::kBFloat16);
    int64_t st[24];
    int i = 0;
    for (const Tensor* t : {&q, &k, &v, &out, &g, &dq, &dk, &dv}) strides_of(*t, "attention", st + 3 * i++);
    const Tensor ws = workspace(q, artk_attn_bwd_rows_workspace_bytes(B, S, (int32_t)Hq, (int32_t)Hkv, (int32_t)D));
    check(artk_attn_bwd_rows(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                             g.data_ptr(), plan.data_ptr(), B, S, (int32_t)Hq, (int32_t)Hkv, (int32_t)D, st,
                             (float)ctx->saved_data["scale"].toDouble(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                             ws.data_ptr(), ws.numel(), stream_of(q)));
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};

Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& plan, std::optional<double> scale) {
  need_heads(q, "q");
  return AttentionFunction::apply(q, k, v, plan, scale ? *scale : 1.0 / std::sqrt((double)q.size(3)));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  // (the wrapper hands Python exceptions on as they are and releases the interpreter lock)
  m.def("lora_multi", torch::wrap_pybind_function_no_gil(&lora_multi), py::arg("x"), py::arg("W"), py::arg("W_t"),
        py::arg("A"), py::arg("B"), py::arg("bias"), py::arg("scale"));
  m.def("lora_nf4", torch::wrap_pybind_function_no_gil(&lora_nf4), py::arg("x"), py::arg("packed"), py::arg("absmax"),
        py::arg("absmax_q"), py::arg("code2"), py::arg("absmax2"), py::arg("offset"), py::arg("blocksize"),
        py::arg("out"), py::arg("in_"), py::arg("A"), py::arg("B"), py::arg("bias"), py::arg("scale"));
  m.def("attention", torch::wrap_pybind_function_no_gil(&attention), py::arg("q"), py::arg("k"), py::arg("v"),
        py::arg("plan"), py::arg("scale"));
  m.def("_check", torch::wrap_pybind_function_no_gil(&check), py::arg("rc"));
}
