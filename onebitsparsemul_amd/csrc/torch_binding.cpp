// pybind11 / ATen binding `onebit_sparse_cuda.onebit_mul(A, B, meta, C)`.
// Same module name, function name, positional order and docstring as the reference binding
// (onebit_sparse_mul/torch_kernel_cuda.cpp:10-38; module name from setup.py:14). The reference derives
// m and k from A's shape, which matches none of the layouts its own Python side produces, and raises when
// the shapes agree (:13-18); here the problem size comes from the operands' defined shapes and every
// mismatch raises a Python exception:
//   A    uint8  (k/2, m/8)   one-bit values as written by BinaryLinear_2_4.pack()
//   B    fp16   (k, n)       contiguous
//   meta int16  (m, k/16)    reordered metadata
//   C    fp32 or fp16 (m, n) destination (the reference passes it as both source and destination, :23-24)
// The work is enqueued on PyTorch's current HIP stream of C's device.
//
// The package's own calls (layer forward, grouped forward, prepared product, one-call product, packing) have their host
// side here too: a decode-sized product takes 4 to 7 us on the GPU, and checking the operands, allocating the result and
// making the library call from Python took 9 to 27 us.
#include <torch/extension.h>
// PyTorch on ROCm presents its devices as type "cuda"; these are the guard and stream accessors for that.
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include "onebit_sparse_tensor.h"

namespace {

void check_operand(const torch::Tensor& t, const char* name, c10::ScalarType dtype, const c10::Device& device) {
  TORCH_CHECK(t.device() == device, name, " must be on ", device, ", got ", t.device());
  TORCH_CHECK(t.scalar_type() == dtype, name, " must have dtype ", dtype, ", got ", t.scalar_type());
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

void onebit_mul(const torch::Tensor& A, const torch::Tensor& B, const torch::Tensor& meta, torch::Tensor& C) {
  TORCH_CHECK(C.is_cuda(), "C must be a GPU tensor");
  TORCH_CHECK(meta.dim() == 2 && B.dim() == 2 && C.dim() == 2, "meta, B and C must be 2-dimensional");
  const c10::Device device = C.device();
  check_operand(A, "A", torch::kUInt8, device);
  check_operand(B, "B", torch::kFloat16, device);
  check_operand(meta, "meta", torch::kInt16, device);
  TORCH_CHECK(C.scalar_type() == torch::kFloat32 || C.scalar_type() == torch::kFloat16,
              "C must be float32 or float16, got ", C.scalar_type());
  TORCH_CHECK(C.is_contiguous(), "C must be contiguous");

  const int64_t prob_m = meta.size(0);
  const int64_t prob_k = meta.size(1) * 16;
  const int64_t prob_n = B.size(1);
  TORCH_CHECK(A.numel() == prob_m * prob_k / 16, "A holds ", A.numel(), " bytes, expected m*k/16 = ",
              prob_m * prob_k / 16, " for meta of shape (", prob_m, ", ", meta.size(1), ")");
  TORCH_CHECK(B.size(0) == prob_k, "B.size(0) = ", B.size(0), " != k = ", prob_k);
  TORCH_CHECK(C.size(0) == prob_m && C.size(1) == prob_n, "C must have shape (", prob_m, ", ", prob_n, ")");
  TORCH_CHECK(prob_m < (1ll << 31) && prob_n < (1ll << 31) && prob_k < (1ll << 31), "problem size exceeds int range");

  const c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
  void* stream = static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream());
  const int d_dtype = C.scalar_type() == torch::kFloat16 ? ONEBIT_DTYPE_F16 : ONEBIT_DTYPE_F32;
  const int rc = onebit_sparse_matmul_ex(A.data_ptr(), B.data_ptr(), C.data_ptr(), C.data_ptr(), meta.data_ptr(),
                                         (int)prob_m, (int)prob_n, (int)prob_k, 1.0f, 0.0f, d_dtype, d_dtype,
                                         ONEBIT_META_REFERENCE, stream);
  TORCH_CHECK(rc == ONEBIT_OK, "onebit_sparse_matmul_ex failed: ", onebit_sparse_last_error());
}

using OptionalTensor = std::optional<torch::Tensor>;

int dtype_code(c10::ScalarType type) {
  switch (type) {
    case torch::kFloat32: return ONEBIT_DTYPE_F32;
    case torch::kFloat16: return ONEBIT_DTYPE_F16;
    case torch::kBFloat16: return ONEBIT_DTYPE_BF16;
    default: return -1;
  }
}

void* current_stream(const c10::Device& device) {
  return static_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream());
}

void check_status(int rc) {
  TORCH_CHECK(rc == ONEBIT_OK, "libonebitmul: ", onebit_sparse_last_error(), " (status ", rc, ")");
}

// every operand on one GPU, contiguous
void check_placement(const torch::Tensor& t, const c10::Device& device) {
  TORCH_CHECK_VALUE(t.is_cuda(), "all operands must live on the GPU");
  TORCH_CHECK_VALUE(t.is_contiguous(), "all operands must be contiguous");
  TORCH_CHECK_VALUE(t.device() == device, "all operands must be on the same device");
}

torch::Tensor empty_result(at::IntArrayRef sizes, c10::ScalarType type, const c10::Device& device) {
  return at::empty(sizes, at::TensorOptions().dtype(type).device(device));
}

size_t prepared_bytes(int64_t m, int64_t k) { return ((size_t)m + 31) / 32 * (((size_t)k + 255) / 256) * 1536; }

// Type the kernels read and type they write for activations of type `x`; `out`: the layer's out_dtype, if it has one. bf16
// activations are multiplied as they are, all others as fp16 with an fp32 result unless they are fp16 themselves.
struct LayerTypes {
  c10::ScalarType in, out;
};
LayerTypes layer_types(c10::ScalarType x, std::optional<c10::ScalarType> out) {
  if (x == torch::kBFloat16 && out != torch::kFloat16) return {torch::kBFloat16, out.value_or(torch::kBFloat16)};
  return {torch::kFloat16, out.value_or(x == torch::kFloat16 ? torch::kFloat16 : torch::kFloat32)};
}

// The activations as the kernels read them: (tokens, k), contiguous, 16-byte aligned, of type `type`.
torch::Tensor kernel_input(const torch::Tensor& x, c10::ScalarType type) {
  torch::Tensor t = x.scalar_type() == type ? x : x.to(type);
  if (!t.is_contiguous()) t = t.contiguous();
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t;  // a view may start inside a 16-byte unit
}

torch::Tensor kernel_bias(const torch::Tensor& bias, const c10::Device& device, int64_t m) {
  torch::Tensor t = dtype_code(bias.scalar_type()) < 0 || bias.device() != device ? bias.to(device, torch::kFloat32) : bias;
  if (!t.is_contiguous()) t = t.contiguous();
  TORCH_CHECK_VALUE(t.dim() == 1 && t.size(0) == m, "bias must have shape (", m, ",)");
  return t;
}

std::vector<int64_t> result_sizes(const torch::Tensor& x, int64_t m) {
  std::vector<int64_t> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = m;
  return sizes;
}

int64_t token_count(const torch::Tensor& x, int64_t k) {
  TORCH_CHECK(x.dim() >= 1 && x.size(-1) == k, "the last dimension of x must be ", k, " (got shape ", x.sizes(), ")");
  const int64_t tokens = x.numel() / k;
  TORCH_CHECK_VALUE(tokens < (1ll << 31), "too many tokens");
  return tokens;
}

// Whether the values of a contiguous tensor are what lies in its memory: a negated view's sign is applied by the next operation on it
// (here a conversion), and a subclass that handles operations itself may keep its values elsewhere.
bool values_in_memory(const torch::Tensor& x) {
  return !x.is_neg() && !x._is_zerotensor() && !x.unsafeGetTensorImpl()->is_python_dispatch();
}

// BinaryLinear_2_4.forward behind its bookkeeping: y = x W^T (+ bias), shape and type of the layer's result. Nothing where x is on
// another device than the prepared weight: the layer then prepares its weight there.
OptionalTensor layer_forward(const torch::Tensor& prepared, const torch::Tensor& x, const OptionalTensor& bias, int64_t m,
                            int64_t k, std::optional<c10::ScalarType> out_dtype) {
  if (prepared.device() != x.device()) return std::nullopt;
  at::AutoDispatchBelowADInplaceOrView guard_dispatch;
  if (x.numel() == 0) return at::zeros(result_sizes(x, m), x.options());  // an empty batch: nothing to launch
  const int64_t tokens = token_count(x, k);
  const c10::Device device = x.device();
  check_placement(prepared, device);
  TORCH_CHECK_VALUE(prepared.nbytes() == prepared_bytes(m, k), "prepared operand does not match m, k");
  const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(device);
  const LayerTypes types = layer_types(x.scalar_type(), out_dtype);
  // fp32 activations of a few tokens are rounded by the kernel that reads them, all others by a conversion in front of it
  const bool read_f32 = x.scalar_type() == torch::kFloat32 && x.is_contiguous() && values_in_memory(x) &&
                        reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                        onebit_sparse_linear_reads_f32((int)tokens, (int)m, (int)k, current_stream(device));
  const torch::Tensor in = read_f32 ? x : kernel_input(x, types.in);
  OptionalTensor b;
  if (bias.has_value()) b = kernel_bias(*bias, device, m);
  torch::Tensor y = empty_result(result_sizes(x, m), types.out, device);
  const void* const bias_data = b.has_value() ? b->data_ptr() : nullptr;
  const int bias_code = b.has_value() ? dtype_code(b->scalar_type()) : ONEBIT_DTYPE_F16;
  check_status(read_f32
                   ? onebit_sparse_linear_prepared_f32(prepared.data_ptr(), in.data_ptr(), bias_data, y.data_ptr(), (int)tokens,
                                                       (int)m, (int)k, bias_code, dtype_code(types.out), current_stream(device))
                   : onebit_sparse_linear_prepared_typed(prepared.data_ptr(), in.data_ptr(), bias_data, y.data_ptr(), (int)tokens,
                                                         (int)m, (int)k, dtype_code(types.in), bias_code, dtype_code(types.out),
                                                         current_stream(device)));
  return out_dtype.has_value() || types.out == x.scalar_type() ? y : y.to(x.scalar_type());
}

// Several layers on activations with the same number of tokens in one library call. Returns an empty vector when the layers
// do not share a token count, a type or a bias type: the caller then runs them one by one. xs: one tensor for all layers,
// or one per layer.
std::vector<torch::Tensor> grouped_forward(const std::vector<torch::Tensor>& prepared, const std::vector<torch::Tensor>& xs,
                                           const std::vector<OptionalTensor>& biases, const std::vector<int64_t>& ms,
                                           const std::vector<int64_t>& ks,
                                           const std::vector<std::optional<c10::ScalarType>>& out_dtypes) {
  at::AutoDispatchBelowADInplaceOrView guard_dispatch;
  const size_t count = prepared.size();
  auto x_of = [&](size_t i) -> const torch::Tensor& { return xs[xs.size() == 1 ? 0 : i]; };
  const c10::Device device = xs[0].device();
  const int64_t tokens = xs[0].numel() == 0 ? 0 : token_count(xs[0], ks[0]);
  if (tokens == 0) return {};
  const LayerTypes types = layer_types(xs[0].scalar_type(), out_dtypes[0]);
  std::optional<c10::ScalarType> bias_type;
  for (size_t i = 0; i < count; ++i) {
    const torch::Tensor& x = x_of(i);
    if (x.numel() == 0 || x.device() != device || token_count(x, ks[i]) != tokens) return {};
    const LayerTypes own = layer_types(x.scalar_type(), out_dtypes[i]);
    if (own.in != types.in || own.out != types.out) return {};
    if (biases[i].has_value()) {
      const c10::ScalarType type = dtype_code(biases[i]->scalar_type()) < 0 || biases[i]->device() != device
                                       ? torch::kFloat32 : biases[i]->scalar_type();
      if (bias_type.has_value() && *bias_type != type) return {};
      bias_type = type;
    }
  }
  const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(device);
  std::vector<torch::Tensor> ys(count), inputs(xs.size()), kept(count);
  for (size_t i = 0; i < xs.size(); ++i) {
    inputs[i] = torch::Tensor();
    for (size_t j = 0; j < i && !inputs[i].defined(); ++j)  // one tensor handed in several times is brought in once
      if (xs[j].is_same(xs[i])) inputs[i] = inputs[j];
    if (!inputs[i].defined()) inputs[i] = kernel_input(xs[i], types.in);
  }
  std::vector<onebit_linear_problem> problems(count);
  for (size_t i = 0; i < count; ++i) {
    check_placement(prepared[i], device);
    TORCH_CHECK_VALUE(prepared[i].nbytes() == prepared_bytes(ms[i], ks[i]), "prepared operand does not match m, k");
    if (biases[i].has_value()) kept[i] = kernel_bias(*biases[i], device, ms[i]);
    ys[i] = empty_result(result_sizes(x_of(i), ms[i]), types.out, device);
    problems[i] = onebit_linear_problem{prepared[i].data_ptr(), inputs[xs.size() == 1 ? 0 : i].data_ptr(),
                                        kept[i].defined() ? kept[i].data_ptr() : nullptr, ys[i].data_ptr(), (int)ms[i],
                                        (int)ks[i]};
  }
  check_status(onebit_sparse_linear_prepared_grouped_typed(
      problems.data(), (int)count, (int)tokens, dtype_code(types.in),
      bias_type.has_value() ? dtype_code(*bias_type) : ONEBIT_DTYPE_F16, dtype_code(types.out), current_stream(device)));
  for (size_t i = 0; i < count; ++i)
    if (!out_dtypes[i].has_value() && types.out != x_of(i).scalar_type()) ys[i] = ys[i].to(x_of(i).scalar_type());
  return ys;
}

// forward_grouped: the layers' attributes are read here (in Python their lists took as long as the launch). None where a layer has
// no weight prepared on its input's device.
py::object grouped_forward_layers(const py::list& layers, const std::vector<torch::Tensor>& xs) {
  static PyObject* const names[] = {PyUnicode_InternFromString("_prepared"), PyUnicode_InternFromString("vaild"),
                                    PyUnicode_InternFromString("buffer"), PyUnicode_InternFromString("bias"),
                                    PyUnicode_InternFromString("outfeatures"), PyUnicode_InternFromString("infeatures"),
                                    PyUnicode_InternFromString("out_dtype")};
  auto get = [](const py::handle& object, int name) {
    PyObject* value = PyObject_GetAttr(object.ptr(), names[name]);
    if (!value) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(value);
  };
  const size_t count = layers.size();
  std::vector<torch::Tensor> prepared(count);
  std::vector<OptionalTensor> biases(count);
  std::vector<int64_t> ms(count), ks(count);
  std::vector<std::optional<c10::ScalarType>> out_dtypes(count);
  for (size_t i = 0; i < count; ++i) {
    const py::handle layer = layers[i];
    const py::object own = get(layer, 0);
    if (own.is_none() || !py::cast<bool>(get(layer, 1))) return py::none();
    prepared[i] = py::cast<torch::Tensor>(get(own, 2));
    if (prepared[i].device() != xs[xs.size() == 1 ? 0 : i].device()) return py::none();
    biases[i] = py::cast<OptionalTensor>(get(layer, 3));
    ms[i] = py::cast<int64_t>(get(layer, 4));
    ks[i] = py::cast<int64_t>(get(layer, 5));
    out_dtypes[i] = py::cast<std::optional<c10::ScalarType>>(get(layer, 6));
  }
  std::vector<torch::Tensor> ys;
  {
    const py::gil_scoped_release release;
    ys = grouped_forward(prepared, xs, biases, ms, ks, out_dtypes);
  }
  return py::cast(std::move(ys));
}

// PreparedWeight.matmul: D = alpha A B + beta C into `out`, or into a new tensor of type out_dtype (None: torch's default).
torch::Tensor matmul_prepared(const torch::Tensor& prepared, const torch::Tensor& b, const OptionalTensor& c,
                              const OptionalTensor& out, int64_t m, int64_t k, double alpha, double beta,
                              std::optional<c10::ScalarType> out_dtype) {
  at::AutoDispatchBelowADInplaceOrView guard_dispatch;
  const c10::Device device = b.device();
  check_placement(b, device);
  check_placement(prepared, device);
  TORCH_CHECK_VALUE(b.scalar_type() == torch::kFloat16 && b.dim() == 2 && b.size(0) == k, "B must be float16 of shape (k, n)");
  const int64_t n = b.size(1);
  TORCH_CHECK_VALUE(n < (1ll << 31), "too many columns");
  TORCH_CHECK_VALUE(prepared.nbytes() == prepared_bytes(m, k), "prepared operand does not match m, k");
  auto check_result = [&](const torch::Tensor& t) {
    check_placement(t, device);
    TORCH_CHECK_VALUE(t.dim() == 2 && t.size(0) == m && t.size(1) == n, "C / D must have shape (m, n)");
    TORCH_CHECK_TYPE(t.scalar_type() == torch::kFloat32 || t.scalar_type() == torch::kFloat16,
                     "C / D must be float32 or float16, got ", t.scalar_type());
  };
  if (c.has_value()) check_result(*c);
  const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(device);
  torch::Tensor d = out.has_value() ? *out : empty_result({m, n}, out_dtype.value_or(c10::get_default_dtype_as_scalartype()), device);
  check_result(d);
  check_status(onebit_sparse_matmul_prepared(prepared.data_ptr(), b.data_ptr(), c.has_value() ? c->data_ptr() : nullptr,
                                             d.data_ptr(), (int)m, (int)n, (int)k, (float)alpha, (float)beta,
                                             c.has_value() ? dtype_code(c->scalar_type()) : ONEBIT_DTYPE_F32,
                                             dtype_code(d.scalar_type()), current_stream(device)));
  return d;
}

// cuda_binary_mul: the product into a new fp32 tensor.
torch::Tensor binary_mul(const torch::Tensor& A, const torch::Tensor& B, const torch::Tensor& meta) {
  at::AutoDispatchBelowADInplaceOrView guard_dispatch;
  TORCH_CHECK_VALUE(meta.dim() == 2, "meta must be 2-dimensional");
  const int64_t m = meta.size(0), k = meta.size(1) * 16;
  TORCH_CHECK_VALUE(A.scalar_type() == torch::kUInt8 && A.numel() == m * k / 16, "A must be uint8 with m*k/16 = ", m * k / 16,
                    " bytes (shape (k/2, m/8)), got ", A.sizes());
  TORCH_CHECK_VALUE(B.dim() == 2 && B.size(0) == k, "B must have shape (k=", k, ", n), got ", B.sizes());
  torch::Tensor C = empty_result({m, B.size(1)}, torch::kFloat32, B.device());
  onebit_mul(A, B, meta, C);
  return C;
}

// The kernels' operand from the stored ones (PreparedWeight).
torch::Tensor prepare(const torch::Tensor& a, const torch::Tensor& meta, int64_t m, int64_t k, int64_t layout) {
  at::AutoDispatchBelowADInplaceOrView guard_dispatch;
  const c10::Device device = a.device();
  check_placement(a, device);
  check_placement(meta, device);
  TORCH_CHECK_VALUE((int64_t)a.nbytes() == m * k / 16 && (int64_t)meta.nbytes() == m * k / 8, "operand sizes do not match m, k");
  const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(device);
  torch::Tensor out = empty_result({(int64_t)prepared_bytes(m, k)}, torch::kUInt8, device);
  check_status(onebit_sparse_prepare(a.data_ptr(), meta.data_ptr(), (int)m, (int)k, (int)layout, out.data_ptr(),
                                     current_stream(device)));
  return out;
}

// The stored operands of a dense weight (BinaryLinear_2_4.pack).
std::tuple<torch::Tensor, torch::Tensor> pack_weight(const torch::Tensor& weight, bool prune, int64_t layout) {
  at::AutoDispatchBelowADInplaceOrView guard_dispatch;
  const c10::Device device = weight.device();
  check_placement(weight, device);
  TORCH_CHECK_TYPE(weight.dim() == 2 && dtype_code(weight.scalar_type()) >= 0,
                   "weight must be a 2-dimensional float16, bfloat16 or float32 tensor");
  const int64_t m = weight.size(0), k = weight.size(1);
  TORCH_CHECK_VALUE(m < (1ll << 31) && k < (1ll << 31), "weight too large");
  const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(device);
  torch::Tensor a = empty_result({k / 2, m / 8}, torch::kUInt8, device);
  torch::Tensor meta = empty_result({m, k / 16}, torch::kInt16, device);
  check_status(onebit_sparse_pack_typed(weight.data_ptr(), dtype_code(weight.scalar_type()), (int)m, (int)k, prune ? 1 : 0,
                                        a.data_ptr(), meta.data_ptr(), (int)layout, current_stream(device)));
  return {a, meta};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  // Without the interpreter lock: a call may wait for another thread's, or for the device when a buffer has to grow.
  using NoGil = pybind11::call_guard<pybind11::gil_scoped_release>;
  m.def("onebit_mul", &onebit_mul, "A32 = Sparse W1 * A16 matmul.", NoGil());
  m.def("layer_forward", &layer_forward, NoGil());
  m.def("grouped_forward", &grouped_forward_layers);
  m.def("matmul_prepared", &matmul_prepared, NoGil());
  m.def("binary_mul", &binary_mul, NoGil());
  m.def("prepare", &prepare, NoGil());
  m.def("pack_weight", &pack_weight, NoGil());
}
