// Native call path of the Python modules: operand checks, output and scratch
// tensors and the C ABI call in one step.
//
// The ctypes binding (actune_amd/_native.py) spends about 15 us of host time
// on a call whose kernel takes 4 us: attribute checks on seven tensors, three
// allocations, the current stream and seventeen converted arguments. Each
// function here takes the plain case of one of its calls: every operand on
// one GPU, contiguous, of the expected type and shape, 16-byte aligned, no
// caller-owned buffers. Anything else, an argument of another type included,
// returns None, and the ctypes path, which names what is wrong or makes an
// aligned copy, takes the call. Output and scratch come from torch's caching
// allocator on the current stream, as there; nothing is kept between calls.
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <torch/version.h>

#include <cstring>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/actune_hip.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

struct Api {
  decltype(&actune_quantize_groups) quantize_groups;
  decltype(&actune_quantize_gated) quantize_gated;
  decltype(&actune_grouped_linear) grouped_linear;
  decltype(&actune_grouped_forward_multi) grouped_forward_multi;
  decltype(&actune_tokenwise_quantize) tokenwise_quantize;
  decltype(&actune_tokenwise_workspace_bytes) tokenwise_workspace_bytes;
  decltype(&actune_tokenwise_linear) tokenwise_linear;
  decltype(&actune_tokenwise_linear_x) tokenwise_linear_x;
  decltype(&actune_tokenwise_linear_multi) tokenwise_linear_multi;
  decltype(&actune_last_error) last_error;
};
Api api{};

// The library's functions by address: this module runs the copy that the
// ctypes binding loaded.
void init(const std::vector<uintptr_t>& f) {
  TORCH_CHECK(f.size() == sizeof(Api) / sizeof(void*), "one address per function");
  std::memcpy(&api, f.data(), sizeof(Api));
}

void check(int rc) {
  if (rc == ACTUNE_OK) return;
  const std::string msg = api.last_error();
  if (rc == ACTUNE_ERR_DEVICE) throw std::runtime_error(msg);
  throw py::value_error(msg);
}

int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? 0 : t == at::kHalf ? 1 : t == at::kFloat ? 2 : -1; }
at::ScalarType dtype_of(int code) { return code == 0 ? at::kBFloat16 : code == 1 ? at::kHalf : at::kFloat; }
bool width_ok(int64_t b) { return b == 2 || b == 4 || b == 8; }

bool plain(const Tensor& t, const at::Device& dev) { return t.defined() && t.device() == dev && t.is_contiguous(); }
bool plain(const Tensor& t, const at::Device& dev, at::ScalarType type) {
  return plain(t, dev) && t.scalar_type() == type;
}
bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }

// A [M, K] GPU tensor of a float type, 16-byte aligned
bool rows_ok(const Tensor& x) {
  return x.defined() && x.is_cuda() && x.dim() == 2 && x.is_contiguous() && dtype_code(x.scalar_type()) >= 0 && aligned(x);
}
bool scale_ok(const OptTensor& s, const Tensor& x) {
  return !s || (plain(*s, x.device(), x.scalar_type()) && s->numel() == x.size(1) && aligned(*s));
}
bool bias_ok(const OptTensor& b, const at::Device& dev, int64_t n) {
  return !b || (plain(*b, dev) && dtype_code(b->scalar_type()) >= 0 && b->numel() == n);
}
bool weights_ok(const Tensor& w, const Tensor& ws, const OptTensor& b, const at::Device& dev, int64_t k, int64_t W) {
  return plain(w, dev, at::kByte) && w.dim() == 2 && w.size(1) == k * W / 8 && plain(ws, dev, at::kFloat) &&
         ws.numel() == w.size(0) && bias_ok(b, dev, w.size(0));
}
const void* ptr(const OptTensor& t) { return t ? t->const_data_ptr() : nullptr; }
int bias_code(const OptTensor& b) { return b ? dtype_code(b->scalar_type()) : 2; }
void* stream(const at::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }
Tensor empty(at::IntArrayRef size, const at::Device& dev, at::ScalarType type) {
  return at::empty(size, at::TensorOptions().device(dev).dtype(type));
}

// Codes and group scales of [m, k] rows in one allocation.
struct CodeBuffer {
  Tensor raw;
  uint8_t* codes;
  float* scales;
  CodeBuffer(int64_t m, int64_t k, int64_t A, const at::Device& dev) {
    const int64_t bytes = (m * k * A / 8 + 255) / 256 * 256;
    raw = empty({bytes + m * (k / 64) * 4}, dev, at::kByte);
    codes = static_cast<uint8_t*>(raw.mutable_data_ptr());
    scales = reinterpret_cast<float*>(codes + bytes);
  }
};

py::object quantize_groups(const Tensor& x, int64_t A, const OptTensor& scale) {
  if (!rows_ok(x) || !width_ok(A) || x.size(1) % 64 || !scale_ok(scale, x)) return py::none();
  const int64_t m = x.size(0), k = x.size(1);
  Tensor packed = empty({m, k * A / 8}, x.device(), at::kByte), scales = empty({m, k / 64}, x.device(), at::kFloat);
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.quantize_groups(x.const_data_ptr(), dtype_code(x.scalar_type()), ptr(scale), m, k, (int)A,
                             packed.mutable_data_ptr<uint8_t>(), scales.mutable_data_ptr<float>(), stream(x.device()));
  }
  check(rc);
  return py::make_tuple(packed, scales);
}

py::object quantize_gated(const Tensor& gate, const Tensor& up, int64_t act, int64_t A, const OptTensor& scale) {
  if (!rows_ok(gate) || !rows_ok(up) || up.sizes() != gate.sizes() || up.scalar_type() != gate.scalar_type() ||
      up.device() != gate.device() || !width_ok(A) || gate.size(1) % 64 || !scale_ok(scale, gate))
    return py::none();
  const int64_t m = gate.size(0), k = gate.size(1);
  Tensor packed = empty({m, k * A / 8}, gate.device(), at::kByte), scales = empty({m, k / 64}, gate.device(), at::kFloat);
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.quantize_gated(gate.const_data_ptr(), up.const_data_ptr(), dtype_code(gate.scalar_type()), (int)act,
                            ptr(scale), m, k, (int)A, packed.mutable_data_ptr<uint8_t>(),
                            scales.mutable_data_ptr<float>(), stream(gate.device()));
  }
  check(rc);
  return py::make_tuple(packed, scales);
}

py::object grouped_linear(const Tensor& a, const Tensor& as, const Tensor& w, const Tensor& ws, const OptTensor& bias,
                          int64_t m, int64_t k, int out_code, int64_t W, int64_t A, int config) {
  if (!a.is_cuda() || !width_ok(W) || !width_ok(A) || k <= 0 || k % 64 || out_code < 0) return py::none();
  const at::Device dev = a.device();
  if (!plain(a, dev, at::kByte) || a.dim() != 2 || a.size(0) != m || a.size(1) != k * A / 8 || !plain(as, dev, at::kFloat) ||
      as.dim() != 2 || as.size(0) != m || as.size(1) != k / 64 || !weights_ok(w, ws, bias, dev, k, W) ||
      w.size(0) == 0)
    return py::none();
  const int64_t n = w.size(0);
  Tensor out = empty({m, n}, dev, dtype_of(out_code));
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.grouped_linear(a.const_data_ptr<uint8_t>(), as.const_data_ptr<float>(), w.const_data_ptr<uint8_t>(),
                            ws.const_data_ptr<float>(), ptr(bias), bias_code(bias), out.mutable_data_ptr(), out_code, m, n,
                            k, (int)W, (int)A, config, stream(dev));
  }
  check(rc);
  return py::cast(out);
}

bool is_tensor(const py::object& o) { return THPVariable_Check(o.ptr()); }

// targets: sequences (w, w_scale, bias or None, None[, W])
py::object grouped_forward_multi(const Tensor& x, const py::sequence& targets, int64_t W, int64_t A,
                                 const OptTensor& scale, int config) {
  const size_t count = targets.size();
  if (count < 1 || count > ACTUNE_MAX_TARGETS || !rows_ok(x) || !width_ok(W) || !width_ok(A) || x.size(1) <= 0 ||
      x.size(1) % 64 || !scale_ok(scale, x))
    return py::none();
  const at::Device dev = x.device();
  const int64_t m = x.size(0), k = x.size(1);
  actune_linear_target t[ACTUNE_MAX_TARGETS];
  std::vector<Tensor> outs;
  Tensor weights[ACTUNE_MAX_TARGETS], scales[ACTUNE_MAX_TARGETS];  // held over the call (lists can change under it)
  OptTensor biases[ACTUNE_MAX_TARGETS];
  int bias_type = 2;
  for (size_t i = 0; i < count; ++i) {
    const py::object target = targets[i];
    if (!PyTuple_Check(target.ptr()) && !PyList_Check(target.ptr())) return py::none();
    const auto g = py::reinterpret_borrow<py::sequence>(target);
    const size_t fields = g.size();
    if (fields < 4) return py::none();
    const py::object gw = g[0], gs = g[1], gb = g[2], go = g[3], gn = fields > 4 ? py::object(g[4]) : py::none();
    if (!is_tensor(gw) || !is_tensor(gs) || !(gb.is_none() || is_tensor(gb)) || !go.is_none() ||
        !(fields < 5 || PyLong_Check(gn.ptr())))
      return py::none();
    const Tensor &w = weights[i] = gw.cast<Tensor>(), &scale_w = scales[i] = gs.cast<Tensor>();
    const OptTensor& bias = biases[i] = gb.cast<OptTensor>();
    int overflow = 0;
    const int64_t width = fields > 4 ? PyLong_AsLongLongAndOverflow(gn.ptr(), &overflow) : W;
    if (overflow || !width_ok(width) || !weights_ok(w, scale_w, bias, dev, k, width)) return py::none();
    const bool same = i == 0 || ((t[0].bias != nullptr) == bias.has_value() && bias_type == bias_code(bias));
    if (!same) return py::none();
    bias_type = bias_code(bias);
    outs.push_back(empty({m, w.size(0)}, dev, x.scalar_type()));
    t[i] = actune_linear_target{w.const_data_ptr<uint8_t>(), scale_w.const_data_ptr<float>(), ptr(bias),
                                outs[i].mutable_data_ptr(), w.size(0), (int32_t)width};
  }
  const CodeBuffer codes(m, k, A, dev);
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.grouped_forward_multi(x.const_data_ptr(), dtype_code(x.scalar_type()), ptr(scale), codes.codes, codes.scales,
                                   t, (int)count, bias_type, m, k, (int)W, (int)A, config, stream(dev));
  }
  check(rc);
  return py::cast(outs);
}

py::object grouped_forward(const Tensor& x, const Tensor& w, const Tensor& ws, const OptTensor& bias, int64_t W, int64_t A,
                           const OptTensor& scale, int config) {
  if (!rows_ok(x) || !width_ok(W) || !width_ok(A) || x.size(1) <= 0 || x.size(1) % 64 || !scale_ok(scale, x) ||
      !weights_ok(w, ws, bias, x.device(), x.size(1), W))
    return py::none();
  const at::Device dev = x.device();
  const int64_t m = x.size(0), k = x.size(1), n = w.size(0);
  Tensor out = empty({m, n}, dev, x.scalar_type());
  const actune_linear_target t{w.const_data_ptr<uint8_t>(), ws.const_data_ptr<float>(), ptr(bias), out.mutable_data_ptr(),
                               n, (int32_t)W};
  const CodeBuffer codes(m, k, A, dev);
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.grouped_forward_multi(x.const_data_ptr(), dtype_code(x.scalar_type()), ptr(scale), codes.codes, codes.scales,
                                   &t, 1, bias_code(bias), m, k, (int)W, (int)A, config, stream(dev));
  }
  check(rc);
  return py::cast(out);
}

// ------------------------------------------------------------- tokenwise
// bytes of a tokenwise weight buffer, 0 for an unknown layout
int64_t tw_bytes(int layout, int64_t n, int64_t k) {
  switch (layout) {
    case ACTUNE_TW_KMAJOR_W8: return k * n;
    case ACTUNE_TW_KMAJOR_W4: case ACTUNE_TW_KMAJOR_W4R4: case ACTUNE_TW_ROWS_S4: return k / 2 * n;
    case ACTUNE_TW_KMAJOR_W2: case ACTUNE_TW_ROWS_S2: return k / 4 * n;
    default: return 0;
  }
}
bool tw_weights_ok(const Tensor& w, int layout, const Tensor& ws, const OptTensor& bias, const at::Device& dev, int64_t n,
                   int64_t k) {
  return plain(w, dev) && w.element_size() == 1 && n > 0 && k > 0 && w.numel() == tw_bytes(layout, n, k) && aligned(w) &&
         plain(ws, dev, at::kFloat) && ws.numel() == n && bias_ok(bias, dev, n);
}

py::object tokenwise_quantize(const Tensor& x, int bits) {
  if (!rows_ok(x) || (bits != 8 && bits != 4) || x.size(1) <= 0 || x.size(1) % 8) return py::none();
  const int64_t m = x.size(0), k = x.size(1);
  Tensor codes = empty({m, bits == 8 ? k : k / 2}, x.device(), bits == 8 ? at::kChar : at::kByte);
  Tensor scales = empty({m}, x.device(), at::kFloat);
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.tokenwise_quantize(x.const_data_ptr(), dtype_code(x.scalar_type()), m, k, bits, codes.mutable_data_ptr(),
                                scales.mutable_data_ptr<float>(), stream(x.device()));
  }
  check(rc);
  return py::make_tuple(codes, scales);
}

// The GEMM on codes, its split-K workspace included.
py::object tokenwise_linear(const Tensor& a, int a_layout, const Tensor& as, const Tensor& w, int w_layout,
                            const Tensor& ws, const OptTensor& bias, int64_t n, int64_t k, int epilogue, int out_code) {
  if (!a.is_cuda() || a.dim() != 2 || out_code < 0 || (a_layout != ACTUNE_TW_ACT_A8 && a_layout != ACTUNE_TW_ACT_A4))
    return py::none();
  const at::Device dev = a.device();
  const int64_t m = a.size(0);
  if (!plain(a, dev, a_layout == ACTUNE_TW_ACT_A8 ? at::kChar : at::kByte) || !aligned(a) ||
      a.size(1) != (a_layout == ACTUNE_TW_ACT_A8 ? k : k / 2) || !plain(as, dev, at::kFloat) || as.numel() != m ||
      w_layout == ACTUNE_TW_KMAJOR_W4R4 || !tw_weights_ok(w, w_layout, ws, bias, dev, n, k))
    return py::none();
  const int64_t need = api.tokenwise_workspace_bytes(m, n, k, w_layout, a_layout);
  if (need < 0) return py::none();
  Tensor out = empty({m, n}, dev, dtype_of(out_code)), work;
  if (need) work = empty({need}, dev, at::kByte);
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.tokenwise_linear(a.const_data_ptr(), a_layout, as.const_data_ptr<float>(), w.const_data_ptr(), w_layout,
                              ws.const_data_ptr<float>(), ptr(bias), bias_code(bias), out.mutable_data_ptr(), out_code, m,
                              n, k, epilogue, need ? work.mutable_data_ptr() : nullptr, need, stream(dev));
  }
  check(rc);
  return py::cast(out);
}

// Rows quantized inside the GEMM launch (1 to 8 rows of a K-major layout).
py::object tokenwise_linear_x(const Tensor& x, const Tensor& w, int w_layout, const Tensor& ws, const OptTensor& bias,
                              int64_t n, int64_t k, int epilogue) {
  if (!rows_ok(x) || x.size(0) < 1 || x.size(0) > 8 || x.size(1) != k ||
      !tw_weights_ok(w, w_layout, ws, bias, x.device(), n, k) || w_layout == ACTUNE_TW_KMAJOR_W4R4)
    return py::none();
  const at::Device dev = x.device();
  const int64_t m = x.size(0), need = api.tokenwise_workspace_bytes(m, n, k, w_layout, ACTUNE_TW_ACT_A8);
  if (need < 0) return py::none();
  const int code = dtype_code(x.scalar_type());
  // scales of the rows, then the split-K partial sums
  Tensor out = empty({m, n}, dev, x.scalar_type()), work = empty({256 + need}, dev, at::kByte);
  uint8_t* const base = static_cast<uint8_t*>(work.mutable_data_ptr());
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.tokenwise_linear_x(x.const_data_ptr(), code, reinterpret_cast<float*>(base), w.const_data_ptr(), w_layout,
                                ws.const_data_ptr<float>(), ptr(bias), bias_code(bias), out.mutable_data_ptr(), code, m, n,
                                k, epilogue, need ? base + 256 : nullptr, need, stream(dev));
  }
  check(rc);
  return py::cast(out);
}

// Sibling projections of one row, quantized inside the GEMM launch: outputs
// [groups, n]. residuals: one per projection, or none at all.
py::object tokenwise_decode(const Tensor& x, const std::vector<Tensor>& weights, const std::vector<OptTensor>& residuals,
                            const std::vector<Tensor>& scales, const std::vector<OptTensor>& biases, int w_layout,
                            int64_t n, int64_t k, int epilogue) {
  const size_t count = weights.size();
  if (!rows_ok(x) || x.size(0) != 1 || x.size(1) != k || count < 1 || count > ACTUNE_MAX_TARGETS || scales.size() != count ||
      biases.size() != count || residuals.size() != count)
    return py::none();
  const at::Device dev = x.device();
  const int code = dtype_code(x.scalar_type());
  actune_tw_target t[ACTUNE_MAX_TARGETS];
  const int64_t need = api.tokenwise_workspace_bytes(1, n, k, w_layout, ACTUNE_TW_ACT_A8);
  if (need < 0) return py::none();
  Tensor out = empty({(int64_t)count, n}, dev, x.scalar_type()), work = empty({256 + (int64_t)count * need}, dev, at::kByte);
  uint8_t* const base = static_cast<uint8_t*>(work.mutable_data_ptr());
  for (size_t i = 0; i < count; ++i) {
    if (!tw_weights_ok(weights[i], w_layout, scales[i], biases[i], dev, n, k) ||
        (residuals[i] && (!plain(*residuals[i], dev, at::kByte) || residuals[i]->numel() != tw_bytes(w_layout, n, k) ||
                          !aligned(*residuals[i]))) ||
        biases[i].has_value() != biases[0].has_value() || bias_code(biases[i]) != bias_code(biases[0]))
      return py::none();
    t[i] = actune_tw_target{weights[i].const_data_ptr(), ptr(residuals[i]), scales[i].const_data_ptr<float>(),
                            ptr(biases[i]), static_cast<uint8_t*>(out.mutable_data_ptr()) + i * n * x.element_size()};
  }
  int rc;
  {
    py::gil_scoped_release nogil;
    rc = api.tokenwise_linear_multi(nullptr, ACTUNE_TW_ACT_A8, x.const_data_ptr(), code, reinterpret_cast<float*>(base),
                                    w_layout, t, (int)count, bias_code(biases[0]), code, 1, n, k, epilogue,
                                    need ? base + 256 : nullptr, (int64_t)count * need, stream(dev));
  }
  check(rc);
  return py::cast(out);
}

}  // namespace

// A call whose arguments do not convert falls to the second overload.
template <typename F>
void def(py::module_& m, const char* name, F f) {
  m.def(name, f);
  m.def(name, [](const py::args&) { return py::none(); });
}

PYBIND11_MODULE(_actune_fast, m) {
  m.attr("torch_version") = TORCH_VERSION;
  m.def("init", &init);
  def(m, "quantize_groups", &quantize_groups);
  def(m, "quantize_gated", &quantize_gated);
  def(m, "grouped_linear", &grouped_linear);
  def(m, "grouped_forward", &grouped_forward);
  def(m, "grouped_forward_multi", &grouped_forward_multi);
  def(m, "tokenwise_quantize", &tokenwise_quantize);
  def(m, "tokenwise_linear", &tokenwise_linear);
  def(m, "tokenwise_linear_x", &tokenwise_linear_x);
  def(m, "tokenwise_decode", &tokenwise_decode);
}
