// MakePytorchBackend: the compiled extension module of the reference (pybind/bind.cpp:10-24,
// pybind/extern.hpp:1-9) re-built over libwinoconv_hip.so.  Same names, same positional signatures:
// Foo, AddGPU, WinoSplit, WinoConcat, DWM - plus the two entry points named after the reference's
// source files, winograd_conv (src/winograd_conv.cpp) and split_and_concat (src/split_and_concat.cpp).
//
// This file is plain C++ (g++, no device code): it checks devices, dtypes, shapes and contiguity,
// takes scratch memory from torch's caching allocator and the stream from torch's current HIP
// stream, releases the GIL, and calls the C ABI of include/winoconv.h.  Errors become Python
// exceptions (the reference prints and calls exit(-1): src/winograd_conv.cpp:80-84,116-126).
// Wider than the reference: float16 and bfloat16 are dispatched by tensor dtype (the reference binds
// float only: bind.cpp:19-23), stride 2 and every kernel extent 1..10 work.
#include <torch/extension.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <optional>
#include <sstream>
#include <stdexcept>
#include <string>
#include <thread>
#include <tuple>
#include <vector>

#include "../../../include/winoconv.h"

namespace py = pybind11;

namespace {

struct Unsupported : std::runtime_error { using std::runtime_error::runtime_error; };
struct WinoconvError : std::runtime_error { using std::runtime_error::runtime_error; };

// wc_status -> C++ exception (translated to ValueError / NotImplementedError / WinoconvError below)
void check(int rc) {
  if (rc == WC_OK) return;
  const std::string msg = wc_last_error();
  if (rc == WC_ERR_BAD_ARG) throw std::invalid_argument(msg);
  if (rc == WC_ERR_UNSUPPORTED) throw Unsupported(msg);
  throw WinoconvError("winoconv error " + std::to_string(rc) + ": " + msg);
}

int dtype_of(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return WC_F32;
    case at::kHalf: return WC_F16;
    case at::kBFloat16: return WC_BF16;
    default: {
      std::ostringstream os;
      os << "winoconv supports float32, float16 and bfloat16, got " << t.scalar_type();
      throw py::type_error(os.str());
    }
  }
}

void require_gpu(const at::Tensor& t, const char* what) {
  if (!t.is_cuda()) {
    std::ostringstream os;
    os << what << ": winoconv runs on the GPU only: got a " << t.device() << " tensor";
    throw std::invalid_argument(os.str());
  }
  dtype_of(t);
}

void* stream_of(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// Workspace of a call.  Small ones (the filter of a one-kernel layer: a few hundred KB, where the 1.6 us of an
// allocation is a visible part of a 10 us call) are kept per thread, device and stream: calls on one stream
// run in order, so the next call may write where the last one read.  A thread keeps at most kKeptSlots of them
// (4 MB): a further (device, stream) pair takes the slot used longest ago, whose tensor goes back to the caching
// allocator, which hands a block to later allocations of the stream it was allocated on only, in stream order.
// A thread that ends returns its workspaces; the thread that imported the module keeps them until the process ends
// (its thread-local objects are destroyed during exit(), when the interpreter has already been finalised).
// A stream under capture gets a fresh allocation from the graph's own pool instead.
const std::thread::id g_import_thread = std::this_thread::get_id();

struct KeptWorkspaces {
  struct Kept { int device; void* stream; at::Tensor ws; uint64_t used; };
  std::vector<Kept> slots;
  uint64_t clock = 0;
  ~KeptWorkspaces() {
    if (std::this_thread::get_id() == g_import_thread) new std::vector<Kept>(std::move(slots));   // never freed
  }
};

bool capturing(void* stream) {
  if (stream == nullptr) return false;          // the default stream cannot be captured
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(static_cast<hipStream_t>(stream), &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

at::Tensor workspace_for(const at::Tensor& like, size_t bytes, void* stream) {
  constexpr size_t kKept = 1u << 20;
  constexpr size_t kKeptSlots = 4;
  auto fresh = [&](size_t n) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); };
  if (bytes > kKept || capturing(stream)) return fresh(bytes);
  thread_local KeptWorkspaces kept;
  const int device = like.device().index();
  for (auto& k : kept.slots)
    if (k.device == device && k.stream == stream) {
      k.used = ++kept.clock;
      return k.ws;
    }
  if (kept.slots.size() < kKeptSlots) {
    kept.slots.push_back(KeptWorkspaces::Kept{device, stream, fresh(kKept), ++kept.clock});
    return kept.slots.back().ws;
  }
  auto* oldest = &kept.slots[0];
  for (auto& k : kept.slots)
    if (k.used < oldest->used) oldest = &k;
  *oldest = KeptWorkspaces::Kept{device, stream, fresh(kKept), ++kept.clock};
  return oldest->ws;
}

std::string shape_str(at::IntArrayRef s) {
  std::ostringstream os;
  os << "(";
  for (size_t i = 0; i < s.size(); ++i) os << (i ? ", " : "") << s[i];
  os << ")";
  return os.str();
}

void check_out(const at::Tensor& out, const std::vector<int64_t>& shape, const at::Tensor& like, const char* what) {
  if (out.sizes().vec() != shape || out.scalar_type() != like.scalar_type() || out.device() != like.device() ||
      !out.is_contiguous()) {
    std::ostringstream os;
    os << what << ": output must be a contiguous " << like.scalar_type() << " tensor of shape " << shape_str(shape)
       << " on " << like.device() << ", got " << shape_str(out.sizes());
    throw std::invalid_argument(os.str());
  }
}

// ---- template demo of the reference (src/foo.cpp, src/add.cpp:9-31), kept importable -----------------------
class Foo {
 public:
  void setKey(int key) { key_ = key; }
  int getKey() const { return key_; }
  std::string toString() const { return "< Foo, key: " + std::to_string(key_) + " > "; }
 private:
  int key_ = 0;
};

void AddGPU(at::Tensor in_a, at::Tensor in_b, at::Tensor out_c) {
  if (in_a.numel() != in_b.numel())
    throw std::invalid_argument("AddGPU: inputs must have the same number of elements");   // src/add.cpp:14-17
  out_c.resize_(in_a.sizes());
  at::add_out(out_c, in_a, in_b.view_as(in_a));
}

// ---- tile copies (src/split_and_concat.cpp:14-76) ---------------------------------------------------------------
void WinoSplit(at::Tensor in_a, at::Tensor out, int block_D, int block_H, int block_W, int output_block_size,
               int nD, int nH, int nW, bool two_dimension) {
  require_gpu(in_a, "WinoSplit");
  require_gpu(out, "WinoSplit");
  if (!in_a.is_contiguous()) throw std::invalid_argument("WinoSplit: in_a must be contiguous channel-last");
  if (in_a.dim() != (two_dimension ? 4 : 5))
    throw std::invalid_argument("WinoSplit: in_a must be (B, H, W, C) or (B, D, H, W, C), got " + shape_str(in_a.sizes()));
  const int es = (int)in_a.element_size(), m = output_block_size;
  void* st = stream_of(in_a);
  if (two_dimension) {
    const int B = in_a.size(0), H = in_a.size(1), W = in_a.size(2), C = in_a.size(3);
    check_out(out, {(int64_t)B * nH * nW, C, block_H, block_W}, in_a, "WinoSplit");
    py::gil_scoped_release nogil;
    check(wc_wino_split2d(in_a.data_ptr(), out.data_ptr(), B, H, W, C, block_H, block_W, m, nH, nW, es, st));
  } else {
    const int B = in_a.size(0), D = in_a.size(1), H = in_a.size(2), W = in_a.size(3), C = in_a.size(4);
    check_out(out, {(int64_t)B * nD * nH * nW, C, block_D, block_H, block_W}, in_a, "WinoSplit");
    py::gil_scoped_release nogil;
    check(wc_wino_split3d(in_a.data_ptr(), out.data_ptr(), B, D, H, W, C, block_D, block_H, block_W, m, nD, nH, nW,
                          es, st));
  }
}

// Like the reference (src/split_and_concat.cpp:44-76), the output extents are read from `out` and B follows
// from the tile count.
void WinoConcat(at::Tensor in_a, at::Tensor out, int output_block_size, bool two_dimension) {
  require_gpu(in_a, "WinoConcat");
  require_gpu(out, "WinoConcat");
  if (!in_a.is_contiguous() || !out.is_contiguous()) throw std::invalid_argument("WinoConcat: tensors must be contiguous");
  const int nd = two_dimension ? 2 : 3, m = output_block_size;
  if (in_a.dim() != nd + 2 || out.dim() != nd + 2 || m < 1)
    throw std::invalid_argument("WinoConcat: expected tiles (N, K, [m,] m, m) and a channel-last output");
  for (int a = 0; a < nd; ++a)
    if (in_a.size(2 + a) != m)
      throw std::invalid_argument("WinoConcat: tiles of shape " + shape_str(in_a.sizes()) + " for an output tile of " + std::to_string(m));
  const int64_t N = in_a.size(0), K = in_a.size(1);
  int64_t per = 1;
  for (int a = 0; a < nd; ++a) per *= (out.size(1 + a) + m - 1) / m;
  const int64_t B = per ? N / per : 0;
  if (B * per != N || out.size(0) != B || out.size(nd + 1) != K || out.scalar_type() != in_a.scalar_type()) {
    std::ostringstream os;
    os << "WinoConcat: " << N << " tiles of " << K << " channels do not fill an output of shape " << shape_str(out.sizes());
    throw std::invalid_argument(os.str());
  }
  const int es = (int)in_a.element_size();
  void* st = stream_of(in_a);
  py::gil_scoped_release nogil;
  if (two_dimension)
    check(wc_wino_concat2d(in_a.data_ptr(), out.data_ptr(), (int)B, (int)out.size(1), (int)out.size(2), (int)K, m, es, st));
  else
    check(wc_wino_concat3d(in_a.data_ptr(), out.data_ptr(), (int)B, (int)out.size(1), (int)out.size(2), (int)out.size(3),
                           (int)K, m, es, st));
}

void split_and_concat(const std::string& direction, at::Tensor in_a, at::Tensor out, py::args args) {
  if (direction == "split") {
    if (args.size() != 8) throw std::invalid_argument("split_and_concat('split', in_a, out, block_D, block_H, block_W, "
                                                      "output_block_size, nD, nH, nW, two_dimension)");
    WinoSplit(in_a, out, args[0].cast<int>(), args[1].cast<int>(), args[2].cast<int>(), args[3].cast<int>(),
              args[4].cast<int>(), args[5].cast<int>(), args[6].cast<int>(), args[7].cast<bool>());
  } else if (direction == "concat") {
    if (args.size() != 2) throw std::invalid_argument("split_and_concat('concat', in_a, out, output_block_size, two_dimension)");
    WinoConcat(in_a, out, args[0].cast<int>(), args[1].cast<bool>());
  } else {
    throw std::invalid_argument("split_and_concat: direction must be 'split' or 'concat'");
  }
}

// ---- whole convolution (src/winograd_conv.cpp:17-127) -----------------------------------------------------------------
// Input (B, D, H, W, C) contiguous; Weight any strided view with dims (kD, kH, kW, C, K) (the reference's
// layout, dwm.py:85,133); Output (B, oD, oH, oW, K) contiguous; a 2-D problem has D = kD = 1.  Returns the
// output tile really used (wc_conv_auto may replace 4 by 3 or 2).
int winograd_conv(at::Tensor Input, at::Tensor Weight, at::Tensor Output, std::optional<at::Tensor> bias, int stride,
                  py::object padding, int m, const std::string& algo, std::optional<at::Tensor> U, int chunk_images,
                  py::object stacked) {
  if (algo != "dwm" && algo != "whole") throw std::invalid_argument("winograd_conv: algo must be 'dwm' or 'whole', got '" + algo + "'");
  if (Input.dim() != 5 || Weight.dim() != 5 || Output.dim() != 5)
    throw std::invalid_argument("winograd_conv: expected 5-D channel-last Input/Output and a 5-D Weight");
  const int64_t K = Weight.size(4), C = Weight.size(3);
  if (bias && bias->defined()) {
    if (bias->dim() != 1 || bias->numel() != K)
      throw std::invalid_argument("bias must be a 1-D tensor of " + std::to_string(K) + " values (one per output channel), got shape " +
                                  shape_str(bias->sizes()));
    if (bias->scalar_type() != Input.scalar_type()) *bias = bias->to(Input.scalar_type());
    if (bias->device() != Input.device()) throw std::invalid_argument("bias and Input are on different devices");
    *bias = bias->contiguous();
  }
  if (U && U->defined()) {
    if (U->scalar_type() != Input.scalar_type()) {
      std::ostringstream os;
      os << "the transformed filter is " << U->scalar_type() << ", the input is " << Input.scalar_type()
         << ": transform the filter in the input's dtype";
      throw py::type_error(os.str());
    }
    if (U->device() != Input.device()) throw std::invalid_argument("the transformed filter and Input are on different devices");
  }
  require_gpu(Input, "winograd_conv");
  require_gpu(Weight, "winograd_conv");
  require_gpu(Output, "winograd_conv");
  if (!Input.is_contiguous() || !Output.is_contiguous()) throw std::invalid_argument("winograd_conv: Input and Output must be contiguous");
  if (Weight.scalar_type() != Input.scalar_type() || Output.scalar_type() != Input.scalar_type())
    throw py::type_error("winograd_conv: Input, Weight and Output must share one dtype");
  if (Input.size(4) != C)
    throw std::invalid_argument("winograd_conv: Input has " + std::to_string(Input.size(4)) + " channels, Weight expects " + std::to_string(C));

  wc_conv_desc d{};
  const bool flat = Input.size(1) == 1 && Weight.size(0) == 1;
  d.ndim = flat ? 2 : 3;
  d.N = (int)Input.size(0); d.C = (int)C; d.K = (int)K;
  for (int a = 0; a < 3; ++a) { d.in[a] = (int)Input.size(1 + a); d.kernel[a] = (int)Weight.size(a); }
  if (py::isinstance<py::int_>(padding)) {
    const int p = padding.cast<int>();
    d.pad[0] = flat ? 0 : p; d.pad[1] = p; d.pad[2] = p;
  } else {
    const auto p = padding.cast<std::vector<int>>();
    if (p.size() != 3) throw std::invalid_argument("winograd_conv: padding is one int or (pD, pH, pW)");
    for (int a = 0; a < 3; ++a) d.pad[a] = p[a];
  }
  d.stride = stride; d.m = m; d.dtype = dtype_of(Input);
  d.chunk_images = chunk_images;
  d.whole_kernel = algo == "whole";
  d.stacked = stacked.is_none() ? -1 : (py::isinstance<py::bool_>(stacked) ? (int)stacked.cast<bool>() : stacked.cast<int>());
  if (d.stacked > 2 || d.stacked < -1) throw std::invalid_argument("winograd_conv: stacked is None, False, True or 2");
  // the one-kernel path of thin layers wants 16-byte aligned operands; a legal view can start anywhere
  auto misaligned = [](const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) != 0; };
  d.unfused = misaligned(Input) || misaligned(Output) || (U && U->defined() && misaligned(*U));
  check(wc_conv_auto(&d));
  int out[3], grid[3];
  check(wc_conv_out_dims(&d, out, grid));
  check_out(Output, {d.N, out[0], out[1], out[2], d.K}, Input, "winograd_conv");
  if (U && U->defined()) {
    size_t ue = 0;
    check(wc_conv_u_elems(&d, &ue));
    if (!U->is_contiguous() || (size_t)U->numel() != ue)
      throw std::invalid_argument("U has " + std::to_string(U->numel()) + " elements, this convolution needs a contiguous transformed "
                                  "filter of " + std::to_string(ue) + " (transform_filter must be called with the same options)");
  }
  size_t bytes = 0;
  check(wc_conv_workspace_bytes(&d, &bytes));
  at::Tensor ws = at::empty({(int64_t)bytes}, Input.options().dtype(at::kByte));        // torch's caching allocator
  // Weight is (kD, kH, kW, C, K): its strides in (K, C, kD, kH, kW) order, no copy
  const int64_t s[5] = {Weight.stride(4), Weight.stride(3), Weight.stride(0), Weight.stride(1), Weight.stride(2)};
  void* st = stream_of(Input);
  const void* bp = bias && bias->defined() ? bias->data_ptr() : nullptr;
  const void* up = U && U->defined() ? U->data_ptr() : nullptr;
  {
    py::gil_scoped_release nogil;
    check(wc_conv_forward(&d, Input.data_ptr(), Weight.data_ptr(), s, up, bp, Output.data_ptr(), ws.data_ptr(), bytes, st));
  }
  return d.m;
}

std::vector<int> ints_of(const py::object& v, int nd, const char* what) {
  std::vector<int> r;
  if (py::isinstance<py::int_>(v)) {
    r.assign(nd, v.cast<int>());
  } else {
    r = v.cast<std::vector<int>>();
    if ((int)r.size() != nd) throw std::invalid_argument(std::string(what) + ": expected one int or " + std::to_string(nd) + " values");
  }
  return r;
}

int spatial_dims(at::IntArrayRef x, at::IntArrayRef w) {
  if ((x.size() != 4 && x.size() != 5) || w.size() != x.size())
    throw std::invalid_argument("expected 4-D or 5-D input and matching filter, got " + shape_str(x) + " and " + shape_str(w));
  return (int)x.size() - 2;
}

int one_stride(const py::object& stride, int nd) {
  const auto st = ints_of(stride, nd, "stride");
  for (int a = 1; a < nd; ++a)
    if (st[a] != st[0]) throw Unsupported("stride must be the same on every axis");
  return st[0];
}

// Winograd / DWM convolution of an NC[D]HW tensor with a (K, C, [kD,] kH, kW) filter; returns an NC[D]HW
// tensor whose memory is channel-last (or plain contiguous with channels_first_out).  A channel-last input is
// used without a copy and a contiguous channel-first one is handed to the library as it is
// (wc_conv_desc.x_layout); any other layout is made contiguous first.  The compiled form of the Python callers' common path (dwm.py:5-40, matrix_conv.py:70-135
// of the reference end in the same call).
// `flipped`: the filter is w reversed along every spatial axis, read through negative strides.
// No function from here to the gradients touches Python: they run with and without the interpreter lock.
struct ConvOptions {
  int chunk_images = 0, stacked = -1, direct = 0;      // -1: the library chooses the form of the plan; 0: it may take the direct one
  bool whole_kernel = false, unfused = false, channels_first_out = false, row = false, flipped = false;
};

at::Tensor conv_impl(at::Tensor x, const at::Tensor& w, const std::optional<at::Tensor>& bias, int stride, const std::vector<int>& pd, int m,
                     std::optional<at::Tensor> U, const ConvOptions& o) {
  const int nd = spatial_dims(x.sizes(), w.sizes());
  if (x.size(1) != w.size(1))
    throw std::invalid_argument("input has " + std::to_string(x.size(1)) + " channels, filter expects " + std::to_string(w.size(1)) +
                                " (groups are not supported)");
  const int64_t K = w.size(0);
  if (bias && bias->defined()) {
    if (bias->dim() != 1 || bias->numel() != K)
      throw std::invalid_argument("bias must be a 1-D tensor of " + std::to_string(K) + " values (one per output channel), got shape " +
                                  shape_str(bias->sizes()));
    if (bias->scalar_type() != x.scalar_type()) {
      std::ostringstream os;
      os << "bias is " << bias->scalar_type() << ", the input is " << x.scalar_type() << ": they must share one dtype";
      throw py::type_error(os.str());
    }
    if (bias->device() != x.device()) throw std::invalid_argument("bias and input are on different devices");
  }
  if (U && U->defined()) {
    if (U->scalar_type() != x.scalar_type()) {
      std::ostringstream os;
      os << "the transformed filter is " << U->scalar_type() << ", the input is " << x.scalar_type()
         << ": transform the filter in the input's dtype";
      throw py::type_error(os.str());
    }
    if (U->device() != x.device()) throw std::invalid_argument("the transformed filter and the input are on different devices");
  }
  require_gpu(x, "conv_forward");
  require_gpu(w, "conv_forward");
  if (w.scalar_type() != x.scalar_type()) throw py::type_error("input, filter and bias must share one dtype");
  wc_conv_desc d{};
  d.ndim = nd;
  d.N = (int)(x.size(0) > 0 ? x.size(0) : 1);      // an empty batch: the shape arithmetic runs on one image
  d.C = (int)x.size(1); d.K = (int)K;
  d.in[0] = d.kernel[0] = 1;
  for (int a = 0; a < nd; ++a) {
    d.in[3 - nd + a] = (int)x.size(2 + a);
    d.kernel[3 - nd + a] = (int)w.size(2 + a);
    d.pad[3 - nd + a] = pd[a];
  }
  d.stride = stride; d.m = m; d.dtype = dtype_of(x);
  d.chunk_images = o.chunk_images;
  d.whole_kernel = o.whole_kernel;
  d.stacked = o.stacked;
  d.direct = o.direct;
  d.unfused = o.unfused;
  d.row = o.row && !o.unfused ? -1 : 0;                                   // -1: the library may choose it
  check(wc_conv_auto(&d));
  int out[3], grid[3];
  check(wc_conv_out_dims(&d, out, grid));
  std::vector<int64_t> ys{x.size(0)};                      // channel-last shape of y
  for (int a = 3 - nd; a < 3; ++a) ys.push_back(out[a]);
  ys.push_back(K);
  std::vector<int64_t> to_cl{0}, to_cf{0, nd + 1};
  for (int a = 0; a < nd; ++a) { to_cl.push_back(2 + a); to_cf.push_back(1 + a); }
  to_cl.push_back(1);
  std::vector<int64_t> ys_cf{ys[0], K};
  for (int a = 0; a < nd; ++a) ys_cf.push_back(ys[1 + a]);
  at::Tensor y = at::empty(o.channels_first_out ? ys_cf : ys, x.options());
  if (x.size(0) == 0) return o.channels_first_out ? y : y.permute(to_cf);
  at::Tensor x_mem = x.permute(to_cl);
  if (!x_mem.is_contiguous()) {                            // not channel-last memory: channel-first, read as it is
    x_mem = x.is_contiguous() ? x : x.contiguous();
    d.x_layout = 1;
  }
  d.y_layout = o.channels_first_out;
  auto misaligned = [](const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) != 0; };
  if (d.row) {                                             // the row form reads aligned operands: copies of those that are not
    if (misaligned(x_mem)) x_mem = x_mem.clone();
    if (U && U->defined() && misaligned(*U)) U = U->clone();
  }
  d.unfused = o.unfused || misaligned(x_mem) || (U && U->defined() && misaligned(*U));
  if (U && U->defined()) {
    size_t ue = 0;
    check(wc_conv_u_elems(&d, &ue));
    if (!U->is_contiguous() || (size_t)U->numel() != ue)
      throw std::invalid_argument("U has " + std::to_string(U->numel()) + " elements, this convolution needs a contiguous transformed "
                                  "filter of " + std::to_string(ue) + " (transform_filter must be called with the same options)");
  }
  size_t bytes = 0;
  check(wc_conv_workspace_bytes(&d, &bytes));
  void* stream = stream_of(x);
  at::Tensor ws = workspace_for(x, bytes, stream);
  at::Tensor bc = bias && bias->defined() ? bias->contiguous() : at::Tensor();
  int64_t s[5] = {w.stride(0), w.stride(1), 0, 0, 0};
  for (int a = 0; a < nd; ++a) s[5 - nd + a] = w.stride(2 + a);
  const unsigned char* wp = static_cast<const unsigned char*>(w.data_ptr());
  if (o.flipped)
    for (int a = 0; a < nd; ++a) {
      wp += (w.size(2 + a) - 1) * w.stride(2 + a) * w.element_size();
      s[5 - nd + a] = -w.stride(2 + a);
    }
  check(wc_conv_forward(&d, x_mem.data_ptr(), wp, s, U && U->defined() ? U->data_ptr() : nullptr,
                        bc.defined() ? bc.data_ptr() : nullptr, y.data_ptr(), ws.data_ptr(), bytes, stream));
  return o.channels_first_out ? y : y.permute(to_cf);
}

at::Tensor conv_forward(at::Tensor x, at::Tensor w, std::optional<at::Tensor> bias, py::object stride, py::object padding,
                        int m, std::optional<at::Tensor> U, int chunk_images, bool whole_kernel, py::object stacked,
                        bool unfused, bool channels_first_out, py::object direct, bool row) {
  const int nd = spatial_dims(x.sizes(), w.sizes());
  ConvOptions o;
  o.chunk_images = chunk_images; o.whole_kernel = whole_kernel; o.unfused = unfused; o.channels_first_out = channels_first_out; o.row = row;
  o.stacked = stacked.is_none() ? -1 : (py::isinstance<py::bool_>(stacked) ? (int)stacked.cast<bool>() : stacked.cast<int>());
  o.direct = direct.is_none() ? 0 : (direct.cast<bool>() ? 1 : -1);
  const int st = one_stride(stride, nd);
  const auto pd = ints_of(padding, nd, "padding");
  py::gil_scoped_release nogil;
  return conv_impl(std::move(x), w, bias, st, pd, m, std::move(U), o);
}

// Input gradient of a stride-1 layer: dy convolved with w flipped and its channel axes exchanged; `padding` is that
// convolution's.
at::Tensor backward_input_flipped(const at::Tensor& dy, const at::Tensor& w, const std::vector<int>& pads, int m) {
  ConvOptions o;
  o.row = o.flipped = true;
  return conv_impl(dy, w.transpose(0, 1), std::nullopt, 1, pads, m, std::nullopt, o);
}

at::Tensor conv_backward_input_flipped(at::Tensor dy, at::Tensor w, py::object padding, int m) {
  const auto pads = ints_of(padding, (int)dy.dim() - 2, "padding");
  py::gil_scoped_release nogil;
  return backward_input_flipped(dy, w, pads, m);
}

at::Tensor last_view(const at::Tensor& t) {       // (N, C, *) -> (N, *, C), contiguous
  std::vector<int64_t> order{0};
  for (int64_t a = 2; a < t.dim(); ++a) order.push_back(a);
  order.push_back(1);
  const at::Tensor v = t.permute(order);
  const int es = (int)t.element_size();
  if (v.is_contiguous() || !t.is_contiguous() || t.numel() == 0 || (es != 2 && es != 4)) return v.contiguous();
  // channel-first memory: the library's copy moves 16 bytes a lane (64 x 128 x 112 x 112 fp16 148 us by torch, 13 x 411 x 28 x 19 17)
  at::Tensor out = at::empty(v.sizes(), t.options());
  check(wc_layout_copy(t.data_ptr(), out.data_ptr(), (int)t.size(0), (int)t.size(1), t.numel() / (t.size(0) * t.size(1)), 1, es, stream_of(t)));
  return out;
}

wc_conv_desc desc_of(at::IntArrayRef x, at::IntArrayRef w, const std::vector<int>& pads, int stride, int m, int dtype) {
  const int nd = (int)x.size() - 2;
  wc_conv_desc d{};
  d.ndim = nd;
  d.N = (int)x[0]; d.C = (int)x[1]; d.K = (int)w[0];
  d.in[0] = d.kernel[0] = 1;
  for (int a = 0; a < nd; ++a) {
    d.in[3 - nd + a] = (int)x[2 + a];
    d.kernel[3 - nd + a] = (int)w[2 + a];
    d.pad[3 - nd + a] = pads[a];
  }
  d.stride = stride; d.m = m; d.dtype = dtype;
  return d;
}

void strides_of(const at::Tensor& w, int64_t s[5]) {
  const int nd = (int)w.dim() - 2;
  s[0] = w.stride(0); s[1] = w.stride(1);
  for (int a = 0; a < 3; ++a) s[2 + a] = a < 3 - nd ? 0 : w.stride(2 + a - (3 - nd));
}

// Input gradient of a 2-D layer at stride 2 over the parity classes of its pixels (wc_conv_backward_input); an undefined
// tensor, and nothing launched, where that does not apply.  engine.py's conv_backward_input has checked the padding.
at::Tensor backward_input_strided(const at::Tensor& dy, const at::Tensor& w, at::IntArrayRef x_spatial, const std::vector<int>& pads) {
  require_gpu(dy, "conv_backward_input");
  require_gpu(w, "conv_backward_input");
  wc_conv_desc d = desc_of({dy.size(0), w.size(1), x_spatial[0], x_spatial[1]}, w.sizes(), pads, 2, 2, dtype_of(dy));
  int out[3], grid[3];
  check(wc_conv_out_dims(&d, out, grid));
  if (dy.size(2) != out[1] || dy.size(3) != out[2])
    throw std::invalid_argument("dy of shape " + shape_str(dy.sizes()) + " does not belong to an input of extent " + shape_str(x_spatial));
  size_t bytes = 0;
  if (wc_conv_backward_input_workspace_bytes(&d, &bytes) != WC_OK) return at::Tensor();
  if (w.scalar_type() != dy.scalar_type()) throw py::type_error("dy and the filter must share one dtype");
  const at::Tensor dyl = last_view(dy);
  at::Tensor dx = at::empty({dy.size(0), x_spatial[0], x_spatial[1], w.size(1)}, dy.options());
  void* stream = stream_of(dy);
  at::Tensor ws = workspace_for(dy, bytes, stream);
  int64_t s[5];
  strides_of(w, s);
  check(wc_conv_backward_input(&d, dyl.data_ptr(), w.data_ptr(), s, dx.data_ptr(), ws.data_ptr(), bytes, stream));
  return dx.permute({0, 3, 1, 2});
}

at::Tensor conv_backward_input_strided(at::Tensor dy, at::Tensor w, std::vector<int64_t> x_spatial, std::vector<int> pads) {
  py::gil_scoped_release nogil;
  return backward_input_strided(dy, w, x_spatial, pads);
}

// engine.py's transform_filter with the form left to the library, the row form allowed
at::Tensor transform_filter(at::Tensor w, std::vector<int64_t> x_shape, py::object stride, py::object padding, int m) {
  const int nd = (int)w.dim() - 2;
  require_gpu(w, "transform_filter");
  if ((nd != 2 && nd != 3) || (int)x_shape.size() != nd + 2)
    throw std::invalid_argument("expected 4-D or 5-D input and matching filter, got " + shape_str(x_shape) + " and " + shape_str(w.sizes()));
  if (x_shape[1] != w.size(1))
    throw std::invalid_argument("input has " + std::to_string(x_shape[1]) + " channels, filter expects " + std::to_string(w.size(1)) +
                                " (groups are not supported)");
  const int st = one_stride(stride, nd);
  wc_conv_desc d = desc_of(x_shape, w.sizes(), ints_of(padding, nd, "padding"), st, m, dtype_of(w));
  d.stacked = d.row = -1;
  check(wc_conv_auto(&d));
  wc_plan plan{};
  size_t n = 0;
  check(wc_conv_u_elems(&d, &n));
  std::vector<int64_t> shape{(int64_t)n};
  if (d.direct) {          // taps outermost, channels innermost; first layers have their own rows
    if (nd == 3) shape = {d.K, d.kernel[0] * d.kernel[1], 4, 4};
    else if (n == (size_t)d.K * d.kernel[1] * d.kernel[2] * d.C) shape = {d.K, d.kernel[1], d.kernel[2], d.C};
    else shape = {d.K, d.kernel[1], 8, 4};
  } else if (!d.row) {
    check(wc_plan_conv(&d, &plan));
    shape = {plan.t_total, d.K, (int64_t)wc_padded_channels(d.C) * (d.stacked ? plan.n_pieces : 1)};
  }
  at::Tensor U = at::empty(shape, w.options().memory_format(at::MemoryFormat::Contiguous));
  int64_t s[5];
  strides_of(w, s);
  void* stream = stream_of(w);
  {
    py::gil_scoped_release nogil;
    check(wc_filter_transform(&d, &plan, w.data_ptr(), s, U.data_ptr(), stream));
  }
  return U;
}

// ---- gradients (the reference has no backward pass: src/back/utils.cu:15-24): engine.py's conv_backward_weight with the
// form of the plan left to the library, and bias_gradient
// (dw, db) with `bias`, each of type fp32 or x's
std::pair<at::Tensor, at::Tensor> parameter_gradients(const at::Tensor& x, const at::Tensor& dy, at::IntArrayRef w_shape, int stride,
                                                      const std::vector<int>& pd, int m, bool bias, at::ScalarType w_type, at::ScalarType b_type) {
  const int nd = (int)x.dim() - 2;
  require_gpu(x, "conv_backward_weight");
  require_gpu(dy, "conv_backward_weight");
  if (dy.scalar_type() != x.scalar_type()) throw py::type_error("x and dy must share one dtype");
  if ((nd != 2 && nd != 3) || (int)w_shape.size() != nd + 2)
    throw std::invalid_argument("expected 4-D or 5-D input and matching filter, got " + shape_str(x.sizes()) + " and " + shape_str(w_shape));
  if (x.size(1) != w_shape[1])
    throw std::invalid_argument("input has " + std::to_string(x.size(1)) + " channels, filter expects " + std::to_string(w_shape[1]) +
                                " (groups are not supported)");
  wc_conv_desc d{};
  d.ndim = nd;
  d.C = (int)x.size(1); d.K = (int)w_shape[0];
  d.kernel[0] = d.in[0] = 1;
  for (int a = 0; a < nd; ++a) d.kernel[3 - nd + a] = (int)w_shape[2 + a];
  d.stride = stride; d.m = m; d.dtype = dtype_of(x);
  // the Winograd / DWM form of the forward plan, the direct one aside, whatever the batch; the gradient has no form whose
  // pieces share one transformed input: pieces stacked with their own V
  wc_conv_desc form = d;
  form.N = 1; form.in[0] = 0; form.stacked = -1; form.direct = -1;
  check(wc_conv_auto(&form));
  d.N = (int)x.size(0);
  for (int a = 0; a < nd; ++a) { d.in[3 - nd + a] = (int)x.size(2 + a); d.pad[3 - nd + a] = pd[a]; }
  d.stacked = form.stacked != 0;
  check(wc_conv_auto(&d));
  int out[3], grid[3];
  check(wc_conv_out_dims(&d, out, grid));
  std::vector<int64_t> ys{x.size(0), w_shape[0]};
  for (int a = 3 - nd; a < 3; ++a) ys.push_back(out[a]);
  if (dy.sizes() != at::IntArrayRef(ys)) throw std::invalid_argument("dy has shape " + shape_str(dy.sizes()) + ", the convolution gives " + shape_str(ys));
  at::Tensor dw = at::empty(w_shape, x.options().dtype(w_type)), db;
  if (bias) db = at::empty({w_shape[0]}, x.options().dtype(b_type));
  const bool plain = !bias && w_type == x.scalar_type();
  const at::Tensor xl = last_view(x), dyl = last_view(dy);
  size_t bytes = 0;
  check(plain ? wc_conv_backward_weight_workspace_bytes(&d, &bytes) : wc_conv_backward_parameters_workspace_bytes(&d, &bytes));
  void* stream = stream_of(x);
  at::Tensor ws = workspace_for(x, bytes, stream);
  int64_t s[5] = {dw.stride(0), dw.stride(1), 0, 0, 0};
  for (int a = 0; a < nd; ++a) s[5 - nd + a] = dw.stride(2 + a);
  check(plain ? wc_conv_backward_weight(&d, xl.data_ptr(), dyl.data_ptr(), dw.data_ptr(), s, ws.data_ptr(), bytes, stream)
              : wc_conv_backward_parameters(&d, xl.data_ptr(), dyl.data_ptr(), dw.data_ptr(), s, dtype_of(dw), bias ? db.data_ptr() : nullptr,
                                            bias ? dtype_of(db) : WC_F32, ws.data_ptr(), bytes, stream));
  return {dw, db};
}

at::Tensor conv_backward_weight(at::Tensor x, at::Tensor dy, std::vector<int64_t> w_shape, py::object stride, py::object padding, int m) {
  const int nd = (int)x.dim() - 2, st = one_stride(stride, nd);
  const auto pd = ints_of(padding, nd, "padding");
  py::gil_scoped_release nogil;
  return parameter_gradients(x, dy, w_shape, st, pd, m, false, x.scalar_type(), x.scalar_type()).first;
}

py::object or_none(const at::Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

py::tuple conv_backward_parameters(at::Tensor x, at::Tensor dy, std::vector<int64_t> w_shape, py::object stride, py::object padding, int m,
                                   bool need_db, py::object w_type, py::object b_type) {
  const int nd = (int)x.dim() - 2, st = one_stride(stride, nd);
  const auto pd = ints_of(padding, nd, "padding");
  const auto wt = torch::python::detail::py_object_to_dtype(w_type), bt = torch::python::detail::py_object_to_dtype(b_type);
  std::pair<at::Tensor, at::Tensor> g;
  {
    py::gil_scoped_release nogil;
    g = parameter_gradients(x, dy, w_shape, st, pd, m, need_db, wt, bt);
  }
  return py::make_tuple(g.first, or_none(g.second));
}

at::Tensor bias_gradient(at::Tensor dy) {
  require_gpu(dy, "bias_gradient");
  at::Tensor db = at::empty({dy.size(1)}, dy.options());
  const int64_t rows = dy.numel() / dy.size(1);
  const at::Tensor dyl = last_view(dy);
  size_t bytes = 0;
  check(wc_bias_gradient_workspace_bytes(rows, (int)dy.size(1), dtype_of(dy), &bytes));
  void* stream = stream_of(dy);
  at::Tensor ws = workspace_for(dy, bytes, stream);
  py::gil_scoped_release nogil;
  check(wc_bias_gradient(dyl.data_ptr(), db.data_ptr(), rows, (int)dy.size(1), dtype_of(dy), ws.data_ptr(), bytes, stream));
  return db;
}

bool channel_last_memory(const at::Tensor& t) {
  std::vector<int64_t> last{0};
  for (int64_t a = 2; a < t.dim(); ++a) last.push_back(a);
  last.push_back(1);
  return t.permute(last).is_contiguous();
}

// All gradients of a layer in one call, each in the type of what it belongs to: undefined for what is not asked for and for what
// engine.py's functions have to do (an input gradient that neither function above has, the bias gradient of a dy that is not
// channel-last memory).
struct Gradients { at::Tensor dx, dw, db; };

Gradients backward_all(const at::Tensor& x, const at::Tensor& w, const at::Tensor& dy, int stride, const std::vector<int>& pd, int m,
                       bool need_dx, bool need_dw, bool need_db, at::ScalarType w_type, at::ScalarType b_type) {
  const int nd = spatial_dims(x.sizes(), w.sizes());
  if (dy.dim() != x.dim())
    throw std::invalid_argument("expected 4-D or 5-D input and matching filter, got " + shape_str(x.sizes()) + " and " + shape_str(w.sizes()));
  Gradients g;
  if (need_dx) {
    std::vector<int> flipped(nd);
    bool fits = true;
    for (int a = 0; a < nd; ++a) {
      flipped[a] = (int)w.size(2 + a) - 1 - pd[a];
      fits = fits && flipped[a] >= 0;
    }
    const at::IntArrayRef size = x.sizes().slice(2);
    if (fits && stride == 1) {
      bool threes = true;
      for (int a = 0; a < nd; ++a) threes = threes && w.size(2 + a) == 3;
      const int tile = w.size(0) >= 8 && (m == 2 || nd == 2 || threes) ? m : 2;      // as in engine.py's conv_backward_input
      at::Tensor t = backward_input_flipped(dy, w, flipped, tile);
      if (t.sizes().slice(2) == size) g.dx = t;
    } else if (fits && nd == 2 && stride == 2) {
      g.dx = backward_input_strided(dy, w, size, pd);
    }
  }
  if (need_dw) {
    auto own = [&](at::ScalarType t) { return t == at::kFloat ? t : x.scalar_type(); };      // any other type: a cast of its own
    std::tie(g.dw, g.db) = parameter_gradients(x, dy, w.sizes(), stride, pd, m, need_db && channel_last_memory(dy), own(w_type), own(b_type));
    g.dw = g.dw.to(w_type);
    if (g.db.defined()) g.db = g.db.to(b_type);
  }
  return g;
}

py::tuple conv_backward(at::Tensor x, at::Tensor w, at::Tensor dy, py::object stride, py::object padding, int m, bool need_dx,
                        bool need_dw, bool need_db, py::object w_type, py::object b_type) {
  const int nd = spatial_dims(x.sizes(), w.sizes()), st = one_stride(stride, nd);
  const auto pd = ints_of(padding, nd, "padding");
  auto type = [&](const py::object& t) { return t.is_none() ? x.scalar_type() : torch::python::detail::py_object_to_dtype(t); };
  const at::ScalarType wt = type(w_type), bt = type(b_type);
  Gradients g;
  {
    py::gil_scoped_release nogil;
    g = backward_all(x, w, dy, st, pd, m, need_dx, need_dw, need_db, wt, bt);
  }
  return py::make_tuple(or_none(g.dx), or_none(g.dw), or_none(g.db));
}

// ---- a module's transformed filter between its passes --------------------------------------------------------------------
// It is the filter of one weight in one form of the plan: the weak pointer keeps the storage's identity and not its memory (weights that are new tensors in every pass,
// as functional_call and parametrizations make them, come to lie where the last one did).  It was made on one stream; a pass on another waits for
// that, once, and its memory is given back when the passes of all of them are through with it.  (engine.py's _KeptFilter does the same without
// this module.)
// direct, stacked, tile, row and the elements of the filter (fewer for an image of depth 1, whose plan has no tile along it): what a transformed
// filter depends on beside the weight and the type
using PlanForm = std::tuple<int, int, int, int, int64_t>;

class KeptFilter {
 public:
  // `weight` before anything is read of it: what changes it from here on makes it another one
  KeptFilter(const at::Tensor& weight, const PlanForm& form)
      : form_(form), version_((uint32_t)weight._version()), storage_(weight.storage().getWeakStorageImpl()), data_(weight.data_ptr()), strides_(weight.strides().vec()) {}

  // u: what was launched for it on the current stream
  void made(const at::Tensor& u) {
    U_ = u;
    stream_ = stream_of(u);
    captured_ = capturing(stream_);
  }

  // In the place of `last`: filters that graphs were captured with are kept for as long as those may be replayed, which is the module's life
  void follows(const std::shared_ptr<KeptFilter>& last) { before_ = !last || last->in_graph_ ? last : last->before_; }

  // made inside a capture: there when the graph is replayed, and only then.  Not for other passes
  bool captured() const { return captured_; }

  bool holds(const at::Tensor& weight) const {
    return !weight.is_inference() && (uint32_t)weight._version() == version_ && weight.data_ptr() == data_ && weight.strides() == at::IntArrayRef(strides_) &&
           weight.storage().unsafeGetStorageImpl() == storage_._unsafe_get_target();
  }

  // a 16-byte aligned U of this form and type
  bool suits(const PlanForm& form, at::ScalarType type, at::Device device) const {
    return U_.defined() && form == form_ && U_.numel() == std::get<4>(form) && U_.scalar_type() == type && U_.device() == device && U_.is_contiguous() &&
           (reinterpret_cast<uintptr_t>(U_.data_ptr()) & 15) == 0;
  }

  // U for a launch on the current stream; undefined where that cannot be ordered behind U's making.  (A capture cannot wait for what is outside
  // of it: its caller has, before the first replay, as for every other tensor that a graph reads.)  Undefined too where none was made: the
  // weight of a pass whose kernel took the filter as it is.
  at::Tensor on_stream() const {
    if (!U_.defined()) return U_;
    void* const now = stream_of(U_);
    const bool graph = capturing(now);
    if (graph) in_graph_ = true;
    if (now == stream_ || graph) return U_;
    const std::lock_guard<std::mutex> lock(mutex_);
    if (std::find(ordered_.begin(), ordered_.end(), now) != ordered_.end()) return U_;
    if (capturing(stream_)) return at::Tensor();
    const c10::DeviceGuard device(U_.device());
    hipEvent_t event;
    bool ok = hipEventCreateWithFlags(&event, hipEventDisableTiming) == hipSuccess;
    if (ok) {
      ok = hipEventRecord(event, static_cast<hipStream_t>(stream_)) == hipSuccess && hipStreamWaitEvent(static_cast<hipStream_t>(now), event, 0) == hipSuccess;
      (void)hipEventDestroy(event);
    }
    if (!ok) {                                      // a stream that is no more
      (void)hipGetLastError();
      return at::Tensor();
    }
    U_.record_stream(c10::impl::VirtualGuardImpl(U_.device().type()).getStream(U_.device()));
    ordered_.push_back(now);
    return U_;
  }

 private:
  PlanForm form_;
  uint32_t version_;
  c10::weak_intrusive_ptr<c10::StorageImpl> storage_;
  const void* data_;
  std::vector<int64_t> strides_;
  at::Tensor U_;
  void* stream_ = nullptr;
  bool captured_ = false;
  mutable std::atomic<bool> in_graph_{false};
  std::shared_ptr<KeptFilter> before_;              // read by a graph
  mutable std::mutex mutex_;
  mutable std::vector<void*> ordered_;              // streams that have waited
};

// a tensor with memory of its own on the GPU: no wrapper of a function transform, no subclass, nothing that carries a tangent
bool plain(const at::Tensor& t) {
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped) && !t._fw_grad(0).defined();
}

// Split_and_Concat.py's two functions for the arguments that they are called with in earnest (tensors of the GPU, sequences of ints); None for
// anything else, for what they refuse and for what the library does, which they then find and say themselves.  Through ctypes a call of
// each took 22 to 23 us of host time together, which is what all but the largest images waited for; here 9.5 to 10.3, two launches.
std::optional<std::vector<int64_t>> whole_numbers(py::handle h, size_t count) {
  const bool tuple = PyTuple_Check(h.ptr());
  if ((!tuple && !PyList_Check(h.ptr())) || (size_t)(tuple ? PyTuple_GET_SIZE(h.ptr()) : PyList_GET_SIZE(h.ptr())) != count) return std::nullopt;
  std::vector<int64_t> v(count);
  for (size_t i = 0; i < count; ++i) {
    PyObject* const o = tuple ? PyTuple_GET_ITEM(h.ptr(), i) : PyList_GET_ITEM(h.ptr(), i);
    if (!PyLong_CheckExact(o)) return std::nullopt;
    int over = 0;
    v[i] = PyLong_AsLongLongAndOverflow(o, &over);
    if (over || v[i] < 1 || v[i] >= (1 << 30)) return std::nullopt;
  }
  return v;
}

// a tensor of the kernels' types with memory of its own on the GPU, its extents ints
const at::Tensor* tile_tensor(py::handle h) {
  if (!THPVariable_Check(h.ptr())) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(h.ptr());
  const auto type = t.scalar_type();
  if (!plain(t) || (type != at::kFloat && type != at::kHalf && type != at::kBFloat16) || torch::jit::tracer::isTracing()) return nullptr;
  for (const int64_t v : t.sizes())
    if (v < 1 || v >= (1 << 30)) return nullptr;
  return &t;
}

std::optional<int> tile_extent(py::handle h) {
  if (!PyLong_CheckExact(h.ptr())) return std::nullopt;
  int over = 0;
  const int64_t m = PyLong_AsLongLongAndOverflow(h.ptr(), &over);
  return over || m < 1 || m > 1024 ? std::nullopt : std::optional<int>((int)m);
}

py::object wino_split(py::handle a_, py::handle w_shape, py::handle m_) {
  const at::Tensor* const a = tile_tensor(a_);
  const auto m = tile_extent(m_);
  if (!a || !m) return py::none();
  const int nd = (int)a->dim() - 2;
  if (nd != 2 && nd != 3) return py::none();
  const auto w = whole_numbers(w_shape, nd + 2);
  if (!w) return py::none();
  int sp[3] = {1, 1, 1}, block[3] = {1, 1, 1}, n[3] = {1, 1, 1};
  int64_t tiles = a->size(0);
  std::vector<int64_t> shape{0, a->size(1)};
  for (int q = 0; q < nd; ++q) {
    const int at = 3 - nd + q;
    sp[at] = (int)a->size(2 + q);
    const int64_t extent = (*w)[2 + q] + *m - 1;
    if (extent > sp[at]) return py::none();
    block[at] = (int)extent;
    n[at] = (sp[at] - block[at] + 1) / *m + 1;         // of a float's whole part: 1 + (X + 1 - b) / m
    tiles *= n[at];
    shape.push_back(extent);
  }
  shape[0] = tiles;
  at::Tensor out, src;
  int rc;
  {
    py::gil_scoped_release nogil;
    const int es = (int)a->element_size(), B = (int)a->size(0), C = (int)a->size(1);
    const bool first = a->is_contiguous() && !channel_last_memory(*a) && (es == 4 || (*m % 2 == 0 && block[2] % 2 == 0));
    src = first ? *a : last_view(*a).contiguous();
    out = at::empty(shape, a->options());
    void* const stream = stream_of(*a);
    if (first)
      rc = wc_wino_split_channel_first(src.data_ptr(), out.data_ptr(), B, C, sp[0], sp[1], sp[2], block[0], block[1], block[2], *m, n[0], n[1], n[2], es, stream);
    else if (nd == 2)
      rc = wc_wino_split2d(src.data_ptr(), out.data_ptr(), B, sp[1], sp[2], C, block[1], block[2], *m, n[1], n[2], es, stream);
    else
      rc = wc_wino_split3d(src.data_ptr(), out.data_ptr(), B, sp[0], sp[1], sp[2], C, block[0], block[1], block[2], *m, n[0], n[1], n[2], es, stream);
  }
  return rc == WC_OK ? py::cast(out) : py::none();
}

py::object wino_concat(py::handle a_, py::handle size_, py::handle m_) {
  const at::Tensor* const a = tile_tensor(a_);
  const auto m = tile_extent(m_);
  if (!a || !m) return py::none();
  const int nd = (int)a->dim() - 2;
  if (nd != 2 && nd != 3) return py::none();
  const auto size = whole_numbers(size_, nd);
  if (!size) return py::none();
  int64_t per = 1;
  for (int q = 0; q < nd; ++q) {
    if (a->size(2 + q) != *m) return py::none();
    per *= ((*size)[q] + *m - 1) / *m;
    if (per > a->size(0)) return py::none();           // no whole image; and the product of three extents may wrap around to 0
  }
  if (a->size(0) % per) return py::none();
  const int64_t B = a->size(0) / per, K = a->size(1);
  at::Tensor out;
  int rc;
  {
    py::gil_scoped_release nogil;
    const at::Tensor tiles = a->contiguous();
    std::vector<int64_t> shape{B}, order{0, nd + 1};
    for (int q = 0; q < nd; ++q) { shape.push_back((*size)[q]); order.push_back(1 + q); }
    shape.push_back(K);
    const at::Tensor last = at::empty(shape, a->options());
    const int es = (int)a->element_size();
    void* const stream = stream_of(*a);
    rc = nd == 2 ? wc_wino_concat2d(tiles.data_ptr(), last.data_ptr(), (int)B, (int)shape[1], (int)shape[2], (int)K, *m, es, stream)
                 : wc_wino_concat3d(tiles.data_ptr(), last.data_ptr(), (int)B, (int)shape[1], (int)shape[2], (int)shape[3], (int)K, *m, es, stream);
    out = last.permute(order);
  }
  return rc == WC_OK ? py::cast(out) : py::none();
}

// ---- a module's forward pass ----------------------------------------------------------------------------------------
// What WinoConv.py's modules work out anew for an input of another shape: the descriptor, the shape of the result and the
// transformed filter.  Called with an input of the same shape, strides and type and a weight of the same kind, it runs the layer
// without Python, with an autograd node of C++ where a gradient is wanted, and gives a plan with the filter where that has to be
// made; called with anything else it gives None, and the module goes its way.  It never changes after it is made, so
// threads and streams may share it; tensors are compared by what they are, and none but the transformed filter is kept.
// Host time, us, every call by itself | planned: a frozen layer 10.8 | 6.6 (a launch of torch's own 4.8), on two batch sizes in turn 11.1 | 9.9 (a plan
// is made for each, and its filter kept), on a first input 30 | 29; a training step in mixed precision 182 | 122, its backward pass 102 | 69, of
// which 55 are the autograd engine and a thread's waking.
class LayerPlan : public std::enable_shared_from_this<LayerPlan> {
 public:
  at::ScalarType x_type, w_type;
  at::Device device;
  std::vector<int64_t> sizes, strides, w_sizes, y_sizes, y_strides;
  wc_conv_desc d{};
  size_t bytes = 0, u_elems = 0;
  int nd, stride, m;
  std::vector<int> pads;
  std::shared_ptr<KeptFilter> filter, last;         // null: no pass yet; then the one that the first pass's takes the place of

  // None where the layer copies its input first.  `kept`: the filter of the module's last pass, taken where it is this one's
  static std::shared_ptr<LayerPlan> make(const at::Tensor& x, const at::Tensor& weight, int stride, std::vector<int> pads, int m,
                                         const std::shared_ptr<KeptFilter>& kept) {
    const int nd = spatial_dims(x.sizes(), weight.sizes());
    if ((int)pads.size() != nd || x.numel() == 0 || x.size(1) != weight.size(1) || !plain(x) || !plain(weight) || misaligned(x)) return nullptr;
    const bool last = channel_last_memory(x);
    if (!last && !x.is_contiguous()) return nullptr;
    auto p = std::make_shared<LayerPlan>(x, weight, stride, std::move(pads), m);
    p->d = desc_of(x.sizes(), weight.sizes(), p->pads, stride, m, dtype_of(x));
    p->d.stacked = p->d.row = -1;
    check(wc_conv_auto(&p->d));
    p->d.x_layout = !last;
    check(wc_conv_u_elems(&p->d, &p->u_elems));
    if (kept && kept->suits(p->form(), x.scalar_type(), x.device())) p->filter = kept;
    else if (kept && kept->holds(weight)) (p->filter = std::make_shared<KeptFilter>(weight, p->form()))->follows(kept);      // known, its filter not made for this plan
    else p->last = kept;
    int out[3], grid[3];
    check(wc_conv_out_dims(&p->d, out, grid));
    check(wc_conv_workspace_bytes(&p->d, &p->bytes));
    const int64_t K = weight.size(0);
    p->y_sizes = {x.size(0), K};
    p->y_strides = {K * out[0] * out[1] * out[2], 1};
    for (int a = 3 - nd; a < 3; ++a) p->y_sizes.push_back(out[a]);
    if (nd == 3) p->y_strides.push_back(K * out[1] * out[2]);
    p->y_strides.push_back(K * out[2]);
    p->y_strides.push_back(K);
    return p;
  }
  LayerPlan(const at::Tensor& x, const at::Tensor& weight, int s, std::vector<int> p, int m_)
      : x_type(x.scalar_type()), w_type(weight.scalar_type()), device(x.device()), sizes(x.sizes().vec()), strides(x.strides().vec()),
        w_sizes(weight.sizes().vec()), nd((int)x.dim() - 2), stride(s), m(m_), pads(std::move(p)) {}

  PlanForm form() const { return {d.direct, d.stacked, d.m, d.row, (int64_t)u_elems}; }

  at::Tensor run(const at::Tensor& x, const at::Tensor& w, const at::Tensor& bias, const at::Tensor& u) const {
    at::Tensor y = at::empty_strided(y_sizes, y_strides, x.options());
    void* stream = stream_of(x);
    at::Tensor ws = workspace_for(x, bytes, stream);
    int64_t s[5];
    strides_of(w, s);
    check(wc_conv_forward(&d, x.data_ptr(), w.data_ptr(), s, u.defined() ? u.data_ptr() : nullptr, bias.defined() ? bias.data_ptr() : nullptr,
                          y.data_ptr(), ws.data_ptr(), bytes, stream));
    return y;
  }

  at::Tensor transform(const at::Tensor& w) const {
    wc_conv_desc f = d;
    f.x_layout = 0;
    at::Tensor u = at::empty({(int64_t)u_elems}, w.options());
    wc_plan plan{};
    if (!f.direct && !f.row) check(wc_plan_conv(&f, &plan));
    int64_t s[5];
    strides_of(w, s);
    check(wc_filter_transform(&f, &plan, w.data_ptr(), s, u.data_ptr(), stream_of(w)));
    return u;
  }

  // The result; where the weight is another one than in the last pass, outside of captures (result, the plan with its filter, the filter)
  py::object call(const at::Tensor& x, const at::Tensor& weight, const std::optional<at::Tensor>& bias) const;

 private:
  // whether the layer's kernel takes this weight, or a copy of it in x's type, as it is
  bool takes(const at::Tensor& weight) const {
    int yes = 0;
    if (d.row == 1) {
      int64_t s[5];
      strides_of(weight, s);
      check(wc_conv_takes_filter(&d, weight.data_ptr(), s, &yes));
    }
    return yes != 0;
  }
  static bool misaligned(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) != 0; }
  bool fits(const at::Tensor& x, const at::Tensor& weight, const std::optional<at::Tensor>& bias) const {
    return plain(x) && plain(weight) && (!bias || plain(*bias)) && x.scalar_type() == x_type && x.sizes() == at::IntArrayRef(sizes) &&
           x.strides() == at::IntArrayRef(strides) && x.device() == device && !misaligned(x) && weight.scalar_type() == w_type &&
           weight.sizes() == at::IntArrayRef(w_sizes) && weight.device() == device && !weight.is_inference() &&
           (!bias || (bias->dim() == 1 && bias->size(0) == w_sizes[0] && bias->device() == device)) && !torch::jit::tracer::isTracing();
  }
};

struct LayerOperands { std::shared_ptr<const LayerPlan> plan; at::Tensor w, bias, U; };       // w and bias in x's type

struct LayerFunction : torch::autograd::Function<LayerFunction> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& weight, const std::optional<at::Tensor>& bias,
                            const LayerOperands& o) {
    ctx->save_for_backward({x, o.w});
    std::vector<int64_t> conf{o.plan->stride, o.plan->m, (int64_t)weight.scalar_type(), bias ? (int64_t)bias->scalar_type() : -1, weight.requires_grad()};
    for (int p : o.plan->pads) conf.push_back(p);
    ctx->saved_data["conf"] = std::move(conf);
    return o.plan->run(x, o.w, o.bias, o.U);
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &x = saved[0], &w = saved[1], &dy = grads[0];
    const auto conf = ctx->saved_data["conf"].toIntVector();
    const bool has_bias = conf[3] >= 0;
    const int stride = (int)conf[0], m = (int)conf[1];
    const std::vector<int> pads(conf.begin() + 5, conf.end());
    const auto w_type = (at::ScalarType)conf[2], b_type = has_bias ? (at::ScalarType)conf[3] : w_type;
    const bool dx = ctx->needs_input_grad(0), db = has_bias && ctx->needs_input_grad(2);
    const bool dw = ctx->needs_input_grad(1) || (db && conf[4]);      // the sums of a bias gradient are taken beside the weight's
    try {
      Gradients g;
      if (!at::GradMode::is_enabled()) g = backward_all(x, w, dy, stride, pads, m, dx, dw, db, w_type, b_type);
      if ((dx && !g.dx.defined()) || (dw && !g.dw.defined()) || (db && !g.db.defined())) {
        py::gil_scoped_acquire gil;                // what is left to the functions of WinoConv.py
        const py::object rest = py::module_::import("pytorch_winoconv_amd.WinoConv").attr("gradients")(
            x, w, dy, stride, py::tuple(py::cast(pads)), m, dx && !g.dx.defined(), dw && !g.dw.defined(), db && !g.db.defined(),
            py::reinterpret_borrow<py::object>((PyObject*)torch::getTHPDtype(w_type)), py::reinterpret_borrow<py::object>((PyObject*)torch::getTHPDtype(b_type)));
        const py::tuple t = rest.cast<py::tuple>();
        if (!t[0].is_none()) g.dx = t[0].cast<at::Tensor>();
        if (!t[1].is_none()) g.dw = t[1].cast<at::Tensor>();
        if (!t[2].is_none()) g.db = t[2].cast<at::Tensor>();
      }
      return {g.dx, g.dw, g.db, at::Tensor()};
    } catch (py::error_already_set& e) {           // exceptions reach the caller of backward() as the Python ones they are
      py::gil_scoped_acquire gil;
      e.restore();
      raise();
    } catch (const Unsupported& e) {
      py::gil_scoped_acquire gil;
      PyErr_SetString(PyExc_NotImplementedError, e.what());
      raise();
    } catch (const std::invalid_argument& e) {
      py::gil_scoped_acquire gil;
      PyErr_SetString(PyExc_ValueError, e.what());
      raise();
    } catch (const py::builtin_exception& e) {
      py::gil_scoped_acquire gil;
      e.set_error();
      raise();
    }
  }

 private:
  [[noreturn]] static void raise() {
    python_error error;
    error.persist();
    throw error;
  }
};

py::object LayerPlan::call(const at::Tensor& x, const at::Tensor& weight, const std::optional<at::Tensor>& bias) const {
  if (!fits(x, weight, bias)) return py::none();
  at::Tensor y;
  std::shared_ptr<LayerPlan> renewed;               // this plan with the filter, or the knowledge, of a weight that has changed
  {
    py::gil_scoped_release nogil;
    const bool grad = at::GradMode::is_enabled() && (x.requires_grad() || weight.requires_grad() || (bias && bias->requires_grad()));
    // A graph of a pass that is trained is replayed with other weights: it makes its filter itself
    const bool trained = grad && weight.requires_grad(), captured = trained && capturing(stream_of(x)), known = filter && !captured && filter->holds(weight);
    LayerOperands o{shared_from_this(), weight, bias ? *bias : at::Tensor(), known ? filter->on_stream() : at::Tensor()};
    // After a pass with a gradient of its own a weight is likely another one: nothing to make where the kernel takes the filter as it is.  A frozen
    // weight stays, and one that a second pass finds as it was (gradients of several passes added up, passes whose gradients nobody asks for) may
    // stay: their filters are made and kept.  us of a pass, fp16, x needs a gradient: 512 -> 512, 7x7, the filter taken 18.1, kept 9.5, 256 -> 256, 14x14 10.9 | 8.7.
    const bool taken = trained && !known && takes(weight);
    const bool anew = !o.U.defined() && !taken;
    if (anew || (taken && !captured)) {
      renewed = std::make_shared<LayerPlan>(*this);
      renewed->filter = std::make_shared<KeptFilter>(weight, form());
      renewed->filter->follows(filter ? filter : last);
      renewed->last = nullptr;
    }
    const bool cast_w = (grad || anew || taken) && w_type != x_type, cast_b = bias && bias->scalar_type() != x_type;
    if (cast_w || cast_b) {
      at::AutoGradMode no_grad(false);
      if (cast_w && w_type == at::kFloat && weight.is_non_overlapping_and_dense() && weight.numel() > 0) {
        const bool both = cast_b && bias->scalar_type() == at::kFloat && bias->is_contiguous();
        o.w = at::empty_strided(weight.sizes(), weight.strides(), x.options());
        if (both) o.bias = at::empty_strided(bias->sizes(), bias->strides(), x.options());
        check(wc_cast_parameters(weight.data_ptr<float>(), o.w.data_ptr(), weight.numel(), both ? bias->data_ptr<float>() : nullptr,
                                 both ? o.bias.data_ptr() : nullptr, both ? bias->numel() : 0, dtype_of(x), stream_of(x)));
      } else if (cast_w) {
        o.w = weight.to(x_type);
      }
      if (cast_b && o.bias.scalar_type() != x_type) o.bias = bias->to(x_type);
    }
    if (o.bias.defined()) o.bias = o.bias.contiguous();
    if (anew) {
      o.U = transform(o.w);
      renewed->filter->made(o.U);
    }
    y = grad ? LayerFunction::apply(x, weight, bias, o) : run(x, o.w, o.bias, o.U);
  }
  if (renewed && !renewed->filter->captured()) return py::make_tuple(y, renewed, renewed->filter);
  return py::cast(y);
}

// The reference's native entry point (pybind/extern.hpp:7-9): VALID convolution.  The four scratch tensors
// of the reference signature (dwm.py:122-125) are accepted and ignored: the engine sizes its own workspace.
void DWM(at::Tensor Input, at::Tensor Weight, at::Tensor Output, int stride, py::object, py::object, py::object, py::object) {
  winograd_conv(Input, Weight, Output, std::nullopt, stride, py::int_(0), 2, "dwm", std::nullopt, 0, py::none());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "MI355X-native stand-in for the reference extension MakePytorchBackend (pybind/bind.cpp:10-24)";
  static py::exception<WinoconvError> winoconv_error(m, "WinoconvError", PyExc_RuntimeError);
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const Unsupported& e) {
      PyErr_SetString(PyExc_NotImplementedError, e.what());
    }
  });
  py::class_<Foo>(m, "Foo")
      .def(py::init<>())
      .def("setKey", &Foo::setKey)
      .def("getKey", &Foo::getKey)
      .def("__repr__", [](const Foo& a) { return a.toString(); });
  m.def("AddGPU", &AddGPU);
  m.def("WinoSplit", &WinoSplit);
  m.def("WinoConcat", &WinoConcat);
  m.def("wino_split", &wino_split, py::arg("a"), py::arg("w_shape"), py::arg("output_block_size"));
  m.def("wino_concat", &wino_concat, py::arg("a"), py::arg("output_size"), py::arg("output_block_size"));
  m.def("DWM", &DWM, py::arg("Input"), py::arg("Weight"), py::arg("Output"), py::arg("stride"),
        py::arg("tmp_input_buffer") = py::none(), py::arg("tmp_weight_buffer") = py::none(),
        py::arg("tmp_product_buffer") = py::none(), py::arg("tmp_ptr_buffer") = py::none());
  m.def("winograd_conv", &winograd_conv, py::arg("Input"), py::arg("Weight"), py::arg("Output"),
        py::arg("bias") = py::none(), py::arg("stride") = 1, py::arg("padding") = 0, py::arg("m") = 2,
        py::arg("algo") = "dwm", py::arg("U") = py::none(), py::arg("chunk_images") = 0, py::arg("stacked") = py::none());
  m.def("split_and_concat", &split_and_concat);
  m.def("conv_forward", &conv_forward, py::arg("x"), py::arg("w"), py::arg("bias") = py::none(), py::arg("stride") = 1,
        py::arg("padding") = 0, py::arg("m") = 2, py::arg("U") = py::none(), py::arg("chunk_images") = 0,
        py::arg("whole_kernel") = false, py::arg("stacked") = py::none(), py::arg("unfused") = false,
        py::arg("channels_first_out") = false, py::arg("direct") = py::none(), py::arg("row") = false);
  m.def("conv_backward_weight", &conv_backward_weight, py::arg("x"), py::arg("dy"), py::arg("w_shape"), py::arg("stride") = 1,
        py::arg("padding") = 0, py::arg("m") = 2);
  py::class_<KeptFilter, std::shared_ptr<KeptFilter>>(m, "KeptFilter")
      .def(py::init<const at::Tensor&, const PlanForm&>(), py::arg("weight"), py::arg("form"))
      .def("made", &KeptFilter::made, py::arg("U"))
      .def("follows", &KeptFilter::follows, py::arg("last"))
      .def_property_readonly("captured", &KeptFilter::captured)
      .def("holds", &KeptFilter::holds, py::arg("weight"))
      .def("on_stream", [](const KeptFilter& f) { return or_none(f.on_stream()); });
  py::class_<LayerPlan, std::shared_ptr<LayerPlan>>(m, "LayerPlan")
      .def_static("make", &LayerPlan::make, py::arg("x"), py::arg("weight"), py::arg("stride"), py::arg("padding"), py::arg("m"), py::arg("kept"))
      .def_property_readonly("form", &LayerPlan::form)
      .def("__call__", &LayerPlan::call, py::arg("x"), py::arg("weight"), py::arg("bias"));
  m.def("conv_backward_parameters", &conv_backward_parameters, py::arg("x"), py::arg("dy"), py::arg("w_shape"), py::arg("stride"), py::arg("padding"),
        py::arg("m"), py::arg("need_db"), py::arg("w_type"), py::arg("b_type"));
  m.def("conv_backward", &conv_backward, py::arg("x"), py::arg("w"), py::arg("dy"), py::arg("stride"), py::arg("padding"), py::arg("m"),
        py::arg("need_dx"), py::arg("need_dw"), py::arg("need_db"), py::arg("w_type") = py::none(), py::arg("b_type") = py::none());
  m.def("conv_backward_input_flipped", &conv_backward_input_flipped, py::arg("dy"), py::arg("w"), py::arg("padding"), py::arg("m"));
  m.def("conv_backward_input_strided", &conv_backward_input_strided, py::arg("dy"), py::arg("w"), py::arg("x_spatial"), py::arg("pads"));
  m.def("transform_filter", &transform_filter, py::arg("w"), py::arg("x_shape"), py::arg("stride") = 1, py::arg("padding") = 0, py::arg("m") = 2);
  m.def("bias_gradient", &bias_gradient, py::arg("dy"));
  m.def("version", []() { return std::string(wc_version()); });
}
