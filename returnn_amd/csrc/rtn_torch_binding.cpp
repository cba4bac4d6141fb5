// The calls of the package's torch path in native code: argument checks, output and workspace allocation and the call of
// the library's C ABI, on torch tensors.  As Python these took longer than the device on short calls: one step of a layer took
// 123 us per call with five launches of 38 us together, and takes 16.3 with one launch of 8.9, of which host time is what is left.
//
// The library's entry points come in as addresses (init), so that the Python side decides which library is loaded.
#include <torch/extension.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/rtn_native_lstm2.h"

namespace py = pybind11;
using at::Tensor;

namespace {

struct Abi {
  decltype(&rtn_last_error) last_error;
  decltype(&rtn_set_abort_word) set_abort_word;
  decltype(&rtn_native_lstm2_fwd) fwd;
  decltype(&rtn_native_lstm2_fwd_workspace_bytes) fwd_workspace_bytes;
  decltype(&rtn_native_lstm2_fwd_multi) fwd_multi;
  decltype(&rtn_native_lstm2_fwd_multi_workspace_bytes) fwd_multi_workspace_bytes;
  decltype(&rtn_native_lstm2_last_output) last_output;
  decltype(&rtn_native_lstm2_bwd_multi) bwd_multi;
  decltype(&rtn_native_lstm2_bwd_multi_workspace_bytes) bwd_multi_workspace_bytes;
  decltype(&rtn_lstm_step) lstm_step;
  decltype(&rtn_sequence_mask) sequence_mask;
  decltype(&rtn_column_sums) column_sums;
  decltype(&rtn_column_sums_workspace_bytes) column_sums_workspace_bytes;
  decltype(&rtn_transposed_product) transposed_product;
  decltype(&rtn_transposed_product_workspace_bytes) transposed_product_workspace_bytes;
} rtn_abi;
bool ready = false;

void check_rc(int rc) {
  if (rc == RTN_OK) return;
  const char* text = rtn_abi.last_error();
  TORCH_CHECK(false, (text && *text) ? std::string(text) : "NativeLstm2: error code " + std::to_string(rc));
}

hipStream_t current_stream(const at::Device& device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

bool is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return stream && hipStreamIsCapturing(stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// ---- calls whose bounded waits expired ---------------------------------------------------------------------------
// A kernel whose wait for another workgroup runs into its bound writes the number of its call into ONE word of pinned
// host memory (and NaN marks into its results); the next call, or poll(), finds it there.  Nothing is copied, recorded
// or waited for on the way (a copy of the status word and an event per call cost 3.6 us of device and 9 us of host time).
struct Watch {
  std::mutex mu;
  volatile uint32_t* word = nullptr;
  uint32_t next_id = 0;
  struct Call {
    const char* what = "";
    int count = 1;
  } calls[4096];  // the latest calls by number
  unsigned long long issued = 0, checked = 0;
  std::atomic<unsigned> devices{0};  // with calls that drain() has not waited for
  std::atomic<int> synchronous{-1};  // -1: from the environment, read at each call
  py::object exception;

  // 0: off, 1: every call waits for its kernels and is looked at at once, 2: looked at later
  int setting() const {
    const int s = synchronous.load(std::memory_order_relaxed);
    if (s >= 0) return s ? 1 : 2;
    const char* v = getenv("RTN_LSTM2_CHECK_STATUS");
    return !v ? 2 : (strcmp(v, "0") == 0 ? 0 : (strcmp(v, "1") == 0 ? 1 : 2));
  }

  void poll() {
    const volatile uint32_t* w = word;
    if (w && *w) raise();
  }

  void raise() {
    std::string what;
    {
      std::lock_guard<std::mutex> lock(mu);
      const uint32_t id = *word;
      if (!id) return;
      *word = 0;
      const Call& c = calls[id % 4096];
      what = c.what;
      if (c.count > 1) what += " (" + std::to_string(c.count) + " calls)";
    }
    what += ": a bounded wait in the persistent kernel expired (device shared, preempted or paused?); the results of that call "
            "are invalid.  RTN_LSTM2_TIMEOUT_TICKS sets the bound in 10 ns ticks.";
    py::gil_scoped_acquire gil;
    PyErr_SetString(exception.ptr(), what.c_str());
    throw py::error_already_set();
  }

  // In front of a call of the library by this thread; false under capture (a recorded call would be replayed with nobody
  // looking at the word: captured calls rely on the NaN marks) and where the watch is off.
  bool before(const char* what, int count, bool capturing) {
    if (capturing) return false;
    poll();
    if (setting() == 0) return false;
    uint32_t id;
    {
      std::lock_guard<std::mutex> lock(mu);
      if (!word) {
        void* p = nullptr;
        TORCH_CHECK(hipHostMalloc(&p, 256, hipHostMallocPortable | hipHostMallocMapped) == hipSuccess, "NativeLstm2: no pinned host memory");
        memset(p, 0, 256);
        word = (volatile uint32_t*)p;  // (for the life of the process)
      }
      if (++next_id == 0) next_id = 1;
      id = next_id;
      calls[id % 4096].what = what;
      calls[id % 4096].count = count;
      ++issued;
    }
    rtn_abi.set_abort_word((void*)word, id);
    return true;
  }

  void after(const at::Device& device, hipStream_t stream) {
    devices.fetch_or(1u << (device.index() & 31), std::memory_order_relaxed);
    if (setting() == 1) {
      TORCH_CHECK(hipStreamSynchronize(stream) == hipSuccess, "NativeLstm2: the stream ended with an error");
      {
        std::lock_guard<std::mutex> lock(mu);
        checked = issued;
      }
      poll();
    }
  }

  void drain() {
    unsigned long long upto;
    {
      std::lock_guard<std::mutex> lock(mu);
      upto = issued;
    }
    const unsigned seen = devices.exchange(0);
    {
      py::gil_scoped_release no_gil;
      for (int d = 0; d < 32; ++d)
        if (seen >> d & 1u) {
          c10::DeviceGuard guard(at::Device(at::kCUDA, (c10::DeviceIndex)d));
          (void)hipDeviceSynchronize();
        }
    }
    {
      std::lock_guard<std::mutex> lock(mu);
      if (upto > checked) checked = upto;
    }
    poll();
  }
};
Watch& watch() {
  static Watch* w = new Watch();  // (never destroyed: threads may still call at exit)
  return *w;
}

// One call of the library under the watch; whatever happens, the thread's later calls do not report as this one.
struct Watched {
  bool on;
  Watched(const char* what, int count, hipStream_t stream) : on(watch().before(what, count, is_capturing(stream))) {}
  ~Watched() {
    if (on) rtn_abi.set_abort_word(nullptr, 0);
  }
  void done(const at::Device& device, hipStream_t stream) {
    if (on) watch().after(device, stream);
  }
};

// ---- autocast -----------------------------------------------------------------------------------------------------
// In an autocast region the layers' projection is a matrix product like torch's own: its operands take the region's type, by
// casts that autograd sees (the errors come back in the operands' types, and no copy without a way back to its parameter
// lands in the region's cache), and the recurrence runs in the type that the result has for the op (bfloat16, else float32).
// Behind these casts autocast is off: the products below autograd, forward and gradient, choose their types themselves.
std::optional<at::ScalarType> autocast_type() {
  if (!at::autocast::is_autocast_enabled(at::kCUDA)) return std::nullopt;
  return at::autocast::get_autocast_dtype(at::kCUDA);
}

struct NoAutocast {
  c10::impl::ExcludeDispatchKeyGuard guard{c10::autocast_dispatch_keyset};
};

// ---- arguments ----------------------------------------------------------------------------------------------------
Tensor as_type(const Tensor& t, at::ScalarType type) { return t.scalar_type() == type ? t : t.to(type); }
Tensor packed(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }

void check_ndim(const Tensor& t, const char* name, int64_t ndim) {
  TORCH_CHECK(t.dim() == ndim, name, " shape ndim is not ", ndim, ", got shape ", t.sizes());
}

// Row pitch in elements if t [T,B,width] can be handed to the library as it is: unit stride along the last axis, rows of
// consecutive (frame, sequence) pairs a constant number of elements apart, 16-byte aligned rows; 0 if not.
int64_t row_pitch(const Tensor& t) {
  if (t.dim() != 3) return 0;
  const int64_t T = t.size(0), B = t.size(1), width = t.size(2);
  if (T * B * width == 0) return t.is_contiguous() ? width : 0;
  const int64_t ld = B > 1 ? t.stride(1) : (T > 1 ? t.stride(0) : width);
  bool ok = (width == 1 || t.stride(2) == 1) && ld >= width && (B == 1 || t.stride(1) == ld) && (T == 1 || t.stride(0) == B * ld);
  ok = ok && (ld * t.element_size()) % 16 == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0;
  return ok ? ld : 0;
}

struct FwdArgs {
  Tensor X, W, y0, c0, i;
  int64_t T, B, n;
  bool bf16;
  int64_t ldX;  // 0: contiguous
  at::ScalarType act() const { return bf16 ? at::kBFloat16 : at::kFloat; }
  int dtype() const { return bf16 ? RTN_DTYPE_BF16 : RTN_DTYPE_F32; }
};

// Argument handling of the generated wrapper (returnn/torch/util/native_op.py:144-193) plus the op's shape asserts
// (returnn/native_op.py:1215-1223) as hard errors.
FwdArgs fwd_args(const Tensor& X, const Tensor& W, const Tensor& y0, const Tensor& c0, const Tensor& i, bool pitched_x) {
  check_ndim(X, "X", 3);
  check_ndim(W, "W", 2);
  check_ndim(y0, "y0", 2);
  check_ndim(c0, "c0", 2);
  check_ndim(i, "i", 2);
  const std::pair<const char*, const Tensor*> others[] = {{"W", &W}, {"y0", &y0}, {"c0", &c0}, {"i", &i}};
  for (const auto& o : others) TORCH_CHECK(o.second->device() == X.device(), o.first, " is on ", o.second->device(), " but X is on ", X.device());
  FwdArgs a;
  a.bf16 = X.scalar_type() == at::kBFloat16;
  a.X = as_type(X, a.act());
  a.W = packed(as_type(W, a.act()));
  a.y0 = packed(as_type(y0, a.act()));
  a.c0 = packed(as_type(c0, at::kFloat));
  a.i = packed(as_type(i, at::kFloat));
  a.ldX = pitched_x && !a.X.is_contiguous() ? row_pitch(a.X) : 0;
  if (!a.ldX) a.X = packed(a.X);
  a.T = a.i.size(0);
  a.B = a.i.size(1);
  a.n = a.y0.size(1);
  auto expect = [&](const char* name, const Tensor& t, at::IntArrayRef shape) {
    TORCH_CHECK(t.sizes() == shape, "NativeLstm2: ", name, " has shape ", t.sizes(), ", expected ", shape, " (T=", a.T, ", B=", a.B, " from i; n=", a.n, " from y0)");
  };
  expect("X", a.X, {a.T, a.B, 4 * a.n});
  expect("W", a.W, {a.n, 4 * a.n});
  expect("y0", a.y0, {a.B, a.n});
  expect("c0", a.c0, {a.B, a.n});
  return a;
}

Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({(int64_t)(bytes < 256 ? 256 : bytes)}, like.options().dtype(at::kByte));
}

typedef std::tuple<Tensor, Tensor, Tensor, Tensor> Out4;

Out4 fwd_outputs(const FwdArgs& a) {
  const auto act = a.X.options().dtype(a.act()), f32 = a.X.options().dtype(at::kFloat);
  return Out4(at::empty({a.T, a.B, a.n}, act), at::empty({a.T, a.B, a.n}, f32), at::empty({a.T, a.B, 4 * a.n}, act), at::empty({a.B, a.n}, f32));
}

// The forward op on HIP tensors.  (The workspace goes back to the caching allocator at the end; the allocator keeps it out
// of other streams' hands until the work queued on this stream has passed it.)
Out4 lstm2_forward(const Tensor& X, const Tensor& W, const Tensor& y0, const Tensor& c0, const Tensor& i, int64_t start, int64_t step, int mode) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  const FwdArgs a = fwd_args(X, W, y0, c0, i, false);
  c10::DeviceGuard guard(a.X.device());
  const hipStream_t stream = current_stream(a.X.device());
  Watched watched("NativeLstm2", 1, stream);
  Out4 out = fwd_outputs(a);
  const Tensor ws = workspace(rtn_abi.fwd_workspace_bytes(a.T, (int)a.B, (int)a.n, a.dtype(), mode), a.X);
  check_rc(rtn_abi.fwd(a.X.data_ptr(), a.W.data_ptr(), a.y0.data_ptr(), a.c0.data_ptr<float>(), a.i.data_ptr<float>(), (int)start, (int)step,
                   std::get<0>(out).data_ptr(), std::get<1>(out).data_ptr<float>(), std::get<2>(out).data_ptr(), std::get<3>(out).data_ptr<float>(), a.T,
                   (int)a.B, (int)a.n, a.dtype(), mode, ws.data_ptr(), (size_t)ws.numel(), stream));
  watched.done(a.X.device(), stream);
  return out;
}

template <int MODE>
Out4 lstm2_op(const Tensor& X, const Tensor& W, const Tensor& y0, const Tensor& c0, const Tensor& i, int64_t start, int64_t step) {
  return lstm2_forward(X, W, y0, c0, i, start, step, MODE);
}

typedef std::vector<std::pair<int64_t, int64_t>> Frames;  // (start, step) of each call

// Several calls of one shape through rtn_native_lstm2_fwd_multi; `joint`: their Y side by side in one [T,B,count*n] array;
// `last`: takes the final output [B,n] of each call.
std::pair<std::vector<Out4>, Tensor> lstm2_multi(const std::vector<FwdArgs>& args, const Frames& frames, int mode, bool joint, std::vector<Tensor>* last = nullptr) {
  const FwdArgs& f = args[0];
  for (const FwdArgs& a : args) {
    TORCH_CHECK(a.T == f.T && a.B == f.B && a.n == f.n && a.bf16 == f.bf16, "native_lstm2_multi: all calls need the same T, B, n and element type; got (", f.T, ", ", f.B,
                ", ", f.n, ", ", f.bf16, ") and (", a.T, ", ", a.B, ", ", a.n, ", ", a.bf16, ")");
    TORCH_CHECK(a.X.device() == f.X.device(), "native_lstm2_multi: all calls must be on one device");
  }
  TORCH_CHECK(f.X.is_cuda(), "NativeLstm2: this build implements the op for HIP (MI355X) tensors only; got CPU tensors.");
  const int count = (int)args.size();
  c10::DeviceGuard guard(f.X.device());
  const hipStream_t stream = current_stream(f.X.device());
  Watched watched("NativeLstm2", count, stream);
  Tensor Yj;
  const int64_t es = f.bf16 ? 2 : 4;
  const auto act = f.X.options().dtype(f.act()), f32 = f.X.options().dtype(at::kFloat);
  // (columns of the calls that would not be 16-byte aligned: separate arrays, joined below)
  if (joint && (f.n * es) % 16 == 0) Yj = at::empty({f.T, f.B, count * f.n}, act);
  std::vector<Out4> outs;
  std::vector<rtn_lstm2_call> calls(count);
  for (int k = 0; k < count; ++k) {
    const FwdArgs& a = args[k];
    Tensor Y = Yj.defined() ? Yj.slice(2, k * f.n, (k + 1) * f.n) : at::empty({f.T, f.B, f.n}, act);
    outs.emplace_back(Y, at::empty({f.T, f.B, f.n}, f32), at::empty({f.T, f.B, 4 * f.n}, act), at::empty({f.B, f.n}, f32));
    const Out4& o = outs.back();
    calls[k] = {a.X.data_ptr(), a.W.data_ptr(), a.y0.data_ptr(), a.c0.data_ptr<float>(), a.i.data_ptr<float>(), (int)frames[k].first, (int)frames[k].second,
                Y.data_ptr(), std::get<1>(o).data_ptr<float>(), std::get<2>(o).data_ptr(), std::get<3>(o).data_ptr<float>(), a.ldX, Yj.defined() ? count * f.n : 0, nullptr};
    if (last) {
      last->push_back(at::empty({f.B, f.n}, act));
      calls[k].hN = last->back().data_ptr();
    }
  }
  const Tensor ws = workspace(rtn_abi.fwd_multi_workspace_bytes(count, f.T, (int)f.B, (int)f.n, f.dtype(), mode), f.X);
  check_rc(rtn_abi.fwd_multi(calls.data(), count, f.T, (int)f.B, (int)f.n, f.dtype(), mode, ws.data_ptr(), (size_t)ws.numel(), stream));
  watched.done(f.X.device(), stream);
  if (joint && !Yj.defined()) {
    std::vector<Tensor> ys;
    for (const Out4& o : outs) ys.push_back(std::get<0>(o));
    Yj = count == 1 ? ys[0] : at::cat(ys, -1);  // (one array joined with nothing is a copy of all of it: n = 604, T B = 69 696, bf16 29 us)
  }
  return {outs, Yj};
}

py::object py_lstm2_multi(const py::sequence& calls, int mode, bool joint) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  std::vector<FwdArgs> args;
  Frames frames;
  for (const py::handle& h : calls) {
    const py::tuple c = py::reinterpret_borrow<py::object>(h);
    args.push_back(fwd_args(c[0].cast<Tensor>(), c[1].cast<Tensor>(), c[2].cast<Tensor>(), c[3].cast<Tensor>(), c[4].cast<Tensor>(), true));
    frames.emplace_back(c[5].cast<int64_t>(), c[6].cast<int64_t>());
  }
  auto res = lstm2_multi(args, frames, mode, joint);
  py::list outs;
  for (Out4& o : res.first) outs.append(py::cast(o));
  if (!joint) return std::move(outs);
  return py::make_tuple(outs, res.second);
}

// Final output per sequence (returnn/tf/native_op.py:913-929).
Tensor last_output(const Tensor& Y_in, const Tensor& y0_in, const Tensor& i_in, int64_t start, int64_t step) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  TORCH_CHECK(Y_in.is_cuda(), "lstm_last_output: this build implements the op for HIP (MI355X) tensors only");
  const bool bf16 = Y_in.scalar_type() == at::kBFloat16;
  const at::ScalarType act = bf16 ? at::kBFloat16 : at::kFloat;
  Tensor Y = as_type(Y_in, act);
  int64_t ldY = row_pitch(Y);
  if (!ldY) {
    Y = packed(Y);
    ldY = Y.size(2);
  }
  const Tensor y0 = packed(as_type(y0_in, act)), i = packed(as_type(i_in, at::kFloat));
  const int64_t T = Y.size(0), B = Y.size(1), n = Y.size(2);
  TORCH_CHECK(y0.sizes() == at::IntArrayRef({B, n}) && i.sizes() == at::IntArrayRef({T, B}), "lstm_last_output: y0 ", y0.sizes(), " / i ", i.sizes(), " do not match Y ", Y.sizes());
  c10::DeviceGuard guard(Y.device());
  Tensor out = at::empty({B, n}, Y.options());
  check_rc(rtn_abi.last_output(Y.data_ptr(), y0.data_ptr(), i.data_ptr<float>(), (int)start, (int)step, out.data_ptr(), T, (int)B, (int)n, bf16 ? RTN_DTYPE_BF16 : RTN_DTYPE_F32,
                           ldY, current_stream(Y.device())));
  return out;
}

// ---- the gradient op ----------------------------------------------------------------------------------------------
struct BwdArgs {
  Tensor W, y0, c0, i, Y, C, H, DY, Dd;     // (Dd undefined: zero)
  int64_t start, step, T, B, n, ldY, ldDY;  // (pitches: 0 = contiguous)
  bool bf16;
};

BwdArgs bwd_args(const Tensor& W, const Tensor& y0, const Tensor& c0, const Tensor& i, int64_t start, int64_t step, const Tensor& Y, const Tensor& C, const Tensor& H,
                 const Tensor& DY, const Tensor& Dd) {
  TORCH_CHECK(Y.is_cuda(), "NativeLstm2 gradient: this build implements the op for HIP (MI355X) tensors only; got CPU tensors.");
  BwdArgs a;
  a.bf16 = Y.scalar_type() == at::kBFloat16;
  const at::ScalarType act = a.bf16 ? at::kBFloat16 : at::kFloat;
  a.W = packed(as_type(W, act));
  a.y0 = packed(as_type(y0, act));
  a.H = packed(as_type(H, act));
  // (Y and DY may be views with a row pitch, e.g. one direction's half of a [T,B,2n] array: handed over as they are)
  a.Y = as_type(Y, act);
  a.DY = as_type(DY, act);
  a.ldY = a.Y.is_contiguous() ? 0 : row_pitch(a.Y);
  a.ldDY = a.DY.is_contiguous() ? 0 : row_pitch(a.DY);
  if (!a.ldY) a.Y = packed(a.Y);
  if (!a.ldDY) a.DY = packed(a.DY);
  a.c0 = packed(as_type(c0, at::kFloat));
  a.i = packed(as_type(i, at::kFloat));
  a.C = packed(as_type(C, at::kFloat));
  if (Dd.defined()) a.Dd = packed(as_type(Dd, at::kFloat));
  a.start = start;
  a.step = step;
  TORCH_CHECK(a.i.dim() == 2 && a.y0.dim() == 2, "NativeLstm2 gradient: i ", a.i.sizes(), " / y0 ", a.y0.sizes());
  a.T = a.i.size(0);
  a.B = a.i.size(1);
  a.n = a.y0.size(1);
  auto expect = [&](const char* name, const Tensor& t, at::IntArrayRef shape) {
    TORCH_CHECK(t.sizes() == shape, "NativeLstm2 gradient: ", name, " has shape ", t.sizes(), ", expected ", shape);
    TORCH_CHECK(t.device() == a.Y.device(), "NativeLstm2 gradient: ", name, " is on ", t.device(), " but Y is on ", a.Y.device());
  };
  expect("W", a.W, {a.n, 4 * a.n});
  expect("y0", a.y0, {a.B, a.n});
  expect("c0", a.c0, {a.B, a.n});
  expect("Y", a.Y, {a.T, a.B, a.n});
  expect("C", a.C, {a.T, a.B, a.n});
  expect("H", a.H, {a.T, a.B, 4 * a.n});
  expect("DY", a.DY, {a.T, a.B, a.n});
  if (a.Dd.defined()) expect("Dd", a.Dd, {a.B, a.n});
  return a;
}

// (DX, DW, Dy0, Dc0) per call; `joint`: their DX side by side in one [T,B,count*4n] array; `own_type`: DW in the op's type.
std::pair<std::vector<Out4>, Tensor> lstm2_grad_multi(const std::vector<BwdArgs>& args, bool joint, bool own_type = false) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  const BwdArgs& f = args[0];
  for (const BwdArgs& a : args)
    TORCH_CHECK(a.T == f.T && a.B == f.B && a.n == f.n && a.bf16 == f.bf16 && a.Y.device() == f.Y.device(),
                "native_lstm2_grad_multi: all calls must have one shape, dtype and device");
  const int count = (int)args.size();
  const int dtype = f.bf16 ? RTN_DTYPE_BF16 : RTN_DTYPE_F32;
  c10::DeviceGuard guard(f.Y.device());
  const hipStream_t stream = current_stream(f.Y.device());
  Watched watched("NativeLstm2 gradient", count, stream);
  const auto act = f.Y.options(), f32 = f.Y.options().dtype(at::kFloat);
  Tensor DXj;
  if (joint && (4 * f.n * f.Y.element_size()) % 16 == 0) DXj = at::empty({f.T, f.B, count * 4 * f.n}, act);  // (else: separate arrays, joined below)
  std::vector<Out4> outs;
  std::vector<Tensor> sums;  // (DW on its way)
  std::vector<rtn_lstm2_bwd_call> calls(count);
  for (int k = 0; k < count; ++k) {
    const BwdArgs& a = args[k];
    Tensor DX = DXj.defined() ? DXj.slice(2, k * 4 * f.n, (k + 1) * 4 * f.n) : at::empty({f.T, f.B, 4 * f.n}, act);
    outs.emplace_back(DX, at::empty({f.n, 4 * f.n}, f32), at::empty({f.B, f.n}, act), at::empty({f.B, f.n}, f32));
    Out4& o = outs.back();
    void* DW_act = nullptr;
    const Tensor DW = std::get<1>(o);
    if (own_type && f.bf16) {
      sums.push_back(DW);
      std::get<1>(o) = at::empty({f.n, 4 * f.n}, act);
      DW_act = std::get<1>(o).data_ptr();
    }
    calls[k] = {a.W.data_ptr(), a.y0.data_ptr(), a.c0.data_ptr<float>(), a.i.data_ptr<float>(), (int)a.start, (int)a.step, a.Y.data_ptr(), a.C.data_ptr<float>(),
                a.H.data_ptr(), a.DY.data_ptr(), a.Dd.defined() ? a.Dd.data_ptr<float>() : nullptr, DX.data_ptr(), DW.data_ptr<float>(), std::get<2>(o).data_ptr(),
                std::get<3>(o).data_ptr<float>(), a.ldY, a.ldDY, DXj.defined() ? count * 4 * f.n : 0, DW_act, a.Dd.defined() ? 0 : 1};
  }
  const Tensor ws = workspace(rtn_abi.bwd_multi_workspace_bytes(count, f.T, (int)f.B, (int)f.n, dtype), f.Y);
  check_rc(rtn_abi.bwd_multi(calls.data(), count, f.T, (int)f.B, (int)f.n, dtype, ws.data_ptr(), (size_t)ws.numel(), stream));
  watched.done(f.Y.device(), stream);
  if (joint && !DXj.defined()) {
    std::vector<Tensor> dx;
    for (const Out4& o : outs) dx.push_back(std::get<0>(o));
    DXj = count == 1 ? dx[0] : at::cat(dx, -1);
  }
  return {outs, DXj};
}

py::object py_lstm2_grad_multi(const py::sequence& calls, bool joint) {
  std::vector<BwdArgs> args;
  for (const py::handle& h : calls) {
    const py::tuple c = py::reinterpret_borrow<py::object>(h);
    auto t = [&](int k) { return c[k].cast<Tensor>(); };
    args.push_back(bwd_args(t(0), t(1), t(2), t(3), c[4].cast<int64_t>(), c[5].cast<int64_t>(), t(6), t(7), t(8), t(9), t(10)));
  }
  auto res = lstm2_grad_multi(args, joint);
  py::list outs;
  for (Out4& o : res.first) outs.append(py::cast(o));
  if (!joint) return std::move(outs);
  return py::make_tuple(outs, res.second);
}

// ---- layers: projection and one or two directions -------------------------------------------------------------------
Tensor sequence_mask(const Tensor& lengths, int64_t T) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  TORCH_CHECK(lengths.dim() == 1 && lengths.is_cuda(), "sequence_mask: lengths ", lengths.sizes(), " on ", lengths.device());
  const Tensor l = packed(as_type(lengths, at::kLong));
  c10::DeviceGuard guard(l.device());
  Tensor mask = at::empty({T, l.size(0)}, l.options().dtype(at::kFloat));
  check_rc(rtn_abi.sequence_mask(l.data_ptr<int64_t>(), mask.data_ptr<float>(), T, (int)l.size(0), current_stream(l.device())));
  return mask;
}

// Sums over the rows of a contiguous [rows,width] matrix of one of the op's types, as `type` (one of them, too).  (Not torch's
// sum: over many rows that records a memset into a captured graph, whose replays then add to values of other replays.)
Tensor column_sums(const Tensor& m, at::ScalarType type) {
  const int64_t rows = m.size(0), width = m.size(1);
  Tensor out = at::empty({width}, m.options().dtype(type));
  if (m.numel() == 0) return out.zero_();
  auto code = [](at::ScalarType t) { return t == at::kBFloat16 ? RTN_DTYPE_BF16 : RTN_DTYPE_F32; };
  const Tensor ws = workspace(rtn_abi.column_sums_workspace_bytes(rows, (int)width), m);
  check_rc(rtn_abi.column_sums(m.data_ptr(), rows, (int)width, code(m.scalar_type()), out.data_ptr(), code(type), ws.data_ptr(), (size_t)ws.numel(), current_stream(m.device())));
  return out;
}

// a^T b of [rows,m] and [rows,n].  (With gradients of gradients on, the product that autograd knows.)
Tensor transposed_product(const Tensor& a, const Tensor& b) {
  const int64_t rows = a.size(0), m = a.size(1), n = b.size(1);
  const bool known = !at::GradMode::is_enabled() && (a.scalar_type() == at::kBFloat16 || a.scalar_type() == at::kFloat) && a.scalar_type() == b.scalar_type() && a.is_contiguous() && b.is_contiguous() &&
                     rows > 0 && m < (1 << 20) && n < (1 << 20) && (uintptr_t)a.data_ptr() % 16 == 0;
  const int dtype = a.scalar_type() == at::kBFloat16 ? RTN_DTYPE_BF16 : RTN_DTYPE_F32;
  const size_t bytes = known ? rtn_abi.transposed_product_workspace_bytes(rows, (int)m, (int)n, dtype) : 0;
  if (!bytes) return at::mm(a.t(), b);
  c10::DeviceGuard guard(a.device());
  const Tensor out = at::empty({m, n}, a.options()), ws = workspace(bytes, a);
  check_rc(rtn_abi.transposed_product(a.data_ptr(), m, b.data_ptr(), n, rows, (int)m, (int)n, dtype, out.data_ptr(), dtype, ws.data_ptr(), (size_t)ws.numel(),
                                      current_stream(a.device())));
  return out;
}

// One direction: (W [n,4n], y0 [B,n], c0 [B,n], step).
struct Direction {
  Tensor W, y0, c0;
  int64_t step;
};

// P = source . ff + bias, rows of D * 4n gates; then the recurrences on it, their outputs side by side.  (source, ff and bias
// of one type, which need not be one of the op's: the recurrences take P as the op takes its input.)
struct LayerRun {
  std::vector<Out4> outs;  // (Y view, C, H, d) per direction
  Tensor Y;                // [T,B,D*n]
  std::vector<Tensor> last;
};
LayerRun layer_forward(const Tensor& source, const Tensor& ff, const Tensor& bias, const std::vector<Direction>& dirs, const Tensor& mask, bool want_last) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  const int64_t T = source.size(0), B = source.size(1);
  const Tensor src2 = source.reshape({T * B, source.size(2)});
  const Tensor P = (bias.defined() ? at::addmm(bias, src2, ff) : at::mm(src2, ff)).view({T, B, ff.size(1)});
  std::vector<FwdArgs> args;
  Frames frames;
  const int64_t n4 = dirs[0].W.size(1);
  for (size_t k = 0; k < dirs.size(); ++k) {
    args.push_back(fwd_args(dirs.size() == 1 ? P : P.slice(2, k * n4, (k + 1) * n4), dirs[k].W, dirs[k].y0, dirs[k].c0, mask, true));
    frames.emplace_back(0, dirs[k].step);
  }
  LayerRun run;
  auto res = lstm2_multi(args, frames, RTN_MODE_AUTO, true, want_last ? &run.last : nullptr);
  run.outs = std::move(res.first);
  run.Y = res.second;
  return run;
}

// The one-step kernel reads all weights again for every 64 rows; a GEMM and the recurrent kernels take over where that is more
// traffic than they make up for with their launches.  Measured on MI355X (us per call, one-step kernel / GEMM and recurrent
// kernel): bf16 n = 1024 of 512 inputs, 12 to 2048 rows: 9 / 50 ... 148 / 156, 4096 rows (805 MB): 289 / 282; n = 2048 of 2048, 384
// rows (403 MB): 167 / 205, 512 (537 MB): 214 / 142; float32 n = 1024 of 512, 512 rows (201 MB): 118 / 171, 1024 (403 MB): 232 / 191;
// n = 2048 of 2048, 64 rows: 75 / 87, 128 (268 MB): 155 / 130.  Up to 64 rows it is ahead at every width measured (128 to 4096).
constexpr double kStepTrafficBf16 = 410e6, kStepTrafficF32 = 260e6;

// One step of a layer, projection included: (y, h, c) of x [B,in] and the state before (rtn_lstm_step, or a sequence of one frame).
std::tuple<Tensor, Tensor, Tensor> lstm_step(const Tensor& x_in, const Tensor& h_in, const Tensor& c_in, const Tensor& ff_in, const Tensor& rec_in,
                                             const std::optional<Tensor>& bias_in) {
  TORCH_CHECK(ready, "NativeLstm2: the library is not loaded");
  TORCH_CHECK(x_in.is_cuda(), "lstm: this build implements the LSTM for HIP (MI355X) tensors only; got a CPU tensor");
  TORCH_CHECK(x_in.dim() == 2 && rec_in.dim() == 2, "lstm: input ", x_in.sizes(), " / rec ", rec_in.sizes());
  const int64_t B = x_in.size(0), in = x_in.size(1), n = rec_in.size(0);
  TORCH_CHECK(rec_in.size(1) == 4 * n && ff_in.sizes() == at::IntArrayRef({4 * n, in}) && (!bias_in.has_value() || bias_in->sizes() == at::IntArrayRef({4 * n})),
              "lstm: parameters ", ff_in.sizes(), " / ", rec_in.sizes(), " do not match each other or the input ", x_in.sizes());
  TORCH_CHECK(h_in.sizes() == at::IntArrayRef({B, n}) && c_in.sizes() == at::IntArrayRef({B, n}), "lstm: state_h ", h_in.sizes(), " / state_c ", c_in.sizes(), ", expected ",
              at::IntArrayRef({B, n}));
  for (const Tensor* t : {&h_in, &c_in, &ff_in, &rec_in}) TORCH_CHECK(t->device() == x_in.device(), "lstm: a tensor is on ", t->device(), " but the input is on ", x_in.device());
  TORCH_CHECK(!bias_in.has_value() || bias_in->device() == x_in.device(), "lstm: the bias is on another device than the input");
  c10::DeviceGuard guard(x_in.device());
  // the type of the projection: the region's, else the op's
  const at::ScalarType type = autocast_type().value_or(x_in.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat);
  const NoAutocast no_autocast;
  const bool bf16 = type == at::kBFloat16;
  Tensor x = as_type(x_in, type), ff = as_type(ff_in, type), bias;
  if (bias_in.has_value()) bias = as_type(*bias_in, type);
  const int64_t shares = (B + 63) / 64;
  const double traffic = (double)shares * 4 * n * (in + n) * (bf16 ? 2 : 4);
  if ((!bf16 && type != at::kFloat) || (shares > 1 && traffic > (bf16 ? kStepTrafficBf16 : kStepTrafficF32))) {
    const Tensor mask = at::ones({1, B}, x.options().dtype(at::kFloat));
    const LayerRun run = layer_forward(x.unsqueeze(0), ff.t(), bias, {{rec_in, h_in, c_in, 1}}, mask, true);
    return {run.Y.select(0, 0), run.last[0], std::get<3>(run.outs[0])};
  }
  x = packed(x);
  ff = packed(ff);
  if (bias.defined()) bias = packed(bias);
  const Tensor h = packed(as_type(h_in, type)), c = packed(as_type(c_in, at::kFloat)), rec = packed(as_type(rec_in, type));
  Tensor y = at::empty({B, n}, x.options()), h_out = at::empty({B, n}, x.options()), c_out = at::empty({B, n}, c.options());
  check_rc(rtn_abi.lstm_step(x.data_ptr(), h.data_ptr(), c.data_ptr<float>(), ff.data_ptr(), rec.data_ptr(), bias.defined() ? bias.data_ptr() : nullptr, y.data_ptr(),
                         h_out.data_ptr(), c_out.data_ptr<float>(), (int)B, (int)in, (int)n, bf16 ? RTN_DTYPE_BF16 : RTN_DTYPE_F32, current_stream(x.device())));
  return {y, h_out, c_out};
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A layer with its gradient.  Inputs: source, ff, bias (or undefined), mask, then W, y0, c0 per direction; outputs: Y, then d
// per direction.  Gradients as autograd's of the projection and NativeLstm2Function's of the recurrences.
struct LayerFunction : torch::autograd::Function<LayerFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& source, const Tensor& ff, const std::optional<Tensor>& bias, const Tensor& mask, const Tensor& W0,
                               const Tensor& y00, const Tensor& c00, const std::optional<Tensor>& W1, const std::optional<Tensor>& y01, const std::optional<Tensor>& c01,
                               int64_t step0) {
    at::AutoDispatchBelowADInplaceOrView below;
    const NoAutocast no_autocast;
    std::vector<Direction> dirs{{W0, y00, c00, step0}};
    if (W1.has_value()) dirs.push_back({*W1, *y01, *c01, -step0});
    const LayerRun run = layer_forward(source, ff, bias.has_value() ? *bias : Tensor(), dirs, mask, false);
    variable_list saved{source, ff, mask, run.Y}, result{run.Y};
    for (size_t k = 0; k < dirs.size(); ++k) {
      for (const Tensor& t : {dirs[k].W, dirs[k].y0, dirs[k].c0, std::get<1>(run.outs[k]), std::get<2>(run.outs[k])}) saved.push_back(t);
      result.push_back(std::get<3>(run.outs[k]));
    }
    ctx->save_for_backward(saved);
    ctx->saved_data["step"] = step0;
    ctx->saved_data["bias"] = bias.has_value();
    ctx->set_materialize_grads(false);
    return result;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const NoAutocast no_autocast;
    const auto saved = ctx->get_saved_variables();
    const Tensor &source = saved[0], &ff = saved[1], &mask = saved[2], &Y = saved[3];
    const int64_t step0 = ctx->saved_data["step"].toInt();
    const int count = (int)(saved.size() - 4) / 5;
    const Tensor DY = grads[0].defined() ? grads[0] : at::zeros_like(Y);
    std::vector<BwdArgs> args;
    for (int k = 0; k < count; ++k) {
      const Tensor* s = &saved[4 + 5 * k];  // W, y0, c0, C, H
      const int64_t n = s[1].size(1);
      auto half = [&](const Tensor& t) { return count == 1 ? t : t.slice(2, k * n, (k + 1) * n); };
      args.push_back(bwd_args(s[0], s[1], s[2], mask, 0, k ? -step0 : step0, half(Y), s[3], s[4], half(DY), grads[1 + k]));
    }
    bool own_type = true;  // (the weights have the op's type)
    for (int k = 0; k < count; ++k) own_type = own_type && saved[4 + 5 * k].scalar_type() == Y.scalar_type();
    auto res = lstm2_grad_multi(args, true, own_type);
    const int64_t rows = source.size(0) * source.size(1);
    const Tensor DPo = res.second.view({rows, ff.size(1)}), DP = as_type(DPo, ff.scalar_type());  // (the error of a projection of another type than the op's)
    variable_list out(11);
    if (ctx->needs_input_grad(0)) out[0] = at::mm(DP, ff.t()).view(source.sizes());
    // (the gradient of ff comes out in the layout of a [4n,in] parameter, whose transposed view ff usually is)
    if (ctx->needs_input_grad(1)) out[1] = transposed_product(DP, source.reshape({rows, source.size(2)})).t();
    if (ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2)) {
      c10::DeviceGuard guard(DPo.device());
      out[2] = as_type(column_sums(DPo, ff.scalar_type() == DPo.scalar_type() ? DPo.scalar_type() : at::kFloat), ff.scalar_type());
    }
    for (int k = 0; k < count; ++k) {
      const Tensor* s = &saved[4 + 5 * k];
      const Out4& o = res.first[k];
      out[4 + 3 * k] = as_type(std::get<1>(o), s[0].scalar_type());
      out[5 + 3 * k] = as_type(std::get<2>(o), s[1].scalar_type());
      out[6 + 3 * k] = as_type(std::get<3>(o), s[2].scalar_type());
    }
    return out;
  }
};

// The final output per sequence with its gradient, for the right-padded masks that are made of lengths.
struct LastOutputFunction : torch::autograd::Function<LastOutputFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& Y, const Tensor& y0, const Tensor& mask, int64_t step) {
    at::AutoDispatchBelowADInplaceOrView below;
    ctx->save_for_backward({mask});
    ctx->saved_data["step"] = step;
    ctx->saved_data["y0_type"] = (int64_t)y0.scalar_type();
    return last_output(Y, y0, mask, 0, step);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor mask = ctx->get_saved_variables()[0], &g = grads[0];
    const int64_t step = ctx->saved_data["step"].toInt();
    if (!g.defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    // the frame that g belongs to, per sequence: the last one of the mask, or the first where there is one (no sum over the
    // frames: see column_sums)
    const Tensor valid = mask > 0, some = valid.select(0, 0).unsqueeze(1), none = at::zeros_like(valid.narrow(0, 0, 1));
    const int64_t T = valid.size(0);
    const Tensor at_frame = step > 0 ? valid.logical_and(at::cat({valid.narrow(0, 1, T - 1), none}).logical_not())
                                     : at::cat({valid.narrow(0, 0, 1), none.expand({T - 1, valid.size(1)})});
    const Tensor zero = at::zeros({}, g.options()), dY = at::where(at_frame.unsqueeze(2), g.unsqueeze(0), zero);
    return {dY, at::where(some, zero, g).to((at::ScalarType)ctx->saved_data["y0_type"].toInt()), Tensor(), Tensor()};
  }
};

// source [T,B,in], ff [in,D*4n], bias or None, mask [T,B]; W, y0, c0 per direction (the second runs against the first).
// Returns Y [T,B,D*n], the final outputs (want_last) and the final cell states.
py::tuple lstm_layer(Tensor source, Tensor ff, std::optional<Tensor> bias, const Tensor& mask, const std::vector<std::tuple<Tensor, Tensor, Tensor>>& directions,
                     int64_t step, bool want_last) {
  std::vector<Direction> dirs;
  for (const auto& d : directions) dirs.push_back({std::get<0>(d), std::get<1>(d), std::get<2>(d), dirs.empty() ? step : -step});
  TORCH_CHECK(source.dim() == 3 && ff.dim() == 2 && (dirs.size() == 1 || dirs.size() == 2), "lstm_layer: bad arguments");
  if (const auto region = autocast_type()) {
    source = as_type(source, *region);
    ff = as_type(ff, *region);
    if (bias.has_value()) bias = as_type(*bias, *region);
  }
  const NoAutocast no_autocast;
  bool grad = false;
  if (at::GradMode::is_enabled()) {
    grad = source.requires_grad() || ff.requires_grad() || (bias.has_value() && bias->requires_grad());
    for (const Direction& d : dirs) grad = grad || d.W.requires_grad() || d.y0.requires_grad() || d.c0.requires_grad();
  }
  Tensor Y;
  py::list last, cells;
  if (!grad) {
    LayerRun run = layer_forward(source, ff, bias.has_value() ? *bias : Tensor(), dirs, mask, want_last);
    Y = run.Y;
    for (const Tensor& t : run.last) last.append(t);
    for (const Out4& o : run.outs) cells.append(std::get<3>(o));
  } else {
    std::optional<Tensor> W1, y01, c01;
    if (dirs.size() == 2) W1 = dirs[1].W, y01 = dirs[1].y0, c01 = dirs[1].c0;
    const variable_list r = LayerFunction::apply(source, ff, bias, mask, dirs[0].W, dirs[0].y0, dirs[0].c0, W1, y01, c01, step);
    Y = r[0];
    const int64_t n = dirs[0].W.size(0);
    for (size_t k = 0; k < dirs.size(); ++k) {
      if (want_last)
        last.append(LastOutputFunction::apply(dirs.size() == 1 ? Y : Y.slice(2, k * n, (k + 1) * n), dirs[k].y0, mask, dirs[k].step));
      cells.append(r[1 + k]);
    }
  }
  return py::make_tuple(Y, last, cells);
}

template <typename F>
void take(F*& fn, const py::dict& symbols, const char* name) {
  fn = reinterpret_cast<F*>(symbols[name].cast<uintptr_t>());
}

// Addresses of the library's entry points and the exception of an expired wait.
void init(const py::dict& symbols, const py::object& aborted) {
  take(rtn_abi.last_error, symbols, "rtn_last_error");
  take(rtn_abi.set_abort_word, symbols, "rtn_set_abort_word");
  take(rtn_abi.fwd, symbols, "rtn_native_lstm2_fwd");
  take(rtn_abi.fwd_workspace_bytes, symbols, "rtn_native_lstm2_fwd_workspace_bytes");
  take(rtn_abi.fwd_multi, symbols, "rtn_native_lstm2_fwd_multi");
  take(rtn_abi.fwd_multi_workspace_bytes, symbols, "rtn_native_lstm2_fwd_multi_workspace_bytes");
  take(rtn_abi.last_output, symbols, "rtn_native_lstm2_last_output");
  take(rtn_abi.bwd_multi, symbols, "rtn_native_lstm2_bwd_multi");
  take(rtn_abi.bwd_multi_workspace_bytes, symbols, "rtn_native_lstm2_bwd_multi_workspace_bytes");
  take(rtn_abi.lstm_step, symbols, "rtn_lstm_step");
  take(rtn_abi.sequence_mask, symbols, "rtn_sequence_mask");
  take(rtn_abi.column_sums, symbols, "rtn_column_sums");
  take(rtn_abi.column_sums_workspace_bytes, symbols, "rtn_column_sums_workspace_bytes");
  take(rtn_abi.transposed_product, symbols, "rtn_transposed_product");
  take(rtn_abi.transposed_product_workspace_bytes, symbols, "rtn_transposed_product_workspace_bytes");
  watch().exception = aborted;
  ready = true;
}

}  // namespace

// The op's device implementation per execution mode; the schemas are defined by make_op.
TORCH_LIBRARY_IMPL(NativeLstm2, CUDA, m) { m.impl("NativeLstm2", &lstm2_op<RTN_MODE_AUTO>); }
TORCH_LIBRARY_IMPL(NativeLstm2_persistent, CUDA, m) { m.impl("NativeLstm2_persistent", &lstm2_op<RTN_MODE_PERSISTENT>); }
TORCH_LIBRARY_IMPL(NativeLstm2_graph, CUDA, m) { m.impl("NativeLstm2_graph", &lstm2_op<RTN_MODE_GRAPH>); }
TORCH_LIBRARY_IMPL(NativeLstm2_stepwise, CUDA, m) { m.impl("NativeLstm2_stepwise", &lstm2_op<RTN_MODE_STEPWISE>); }

PYBIND11_MODULE(_rtn_torch, m) {
  m.def("init", &init);
  m.def("lstm2_multi", &py_lstm2_multi);
  m.def("last_output", &last_output);
  m.def("lstm_step", &lstm_step);
  m.def("lstm2_grad_multi", &py_lstm2_grad_multi);
  m.def("sequence_mask", &sequence_mask);
  m.def("lstm_layer", &lstm_layer);
  m.def("watch_before", [](const std::string& what, int count) {
    static std::mutex mu;
    static std::vector<std::unique_ptr<std::string>> kept;  // (a handful of texts; the watch keeps pointers)
    const char* text = nullptr;
    {
      std::lock_guard<std::mutex> lock(mu);
      for (const auto& k : kept)
        if (*k == what) text = k->c_str();
      if (!text) {
        kept.push_back(std::make_unique<std::string>(what));
        text = kept.back()->c_str();
      }
    }
    return watch().before(text, count, is_capturing(c10::hip::getCurrentHIPStream().stream()));
  });
  m.def("watch_after", [](bool failed) {
    rtn_abi.set_abort_word(nullptr, 0);
    if (failed) return;
    const auto stream = c10::hip::getCurrentHIPStream();
    watch().after(at::Device(at::kCUDA, stream.device_index()), stream.stream());
  });
  m.def("watch_poll", [] { watch().poll(); });
  m.def("watch_drain", [] { watch().drain(); });
  m.def("watch_checked", [] { return watch().checked; });
  m.def("watch_synchronous", [](int v) { watch().synchronous = v; });
}
