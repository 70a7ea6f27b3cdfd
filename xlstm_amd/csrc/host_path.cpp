// Native host path of the calls a program makes often: a decode step, an inference call and a training call of a cell
// and of a layer (training: in float32).  What the Python layers of cell.py, layer.py and functional.py do for such a call - look at dtypes, strides,
// versions and modes, allocate the outputs, fill an argument block, launch - takes 15 us per cell call and 75 us per
// layer call there, more than the kernels run; here it takes about 4 and 8.
//
// Every function returns None, with nothing launched, for a call that is not one of those it covers (autograd is
// recording, hooks are registered, another dtype or layout ...): the caller then takes its general path.  That is looked at
// in front of everything else and said by return values: an exception costs 7 us and more in a process with as many
// libraries as this one, and programs whose calls all take the general path pay for it on every one.  The results are
// those of the general path: the same kernels with the same arguments.
//
// A plain CPython extension over ATen (no pybind11: its argument casters cost as much as the rest of a step call).
// The engine's C entry points come as addresses from the library that _lib.py has loaded, so that one loaded engine
// serves both.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <vector>

#include "xlstm_amd.h"

namespace {

// ---- what bind() hands over from Python
struct Engine {
  decltype(&xs_slstm_step) step = nullptr;
  decltype(&xs_slstm_forward_watched) forward = nullptr;
  decltype(&xs_slstm_workspace_bytes) workspace_bytes = nullptr;
  decltype(&xs_last_error) last_error = nullptr;
  decltype(&xs_causal_conv_silu) conv = nullptr;
  decltype(&xs_causal_conv_silu_token) conv_token = nullptr;
  decltype(&xs_headwise_gates) gates = nullptr;
  decltype(&xs_headwise_group_norm) norm = nullptr;
  decltype(&xs_slstm_train_coef_floats) coef_floats = nullptr;
  decltype(&xs_slstm_train_exchange_bytes) exchange_bytes = nullptr;
  decltype(&xs_slstm_train_forward) train_forward = nullptr;
  decltype(&xs_slstm_train_backward) train_backward = nullptr;
  decltype(&xs_slstm_backward_params) backward_params = nullptr;
  decltype(&xs_layer_step_fits) layer_step_fits = nullptr;
  decltype(&xs_layer_step) layer_step = nullptr;
  decltype(&xs_layer_front) layer_front = nullptr;
  decltype(&xs_layer_norm) layer_norm = nullptr;
  decltype(&xs_layer_scratch_floats) layer_scratch = nullptr;
  decltype(&xs_layer_front_backward) layer_front_backward = nullptr;
  bool own_parts = true;                  // the parts of a layer's step are the engine's own: one kernel may stand for them
  PyObject *error = nullptr;              // functional.EngineError
  PyObject *global_hooks[2] = {nullptr, nullptr};  // hooks on every module of the process
} g_engine;

// interned attribute and dictionary keys
struct Names {
  PyObject *r, *b, *weight, *bias, *conv_state, *slstm_state, *input_shape, *output_shape, *keep_state_fp32, *config;
  PyObject *modules, *parameters, *forward_hooks, *forward_pre_hooks, *training, *p, *eps, *conv1d, *conv, *fgate, *igate, *zgate, *ogate;
  PyObject *group_norm, *slstm_cell, *dropout, *fused_pre_ops, *bsgnh, *cut, *clipval, *gradients_with_graph;
} g_names;

struct PyRef {  // owns one reference
  PyObject *o;
  explicit PyRef(PyObject *p = nullptr) : o(p) {}
  ~PyRef() { Py_XDECREF(o); }
  PyRef(const PyRef &) = delete;
  PyRef &operator=(const PyRef &) = delete;
  PyObject *release() { PyObject *p = o; o = nullptr; return p; }
};

struct PythonError {};  // a Python exception is set
struct EngineFailed { std::string what; };  // an entry point of the engine said no (thrown without the GIL)
inline void launched(int rc) {
  if (rc != XS_OK) throw EngineFailed{"xlstm_amd error " + std::to_string(rc) + ": " + g_engine.last_error()};
}

// The GIL is given up around allocations (which may reach the driver) and launches (which block when a queue is full), so
// that the other Python threads of a serving process run on.  What a call has of a cell is therefore taken with the GIL
// held - tensors and argument blocks by value, the plan by a reference of its own - and what it leaves there is written
// with the GIL held again: another thread may be in the same cell meanwhile.
struct WithoutGil {
  PyThreadState *state = PyEval_SaveThread();
  WithoutGil() = default;
  ~WithoutGil() { PyEval_RestoreThread(state); }
  WithoutGil(const WithoutGil &) = delete;
  WithoutGil &operator=(const WithoutGil &) = delete;
};

inline const at::Tensor *tensor_of(PyObject *o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }  // or null
inline bool absent(PyObject *o) { return o == nullptr || o == Py_None; }
inline bool optional_tensor(PyObject *o, const at::Tensor *&t) {  // false: neither a tensor nor None
  t = absent(o) ? nullptr : tensor_of(o);
  return t || absent(o);
}

inline void *stream_of(const at::Device &d) { return (void *)c10::hip::getCurrentHIPStream(d.index()).stream(); }
inline int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? XS_BF16 : XS_F32; }
inline bool aligned(const void *p, uintptr_t n) { return ((uintptr_t)p) % n == 0; }

// the version of a tensor's data, or 0 where none is kept (inference mode)
inline uint32_t version_of(const at::Tensor &t) { return t.is_inference() ? 0u : t._version(); }
inline bool versioned(const at::Tensor &t) { return !t.is_inference(); }

bool capturing(const at::Device &d) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  const hipStream_t stream = (hipStream_t)stream_of(d);  // (the null stream cannot be captured)
  return stream && (hipStreamIsCapturing(stream, &st) != hipSuccess || st != hipStreamCaptureStatusNone);
}

// ---- abort words: pinned host words that a sequence kernel writes when one of its bounded waits ran out.  Pages of
// words live as long as the process (a kernel of a cell that is gone may still be running), a word given back is the
// last to be handed out again, and there are no more words than cells were alive at once (rounded up to a page).
class WordPool {
 public:
  uint32_t *take() {
    std::lock_guard<std::mutex> lock(mu_);
    if (next_ == free_.size()) {
      void *page = nullptr;
      if (hipHostMalloc(&page, 4096, hipHostMallocDefault) != hipSuccess) return nullptr;
      free_.clear(); next_ = 0;
      for (int i = 0; i < 4096 / 64; ++i) free_.push_back((uint32_t *)((char *)page + 64 * i));
    }
    uint32_t *w = free_[next_++];
    if (next_ > 1024) { free_.erase(free_.begin(), free_.begin() + (long)next_); next_ = 0; }
    __atomic_store_n(w, 0u, __ATOMIC_RELEASE);
    return w;
  }
  void give_back(uint32_t *w) {
    std::lock_guard<std::mutex> lock(mu_);
    free_.push_back(w);
  }
 private:
  std::mutex mu_;
  std::vector<uint32_t *> free_;  // [next_, end): free words, oldest first
  size_t next_ = 0;
} g_words;
using AbortWord = std::shared_ptr<uint32_t>;  // a cell's, and its backward calls' that are still to come
AbortWord take_word() {
  uint32_t *w = g_words.take();
  return w ? AbortWord(w, [](uint32_t *p) { g_words.give_back(p); }) : nullptr;
}

// ---- the bytes that training forwards have left, per device, for backward calls that are still to come: a share of what a
// device may hold is taken with the coefficients and goes with them
std::atomic<int64_t> g_kept_bytes[64];
class Share {
 public:
  static std::shared_ptr<Share> take(int device, int64_t bytes, int64_t limit) {  // null: that would be more than `limit`
    if (device < 0 || device >= 64) return nullptr;
    int64_t held = g_kept_bytes[device].load();
    do {
      if (bytes > limit - held) return nullptr;
    } while (!g_kept_bytes[device].compare_exchange_weak(held, held + bytes));
    return std::shared_ptr<Share>(new Share(device, bytes));
  }
  ~Share() { g_kept_bytes[device_] -= bytes_; }
 private:
  Share(int device, int64_t bytes) : device_(device), bytes_(bytes) {}
  const int device_;
  const int64_t bytes_;
};

// ---- where calls of a cell may still be running: the streams they went to.  Shared with the backward calls that are still to
// come; used without the GIL.  (An event behind every call would say it to the call, and costs 5 us on the device each:
// 198.9 -> 204.1 us a call of 4 x 256 tokens in float32.)
class CallsInFlight {
 public:
  void add(const at::Device &d) {  // behind a call on the current stream (not under capture: a replay reports to nobody)
    const auto s = c10::hip::getCurrentHIPStream(d.index());
    const Place place{(int)d.index(), (void *)s.stream(), s.stream() && s.id() == (c10::StreamId)(uintptr_t)s.stream()};
    std::lock_guard<std::mutex> lock(mu_);
    for (const Place &p : places_)
      if (p.device == place.device && (p.foreign ? place.foreign : p.stream == place.stream)) return;
    places_.push_back(place);
  }
  void wait() {
    std::vector<Place> waiting;
    {
      std::lock_guard<std::mutex> lock(mu_);
      waiting.swap(places_);  // (calls that come meanwhile are the next wait's)
    }
    for (const Place &p : waiting) {
      c10::OptionalDeviceGuard guard(at::Device(at::kCUDA, (c10::DeviceIndex)p.device));
      // (a stream that torch did not make may be gone by now: its device is waited for)
      if (p.foreign || hipStreamSynchronize((hipStream_t)p.stream) != hipSuccess) (void)hipDeviceSynchronize();
    }
  }
 private:
  struct Place { int device; void *stream; bool foreign; };
  std::mutex mu_;
  std::vector<Place> places_;  // (torch's streams are a few dozen per device, the others count as one)
};

// ---- one cell
struct CellPath {
  PyObject *parameters = nullptr;  // its parameter dict
  int64_t NH = 0, dh = 0;
  // decode: the plan (functional.StepPlan) whose argument block is used, and what it was made for
  PyObject *plan = nullptr;
  std::vector<PyObject *> recorded_plans;  // plans that a recorded graph reads, for as long as the cell lives
  xs_slstm_args *step_args = nullptr;
  int64_t step_B = 0;
  at::ScalarType step_dtype = at::kFloat;
  at::Device device{at::kCPU};
  const void *r_ptr = nullptr, *b_ptr = nullptr;
  uint32_t r_version = 0, b_version = 0;
  at::Tensor last_state, last_h;   // what the last step handed out (float32 state kept), and their versions
  uint32_t last_state_version = 0, last_h_version = 0;
  // sequences: a workspace per (device, stream); a call under capture has one of its own, which is the graph's (graphs that
  // were recorded on one stream may be replayed on several, beside eager calls on that stream)
  struct Workspace { int device; void *stream; at::Tensor t; };
  std::vector<Workspace> workspaces;
  at::Tensor last_workspace;
  AbortWord abort_word;
  std::shared_ptr<CallsInFlight> calls = std::make_shared<CallsInFlight>();

  bool weights(const at::Tensor *&r, const at::Tensor *&b) const {
    PyObject *ro = parameters ? PyDict_GetItem(parameters, g_names.r) : nullptr, *bo = parameters ? PyDict_GetItem(parameters, g_names.b) : nullptr;
    return ro && bo && (r = tensor_of(ro)) && (b = tensor_of(bo));
  }
  ~CellPath() {
    Py_XDECREF(parameters);
    Py_XDECREF(plan);
    for (PyObject *o : recorded_plans) Py_DECREF(o);
  }

  bool records(const at::Tensor &x, const at::Tensor *state, const at::Tensor &r, const at::Tensor &b) const {
    return at::GradMode::is_enabled() && (x.requires_grad() || r.requires_grad() || b.requires_grad() || (state && state->requires_grad()));
  }

  at::Tensor workspace(int64_t B, const at::Device &d) {
    void *stream = stream_of(d);
    const size_t need = g_engine.workspace_bytes((int32_t)B, 1, (int32_t)NH, (int32_t)dh);
    auto find = [&]() -> Workspace * {
      for (auto &it : workspaces)
        if (it.device == d.index() && it.stream == stream) return &it;
      return nullptr;
    };
    Workspace *w = find();
    const bool in_graph = capturing(d);
    if (in_graph || !w || (size_t)w->t.numel() < need) {
      at::Tensor fresh;
      {
        WithoutGil no_gil;
        fresh = at::empty({(int64_t)need}, at::TensorOptions().dtype(at::kByte).device(d));
      }
      if (in_graph) return fresh;
      w = find();
      if (!w) {
        // (a program that makes a new stream per call would otherwise collect workspaces without end; a stream's
        // allocations are handed on in stream order by the caching allocator, so dropping the oldest is safe)
        if (workspaces.size() >= 16) workspaces.erase(workspaces.begin());
        workspaces.push_back(Workspace{(int)d.index(), stream, fresh});
        w = &workspaces.back();
      } else if ((size_t)w->t.numel() < need) {
        w->t = fresh;
      }
    }
    return w->t;
  }

  void raise_if_aborted() {
    if (abort_word && __atomic_load_n(abort_word.get(), __ATOMIC_ACQUIRE)) {
      __atomic_store_n(abort_word.get(), 0u, __ATOMIC_RELEASE);
      PyErr_SetString(g_engine.error,
                      "an earlier sLSTM sequence call (forward or backward) on the hip backend gave up waiting for some of its "
                      "compute units (they were held by other work on the GPU); its outputs were set to NaN");
      throw PythonError{};
    }
  }
};

struct CellPathObject { PyObject_HEAD CellPath *c; };

// the config's output_shape as the strides of [S,B,H] memory: 'BNSH', 'SBH', 'BSH' or 'SBNH'
enum class OutShape { BNSH, SBH, BSH, SBNH };
bool out_shape(PyObject *config, OutShape &shape) {
  PyRef v(PyObject_GetAttr(config, g_names.output_shape));
  if (!v.o) throw PythonError{};
  const char *s = PyUnicode_Check(v.o) ? PyUnicode_AsUTF8(v.o) : nullptr;
  if (!s) { PyErr_Clear(); return false; }
  if (!strcmp(s, "BNSH")) shape = OutShape::BNSH;
  else if (!strcmp(s, "SBH")) shape = OutShape::SBH;
  else if (!strcmp(s, "BSH")) shape = OutShape::BSH;
  else if (!strcmp(s, "SBNH")) shape = OutShape::SBNH;
  else return false;
  return true;
}
struct Shape4 { std::array<int64_t, 4> size, stride; int n; };
Shape4 shape_of(OutShape o, int64_t S, int64_t B, int64_t NH, int64_t dh) {
  const int64_t H = NH * dh;
  switch (o) {
    case OutShape::BNSH: return {{B, NH, S, dh}, {H, dh, B * H, 1}, 4};
    case OutShape::SBH: return {{S, B, H, 0}, {B * H, H, 1, 0}, 3};
    case OutShape::BSH: return {{B, S, H, 0}, {H, B * H, 1, 0}, 3};
    default: return {{S, B, NH, dh}, {B * H, H, dh, 1}, 4};
  }
}
bool input_is_bsgnh(PyObject *config) {
  PyRef v(PyObject_GetAttr(config, g_names.input_shape));
  if (!v.o) throw PythonError{};
  return v.o == g_names.bsgnh || PyUnicode_Compare(v.o, g_names.bsgnh) == 0;
}

// ---- one decode step into given buffers; the plan and the operand hint as sLSTMCell_hip._step_fast chooses them
struct StepBuffers { const at::Tensor *state_out = nullptr, *h_out = nullptr, *h_prev = nullptr; };
bool step_buffers(PyObject *state_out, PyObject *h_out, PyObject *h_prev, StepBuffers &s) {
  return optional_tensor(state_out, s.state_out) && optional_tensor(h_out, s.h_out) && optional_tensor(h_prev, s.h_prev);
}
// whether the cell's plan covers a step of B rows of x (the cell's input, or what a layer makes it from).  Looked at right in front
// of the Step: an attribute read in between may run Python code, and with it another thread that replaces the plan
bool step_fits(const CellPath &c, const at::Tensor &x, const at::Tensor &state, const StepBuffers &s) {
  const at::Tensor *r, *b;
  if (!c.plan || !c.weights(r, b) || r->data_ptr() != c.r_ptr || b->data_ptr() != c.b_ptr || version_of(*r) != c.r_version ||
      version_of(*b) != c.b_version)
    return false;
  const int64_t B = c.step_B, H = c.NH * c.dh;
  const auto dt = c.step_dtype;
  if (x.scalar_type() != dt || !x.is_cuda() || x.device() != c.device || !x.is_contiguous() || x.dim() != 3 || x.size(0) != B || x.size(1) != 1 ||
      c.records(x, &state, *r, *b))
    return false;
  auto state_like = [&](const at::Tensor &t) {
    return t.scalar_type() == at::kFloat && t.is_contiguous() && t.device() == c.device && t.dim() == 3 && t.size(0) == 4 && t.size(1) == B && t.size(2) == H;
  };
  auto h_like = [&](const at::Tensor &t) { return t.scalar_type() == dt && t.numel() == B * H && t.device() == c.device; };
  return state_like(state) && (!s.state_out || state_like(*s.state_out)) && (!s.h_out || (h_like(*s.h_out) && s.h_out->is_contiguous())) &&
         (!s.h_prev || dt != at::kBFloat16 || h_like(*s.h_prev));
}
// one decode step of the cell's plan: made and left with the GIL held, run without it
struct Step {
  CellPath &c;
  PyRef plan;        // (it owns the R and the bias that the argument block points to)
  xs_slstm_args a;
  const int64_t B, H;
  const at::Device device;
  const at::ScalarType dtype;
  at::Tensor last_state, last_h;
  uint32_t last_state_version, last_h_version;
  at::Tensor h, state;  // h: [1,B,H] memory, state: float32 [4,B,H]

  explicit Step(CellPath &cell)
      : c(cell), plan(cell.plan), a(*cell.step_args), B(cell.step_B), H(cell.NH * cell.dh), device(cell.device), dtype(cell.step_dtype),
        last_state(cell.last_state), last_h(cell.last_h), last_state_version(cell.last_state_version), last_h_version(cell.last_h_version) {
    Py_INCREF(plan.o);
    if (capturing(device) && std::find(c.recorded_plans.begin(), c.recorded_plans.end(), plan.o) == c.recorded_plans.end()) {
      c.recorded_plans.push_back(plan.o);  // (steps of another batch size or of changed parameters replace the plan, replays read on)
      Py_INCREF(plan.o);
    }
  }
  // wx: contiguous [B,1,4H]; everything else as step_fits has found it
  void run(const at::Tensor &wx, const at::Tensor &s0, const StepBuffers &s, const Shape4 *h_shape) {
    fill(wx.options(), s0, s, h_shape);
    launch(wx);
  }
  void launch(const at::Tensor &wx) {
    a.wx = wx.data_ptr();
    launched(g_engine.step(&a));
  }
  // the argument block but for wx
  void fill(const at::TensorOptions &opts, const at::Tensor &s0, const StepBuffers &s, const Shape4 *h_shape) {
    if (s.h_out) h = *s.h_out;
    else if (h_shape) h = at::empty_strided(at::IntArrayRef(h_shape->size.data(), h_shape->n), at::IntArrayRef(h_shape->stride.data(), h_shape->n), opts);
    else h = at::empty({1, B, H}, opts);
    state = s.state_out ? *s.state_out : at::empty({4, B, H}, s0.options());
    a.h_prev = nullptr;
    if (dtype == at::kBFloat16) {
      if (s.h_prev) {
        a.h_prev = s.h_prev->data_ptr();
      } else if (last_state.defined() && last_state.is_same(s0) && versioned(s0) && version_of(s0) == last_state_version &&
                 version_of(last_h) == last_h_version && last_h.data_ptr() != h.data_ptr()) {
        // The state this cell handed out last time comes back untouched: the h it returned with it is that state's y
        // plane in bfloat16, the operand the step kernel wants (half the bytes, and the pipelined kernel).
        a.h_prev = last_h.data_ptr();
      }
    }
    a.s0 = (const float *)s0.data_ptr();
    a.s_out = (float *)state.data_ptr();
    a.h_out = h.data_ptr();
    a.stream = stream_of(device);
  }
  void leave(bool keep_state) {
    if (c.plan == plan.o) *c.step_args = a;  // (the plan's block describes its last step)
    if (keep_state && versioned(state) && versioned(h)) {
      c.last_state = state; c.last_state_version = version_of(state);
      c.last_h = h; c.last_h_version = version_of(h);
    } else {
      c.last_state.reset(); c.last_h.reset();
    }
  }
};

bool recording(const CellPath &c, const at::Tensor &x, const at::Tensor *state) {
  if (!at::GradMode::is_enabled()) return false;
  const at::Tensor *r, *b;
  return !c.weights(r, b) || c.records(x, state, *r, *b);
}

// step(input, state, reset_mask, state_out, h_out, h_prev, config, keep_state_fp32) -> (output, state) or None
PyObject *cell_step_(CellPath &c, PyObject *const *args) {
  const at::Tensor *x = tensor_of(args[0]), *state = tensor_of(args[1]);
  StepBuffers s;
  OutShape shape;
  if (!absent(args[2]) || !x || !state || !c.plan || at::autocast::is_autocast_enabled(at::kCUDA) || !step_buffers(args[3], args[4], args[5], s) ||
      !input_is_bsgnh(args[6]) || !out_shape(args[6], shape) || !step_fits(c, *x, *state, s) || x->size(2) != 4 * c.NH * c.dh)
    Py_RETURN_NONE;
  const bool keep = args[7] == Py_True;
  c10::OptionalDeviceGuard guard(c.device);
  const Shape4 s4 = shape_of(shape, 1, c.step_B, c.NH, c.dh);
  Step step(c);
  at::Tensor h, state_out;
  {
    WithoutGil no_gil;
    step.run(*x, *state, s, &s4);
    h = s.h_out ? step.h.as_strided(at::IntArrayRef(s4.size.data(), s4.n), at::IntArrayRef(s4.stride.data(), s4.n)) : step.h;
    state_out = keep || step.dtype == at::kFloat ? step.state : step.state.to(step.dtype);
  }
  step.leave(keep);
  PyRef ph(THPVariable_Wrap(h)), ps(THPVariable_Wrap(state_out));
  if (!ph.o || !ps.o) throw PythonError{};
  return PyTuple_Pack(2, ph.o, ps.o);
}

// ---- a sequence through the cell (no autograd), as sLSTMCell_hip._run and functional.slstm_forward do it
bool mask_fits(const at::Tensor *m, int64_t B, int64_t T) { return !m || (m->is_cuda() && m->dim() == 2 && m->size(0) == B && m->size(1) == T); }
at::Tensor mask_bytes(const at::Tensor &m) {
  at::Tensor r = m;
  if (r.scalar_type() == at::kBool) r = r.is_contiguous() ? r.view(at::kByte) : r.to(at::kByte);
  else if (r.scalar_type() != at::kByte) r = r.ne(0).to(at::kByte);
  return r.stride(1) != 1 ? r.contiguous() : r;
}

// whether the sequence kernels take these tensors; x: [B,T,..] on the GPU
bool sequence_fits(const CellPath &c, const at::Tensor &x, int64_t B, int64_t T, const at::Tensor *state, const at::Tensor *mask) {
  const int64_t H = c.NH * c.dh;
  const auto dt = x.scalar_type();
  const at::Tensor *r, *b;
  if ((dt != at::kFloat && dt != at::kBFloat16) || T < 2 || B < 1 || !mask_fits(mask, B, T) || !c.weights(r, b)) return false;
  if (state && (!state->is_cuda() || state->dim() != 3 || state->size(0) != 4 || state->size(1) != B || state->size(2) != H)) return false;
  return r->device() == x.device() && b->device() == x.device() && r->is_contiguous() && b->is_contiguous() &&
         (r->scalar_type() == at::kFloat || r->scalar_type() == at::kBFloat16) && r->numel() == c.NH * 4 * c.dh * c.dh && b->numel() == 4 * H;
}
// the cell's abort word, made on first use (under capture there is none: no host memory is allocated, and a replay reports to nobody)
bool have_word(CellPath &c, const at::Device &d) {
  if (c.abort_word || capturing(d)) return true;
  AbortWord word;
  {
    WithoutGil no_gil;
    word = take_word();
  }
  if (!c.abort_word) c.abort_word = std::move(word);
  return c.abort_word != nullptr;
}

// A sequence through the cell: made and left with the GIL held, run without it.  train: the forward of a training call, which
// also leaves the backward pass its coefficients (no graph is recorded here)
struct Sequence {
  CellPath &c;
  at::Tensor r, b;
  const bool in_graph;
  AbortWord word;
  at::Tensor ws;
  at::Tensor h, state, coef, mask;  // h: [T,B,H] memory with the strides of `shape`, state: float32, mask: bytes

  Sequence(CellPath &cell, const at::Device &device, int64_t B) : c(cell), in_graph(capturing(device)) {
    const at::Tensor *rp, *bp;
    if (!c.weights(rp, bp)) { PyErr_SetString(PyExc_RuntimeError, "the cell has lost its parameters"); throw PythonError{}; }
    r = *rp; b = *bp;
    if (!in_graph) c.raise_if_aborted();
    word = in_graph ? nullptr : c.abort_word;
    ws = c.workspace(B, device);
  }
  // x: [B,T,4H] as sequence_fits has found it
  void run(at::Tensor x, const at::Tensor *s_in, const at::Tensor *mask_in, OutShape shape, bool train = false) {
    const int64_t H = c.NH * c.dh, B = x.size(0), T = x.size(1);
    const auto dt = x.scalar_type();
    const size_t esz = x.element_size();
    if (x.stride(2) != 1 || !aligned(x.data_ptr(), 16) || (x.stride(0) * esz) % 16 || (x.stride(1) * esz) % 16 || x.stride(1) < 4 * H ||
        (B > 1 && x.stride(0) < 4 * H))
      x = x.contiguous();
    if (dt == at::kFloat && r.scalar_type() != at::kFloat) r = r.to(at::kFloat);
    if (b.scalar_type() != at::kFloat) b = b.to(at::kFloat);  // (on every call: a copy kept would be another stream's, and a graph's)
    at::Tensor s0;
    if (s_in) s0 = s_in->to(at::kFloat).contiguous();
    if (mask_in) mask = mask_bytes(*mask_in);
    const Shape4 s4 = shape_of(shape, T, B, c.NH, c.dh);
    h = at::empty_strided(at::IntArrayRef(s4.size.data(), s4.n), at::IntArrayRef(s4.stride.data(), s4.n), x.options());
    state = at::empty({4, B, H}, x.options().dtype(at::kFloat));
    if (train) {
      const size_t n = g_engine.coef_floats((int32_t)B, (int32_t)T, (int32_t)c.NH, (int32_t)c.dh, dtype_code(dt));
      coef = at::empty({(int64_t)n}, state.options());
    }
    xs_slstm_args a{};
    a.B = (int32_t)B; a.T = (int32_t)T; a.NH = (int32_t)c.NH; a.dh = (int32_t)c.dh;
    a.wx_dtype = dtype_code(dt); a.r_dtype = dtype_code(r.scalar_type());
    a.wx = x.data_ptr(); a.wx_stride_b = x.stride(0); a.wx_stride_t = x.stride(1);
    a.r = r.data_ptr(); a.bias = (const float *)b.data_ptr();
    a.s0 = s_in ? (const float *)s0.data_ptr() : nullptr;
    a.reset = mask_in ? (const uint8_t *)mask.data_ptr() : nullptr; a.reset_stride_b = mask_in ? mask.stride(0) : 0;
    a.h_out = h.data_ptr(); a.s_out = (float *)state.data_ptr();
    a.workspace = ws.data_ptr(); a.workspace_bytes = (size_t)ws.numel();
    a.stream = stream_of(x.device());
    launched(train ? g_engine.train_forward(&a, (float *)coef.data_ptr(), word.get()) : g_engine.forward(&a, word.get()));
    if (!in_graph) c.calls->add(x.device());
  }
  void leave() { c.last_workspace = ws; }
};

// forward(input, state, reset_mask, config, keep_state_fp32) -> (output, state) or None
PyObject *cell_forward_(CellPath &c, PyObject *const *args) {
  const at::Tensor *xp = tensor_of(args[0]), *state, *mask;
  if (!xp || xp->dim() != 3 || !xp->is_cuda() || !optional_tensor(args[1], state) || !optional_tensor(args[2], mask) ||
      at::autocast::is_autocast_enabled(at::kCUDA) || recording(c, *xp, state))
    Py_RETURN_NONE;
  const at::Tensor &x = *xp;
  OutShape shape;
  const bool bsgnh = input_is_bsgnh(args[3]);
  if (!out_shape(args[3], shape) || x.size(2) != 4 * c.NH * c.dh || !sequence_fits(c, x, x.size(bsgnh ? 0 : 1), x.size(bsgnh ? 1 : 0), state, mask)) Py_RETURN_NONE;
  c10::OptionalDeviceGuard guard(x.device());
  if (!have_word(c, x.device())) Py_RETURN_NONE;
  const bool keep = args[4] == Py_True || x.scalar_type() == at::kFloat;
  Sequence s(c, x.device(), x.size(bsgnh ? 0 : 1));
  at::Tensor state_out;
  {
    WithoutGil no_gil;
    s.run(bsgnh ? x : x.permute({1, 0, 2}), state, mask, shape);
    state_out = keep ? s.state : s.state.to(x.scalar_type());
  }
  s.leave();
  PyRef ph(THPVariable_Wrap(s.h)), ps(THPVariable_Wrap(state_out));
  if (!ph.o || !ps.o) throw PythonError{};
  return PyTuple_Pack(2, ph.o, ps.o);
}

// ---- training: the engine's two backward calls (reverse pass, gradients of R and bias) as a node of the autograd graph,
// the way _CellFunction and functional._train_backward do it
struct ReverseInputs {
  at::Tensor r, h, state, mask, coef;  // as the forward used them; h: [T,B,H] memory
  AbortWord word;
  std::shared_ptr<CallsInFlight> calls;
  int64_t B, T, NH, dh;
  bool cut;
  double clip;
};
struct CellGradients { at::Tensor d_wx, d_r, d_bias, d_s0; };
// d_h: [T,B,H] with the strides (d_sb, d_st); d_s: float32 or undefined.  Called without the GIL
[[noreturn]] void engine_failed_in_backward(int rc) {
  const std::string what = g_engine.last_error();
  PyGILState_STATE gil = PyGILState_Ensure();
  PyErr_Format(g_engine.error, "xlstm_amd error %d: %s", rc, what.c_str());
  python_error e;
  e.persist();
  PyGILState_Release(gil);
  throw e;
}
CellGradients run_reverse(const ReverseInputs &in, const at::Tensor &d_h, int64_t d_sb, int64_t d_st, const at::Tensor &d_s) {
  const int64_t B = in.B, T = in.T, NH = in.NH, dh = in.dh, H = NH * dh;
  const auto dt = in.h.scalar_type();
  const auto f32 = in.h.options().dtype(at::kFloat);
  at::Tensor r = in.r;
  if (!(r.scalar_type() == at::kFloat || (r.scalar_type() == at::kBFloat16 && dt == at::kBFloat16))) r = r.to(at::kFloat);
  CellGradients g;
  g.d_wx = at::empty({B, T, 4 * H}, in.h.options());
  g.d_s0 = at::empty({4, B, H}, f32);
  g.d_r = at::empty({NH, 4 * dh, dh}, f32);
  g.d_bias = at::empty({4 * H}, f32);
  xs_slstm_bwd_args a{};
  a.B = (int32_t)B; a.T = (int32_t)T; a.NH = (int32_t)NH; a.dh = (int32_t)dh;
  a.dtype = dtype_code(dt);
  a.coef = (float *)in.coef.data_ptr(); a.d_h = d_h.data_ptr(); a.r = r.data_ptr(); a.h_out = in.h.data_ptr();
  at::Tensor d_s32, s0;
  if (d_s.defined()) { d_s32 = d_s.to(at::kFloat).contiguous(); a.d_s_final = (const float *)d_s32.data_ptr(); }
  if (in.state.defined()) { s0 = in.state.to(at::kFloat).contiguous(); a.s0 = (const float *)s0.data_ptr(); }
  at::Tensor mask = in.mask;
  if (mask.defined()) {
    if (mask.stride(0) >= (1 << 26)) mask = mask.contiguous();  // (the reverse kernel's offsets are 31-bit)
    a.reset = (const uint8_t *)mask.data_ptr(); a.reset_stride_b = mask.stride(0);
  }
  a.d_wx = (float *)g.d_wx.data_ptr(); a.d_wx_stride_b = g.d_wx.stride(0); a.d_wx_stride_t = g.d_wx.stride(1);
  a.d_wx_dtype = dtype_code(dt);
  a.d_s0 = (float *)g.d_s0.data_ptr(); a.d_r = (float *)g.d_r.data_ptr(); a.d_bias = (float *)g.d_bias.data_ptr();
  a.recurrent_cut = in.cut; a.recurrent_clipval = (float)in.clip;
  const size_t xbytes = g_engine.exchange_bytes((int32_t)B, (int32_t)NH, (int32_t)dh, a.dtype);
  at::Tensor exchange;
  if (xbytes) {  // a head spread over compute units: the ring its members exchange through, behind the abort word
    exchange = at::empty({(int64_t)(4096 + xbytes)}, in.h.options().dtype(at::kByte));
    a.counters = (unsigned int *)exchange.data_ptr();
    a.exchange = (char *)exchange.data_ptr() + 4096;
  }
  a.stream = stream_of(in.h.device());
  const bool in_graph = capturing(in.h.device());
  int rc = g_engine.train_backward(&a, d_sb, d_st, dtype_code(r.scalar_type()), in_graph ? nullptr : in.word.get());
  if (rc == XS_OK) rc = g_engine.backward_params(&a);
  if (rc != XS_OK) engine_failed_in_backward(rc);
  if (!in_graph) in.calls->add(in.h.device());
  return g;
}

// the gradient of the output as the reverse pass reads it: [S,B,NH,dh] or [S,B,1,H] of the output's type, with the strides of a
// row and of a step
at::Tensor output_gradient(const ReverseInputs &in, OutShape shape, const at::Tensor &given, int64_t &sb, int64_t &st) {
  const int64_t H = in.NH * in.dh;
  auto sbh = [&](const at::Tensor &t) {
    switch (shape) {
      case OutShape::BNSH: return t.permute({2, 0, 1, 3});
      case OutShape::SBH: return t.unsqueeze(2);
      case OutShape::BSH: return t.permute({1, 0, 2}).unsqueeze(2);
      default: return t;
    }
  };
  at::Tensor d = given.defined() ? sbh(given) : at::zeros({in.T, in.B, 1, H}, in.h.options());
  const int64_t esz = in.h.element_size();
  sb = in.B > 1 ? d.stride(1) : H; st = d.stride(0);
  if (d.scalar_type() != in.h.scalar_type() || d.stride(3) != 1 || (d.size(2) > 1 && d.stride(2) != in.dh) || !aligned(d.data_ptr(), 16) ||
      (sb * esz) % 16 || (st * esz) % 16 || sb >= (1 << 25) || sb < 0 || st < 0) {
    d = d.to(in.h.scalar_type()).contiguous();
    sb = H; st = in.B * H;
  }
  return d;
}

using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// What a call saved, as its kernels left it: hooks on saved tensors may hand back the same values in another memory layout
// (torch.autograd.graph.save_on_cpu(pin_memory=True): contiguous in the order of the dimensions)
at::Tensor laid_out(const at::Tensor &t, at::IntArrayRef stride) {
  if (t.strides() == stride && aligned(t.data_ptr(), 16)) return t;
  at::Tensor out = at::empty_strided(t.sizes(), stride, t.options());
  return out.copy_(t);
}
at::Tensor laid_out(const at::Tensor &t) {  // contiguous
  if (t.is_contiguous() && aligned(t.data_ptr(), 16)) return t;
  return t.clone(at::MemoryFormat::Contiguous);
}
at::Tensor laid_out(const at::Tensor &h, OutShape shape, const ReverseInputs &in) {  // [T,B,H] memory
  const Shape4 s = shape_of(shape, in.T, in.B, in.NH, in.dh);
  TORCH_CHECK(h.sizes() == at::IntArrayRef(s.size.data(), s.n), "the hidden states of a call came back from a saved-tensor hook in another shape");
  return laid_out(h, at::IntArrayRef(s.stride.data(), s.n));
}

struct CellBackward : public torch::autograd::Node {
  // (input and bias are not read again: a change of theirs in front of the backward is refused like one of R.  The
  // coefficients are saved like a tensor of the caller's, so that checkpointing and offloading hooks see them)
  SavedVariable x, r, b, h, state, coef;
  bool has_state = false, transposed_input = false;
  std::shared_ptr<Share> share;  // the coefficients'
  ReverseInputs in;  // (its saved tensors are filled in when the backward runs)
  OutShape shape = OutShape::BNSH;
  at::ScalarType r_dtype = at::kFloat, b_dtype = at::kFloat, s_dtype = at::kFloat;

  std::string name() const override { return "sLSTMCellBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (SavedVariable *v : {&x, &r, &b, &h, &state, &coef}) v->reset_data();
    in.mask.reset();
    share.reset();
  }
  variable_list apply(variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    at::NoGradGuard no_grad;
    ReverseInputs call = in;
    x.unpack();
    b.unpack();
    call.h = h.unpack(shared_from_this());
    c10::OptionalDeviceGuard guard(call.h.device());
    call.h = laid_out(call.h, shape, call);
    call.r = laid_out(r.unpack());
    call.coef = laid_out(coef.unpack());
    if (has_state) call.state = laid_out(state.unpack());
    int64_t sb, st;
    const at::Tensor d = output_gradient(call, shape, grads[0], sb, st);
    CellGradients g = run_reverse(call, d, sb, st, grads[1]);
    variable_list out(has_state ? 4 : 3);
    out[0] = transposed_input ? g.d_wx.permute({1, 0, 2}) : g.d_wx;
    out[1] = g.d_r.to(r_dtype);
    out[2] = g.d_bias.to(b_dtype);
    if (has_state) out[3] = g.d_s0.to(s_dtype);
    return out;
  }
};

// train(input, state, reset_mask, config, keep_state_fp32, bytes of coefficients that a device may hold) -> (output, state) with
// their place in the graph, or None
PyObject *cell_train_(CellPath &c, PyObject *const *args) {
  const at::Tensor *xp = tensor_of(args[0]), *state, *mask, *rp, *bp;
  if (!xp || xp->dim() != 3 || !xp->is_cuda() || !optional_tensor(args[1], state) || !optional_tensor(args[2], mask) ||
      at::autocast::is_autocast_enabled(at::kCUDA) || !c.weights(rp, bp) || !recording(c, *xp, state))
    Py_RETURN_NONE;
  const at::Tensor &x = *xp;
  OutShape shape;
  const bool bsgnh = input_is_bsgnh(args[3]);
  if (!out_shape(args[3], shape) || x.size(2) != 4 * c.NH * c.dh || !sequence_fits(c, x, x.size(bsgnh ? 0 : 1), x.size(bsgnh ? 1 : 0), state, mask) ||
      !g_engine.coef_floats(1, 1, (int32_t)c.NH, (int32_t)c.dh, dtype_code(x.scalar_type())))
    Py_RETURN_NONE;
  for (const at::Tensor *t : {&x, rp, bp, state})
    if (t && t->_fw_grad(0).defined()) Py_RETURN_NONE;  // (forward mode: the general path refuses it)
  PyRef cut(PyObject_GetAttr(args[3], g_names.cut)), clip(PyObject_GetAttr(args[3], g_names.clipval));
  if (!cut.o || !clip.o) throw PythonError{};
  const int cut_on = PyObject_IsTrue(cut.o);
  const double clipval = clip.o == Py_None ? 0.0 : PyFloat_AsDouble(clip.o);
  if (PyErr_Occurred()) throw PythonError{};
  c10::OptionalDeviceGuard guard(x.device());
  if (!have_word(c, x.device())) Py_RETURN_NONE;
  const bool keep = args[4] == Py_True || x.scalar_type() == at::kFloat;
  const int64_t limit = PyLong_AsLongLong(args[5]);
  if (PyErr_Occurred()) throw PythonError{};
  std::shared_ptr<Share> share = Share::take(x.device().index(), 4 * (int64_t)g_engine.coef_floats((int32_t)x.size(bsgnh ? 0 : 1), (int32_t)x.size(bsgnh ? 1 : 0),
                                             (int32_t)c.NH, (int32_t)c.dh, dtype_code(x.scalar_type())), limit);
  if (!share) Py_RETURN_NONE;  // (the backward call of the general path makes them again)
  Sequence s(c, x.device(), x.size(bsgnh ? 0 : 1));
  const at::Tensor r = s.r, b = s.b;
  at::Tensor state_out;
  {
    WithoutGil no_gil;
    {
      at::NoGradGuard no_grad;
      s.run(bsgnh ? x : x.permute({1, 0, 2}), state, mask, shape, true);
    }
    auto node = std::shared_ptr<CellBackward>(new CellBackward(), torch::autograd::deleteNode);
    node->set_next_edges(state ? torch::autograd::collect_next_edges(x, r, b, *state) : torch::autograd::collect_next_edges(x, r, b));
    node->x = SavedVariable(x, false);
    node->r = SavedVariable(r, false);
    node->b = SavedVariable(b, false);
    node->coef = SavedVariable(s.coef, false);
    node->share = std::move(share);
    node->has_state = state != nullptr;
    if (state) { node->state = SavedVariable(*state, false); node->s_dtype = state->scalar_type(); }
    node->transposed_input = !bsgnh;
    node->shape = shape;
    node->r_dtype = r.scalar_type(); node->b_dtype = b.scalar_type();
    node->in.mask = s.mask; node->in.word = s.word; node->in.calls = c.calls;
    node->in.B = s.state.size(1); node->in.T = x.size(bsgnh ? 1 : 0); node->in.NH = c.NH; node->in.dh = c.dh;
    node->in.cut = cut_on != 0; node->in.clip = clipval;
    torch::autograd::set_history(s.h, node);
    torch::autograd::set_history(s.state, node);
    node->h = SavedVariable(s.h, true);
    state_out = keep ? s.state : s.state.to(x.scalar_type());
  }
  s.leave();
  PyRef ph(THPVariable_Wrap(s.h)), ps(THPVariable_Wrap(state_out));
  if (!ph.o || !ps.o) throw PythonError{};
  return PyTuple_Pack(2, ph.o, ps.o);
}

template <PyObject *(*F)(CellPath &, PyObject *const *), int N>
PyObject *cell_call(PyObject *self, PyObject *const *args, Py_ssize_t n) {
  if (n != N) { PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n); return nullptr; }
  try {
    return F(*((CellPathObject *)self)->c, args);
  } catch (const PythonError &) {
    return nullptr;
  } catch (const EngineFailed &e) {
    PyErr_SetString(g_engine.error, e.what.c_str());
    return nullptr;
  } catch (...) {  // (out of memory and the like: as the type that torch raises for it)
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

// set_plan(plan, address of its argument block, B, r, b): the next steps of that batch size and of these parameters
PyObject *cell_set_plan_(CellPath &c, PyObject *const *args) {
  const at::Tensor *rp = tensor_of(args[3]), *bp = tensor_of(args[4]);
  if (!rp || !bp) { PyErr_SetString(PyExc_TypeError, "set_plan: r and b are tensors"); throw PythonError{}; }
  const at::Tensor &r = *rp, &b = *bp;
  c.step_args = (xs_slstm_args *)PyLong_AsVoidPtr(args[1]);
  c.step_B = PyLong_AsLongLong(args[2]);
  c.step_dtype = c.step_args->wx_dtype == XS_BF16 ? at::kBFloat16 : at::kFloat;
  c.device = r.device();
  c.r_ptr = r.data_ptr(); c.b_ptr = b.data_ptr();
  c.r_version = version_of(r); c.b_version = version_of(b);
  Py_INCREF(args[0]);
  Py_XSETREF(c.plan, args[0]);
  Py_RETURN_NONE;
}
// workspace(B, a tensor on the device) -> the workspace of calls on that device's current stream
PyObject *cell_workspace_(CellPath &c, PyObject *const *args) {
  const at::Tensor *like = tensor_of(args[1]);
  if (!like) { PyErr_SetString(PyExc_TypeError, "workspace: a tensor on the device"); throw PythonError{}; }
  return THPVariable_Wrap(c.workspace(PyLong_AsLongLong(args[0]), like->device()));
}
// report_to(handle): the abort word and the calls in flight of another cell (a capsule that owns a Reports) take this one's
struct Reports { AbortWord word; std::shared_ptr<CallsInFlight> calls; };
constexpr const char *kReports = "reports";
PyObject *cell_report_to_(CellPath &c, PyObject *const *args) {
  const Reports *r = (const Reports *)PyCapsule_GetPointer(args[0], kReports);
  if (!r) throw PythonError{};
  c.abort_word = r->word; c.calls = r->calls;
  Py_RETURN_NONE;
}
// last_workspace() -> the workspace of the latest sequence call
PyObject *cell_last_workspace_(CellPath &c, PyObject *const *) {
  if (!c.last_workspace.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(c.last_workspace);
}
// poll(block) -> whether a sequence call gave up since the last poll; block: waits for this cell's calls in flight first
PyObject *cell_poll_(CellPath &c, PyObject *const *args) {
  if (args[0] == Py_True) {
    const std::shared_ptr<CallsInFlight> calls = c.calls;
    WithoutGil no_gil;
    calls->wait();
  }
  if (c.abort_word && __atomic_exchange_n(c.abort_word.get(), 0u, __ATOMIC_ACQ_REL)) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
}

PyObject *cell_new(PyTypeObject *type, PyObject *args, PyObject *) {
  PyObject *parameters;
  long long NH, dh;
  if (!PyArg_ParseTuple(args, "O!LL", &PyDict_Type, &parameters, &NH, &dh)) return nullptr;
  CellPathObject *self = (CellPathObject *)type->tp_alloc(type, 0);
  if (!self) return nullptr;
  self->c = new CellPath;
  Py_INCREF(parameters);
  self->c->parameters = parameters;
  self->c->NH = NH; self->c->dh = dh;
  return (PyObject *)self;
}
// (the parameters' hooks may refer to the cell, which holds this path: the collector has to see through it)
int cell_traverse(PyObject *self, visitproc visit, void *arg) {
  CellPath *c = ((CellPathObject *)self)->c;
  Py_VISIT(Py_TYPE(self));
  if (c) {
    Py_VISIT(c->parameters);
    Py_VISIT(c->plan);
    for (PyObject *o : c->recorded_plans) Py_VISIT(o);
  }
  return 0;
}
int cell_clear(PyObject *self) {
  CellPath *c = ((CellPathObject *)self)->c;
  if (c) {
    c->step_args = nullptr;  // (the plan's)
    Py_CLEAR(c->parameters);
    Py_CLEAR(c->plan);
    std::vector<PyObject *> recorded;
    recorded.swap(c->recorded_plans);
    for (PyObject *o : recorded) Py_DECREF(o);
  }
  return 0;
}
void cell_dealloc(PyObject *self) {
  PyTypeObject *type = Py_TYPE(self);
  PyObject_GC_UnTrack(self);
  delete ((CellPathObject *)self)->c;
  type->tp_free(self);
  Py_DECREF(type);
}

PyMethodDef cell_methods[] = {
    {"step", (PyCFunction)(void *)cell_call<cell_step_, 8>, METH_FASTCALL, nullptr},
    {"forward", (PyCFunction)(void *)cell_call<cell_forward_, 5>, METH_FASTCALL, nullptr},
    {"train", (PyCFunction)(void *)cell_call<cell_train_, 6>, METH_FASTCALL, nullptr},
    {"set_plan", (PyCFunction)(void *)cell_call<cell_set_plan_, 5>, METH_FASTCALL, nullptr},
    {"workspace", (PyCFunction)(void *)cell_call<cell_workspace_, 2>, METH_FASTCALL, nullptr},
    {"last_workspace", (PyCFunction)(void *)cell_call<cell_last_workspace_, 0>, METH_FASTCALL, nullptr},
    {"poll", (PyCFunction)(void *)cell_call<cell_poll_, 1>, METH_FASTCALL, nullptr},
    {"report_to", (PyCFunction)(void *)cell_call<cell_report_to_, 1>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyType_Slot cell_slots[] = {{Py_tp_new, (void *)cell_new}, {Py_tp_dealloc, (void *)cell_dealloc},
                            {Py_tp_traverse, (void *)cell_traverse}, {Py_tp_clear, (void *)cell_clear}, {Py_tp_methods, cell_methods}, {0, nullptr}};
PyType_Spec cell_spec = {"_xlstm_host.CellPath", sizeof(CellPathObject), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC, cell_slots};
PyTypeObject *g_cell_type = nullptr;

// ---- one layer: its submodules are looked up by name in the module dictionaries on every call (they may be replaced)
PyObject *attribute(PyObject *o, PyObject *name) {  // new reference; nn.Module keeps these in its __dict__
  PyObject *v = PyObject_GetAttr(o, name);
  if (!v) throw PythonError{};
  return v;
}
PyObject *module_dict(PyObject *module, PyObject *which) {  // borrowed from the module, or null
  PyRef d(attribute(module, which));
  return PyDict_Check(d.o) ? d.o : nullptr;  // (the module holds it)
}
PyObject *submodule(PyObject *module, PyObject *name) {  // borrowed, or null
  PyObject *modules = module_dict(module, g_names.modules), *m = modules ? PyDict_GetItem(modules, name) : nullptr;
  return absent(m) ? nullptr : m;
}
// a parameter of a module in the type and place of x; None: an undefined tensor.  false: another type, layout or device, or no
// parameter of that name (it may be a plain attribute meanwhile, made from other tensors)
bool parameter(PyObject *module, PyObject *name, const at::Tensor &x, at::Tensor &out) {
  PyObject *parameters = module_dict(module, g_names.parameters), *o = parameters ? PyDict_GetItem(parameters, name) : nullptr;
  const at::Tensor *t;
  if (!o || !optional_tensor(o, t)) return false;
  if (t) out = *t;
  return !t || (t->scalar_type() == x.scalar_type() && t->is_contiguous() && t->device() == x.device() && aligned(t->data_ptr(), 16));
}
bool has_hooks(PyObject *module) {
  PyObject *after = module_dict(module, g_names.forward_hooks), *before = module_dict(module, g_names.forward_pre_hooks);
  return !after || !before || PyDict_Size(after) || PyDict_Size(before);
}

struct LayerParts {
  PyRef cell_config{nullptr};
  CellPath *cell = nullptr;
  bool keep_state = false;
  at::Tensor conv_w, conv_b, gate[4], norm_w;
  double eps = 1e-5;
  int64_t K = 0, NH = 0, dh = 0, D = 0;
  bool float32 = false;
};

// what a layer call needs of its modules; false unless the engine's kernels apply (bfloat16: sLSTMLayer._fused) and a gradient is
// recorded (`train`: dropout and norm behind the cell are called as modules then) or none is
bool collect(PyObject *layer, PyObject *cell_path, const at::Tensor &x, LayerParts &p, bool train = false) {
  p.cell = ((CellPathObject *)cell_path)->c;
  p.NH = p.cell->NH; p.dh = p.cell->dh; p.D = p.NH * p.dh;
  p.float32 = x.scalar_type() == at::kFloat;
  if (x.dim() != 3 || (!p.float32 && x.scalar_type() != at::kBFloat16) || !x.is_cuda() || x.size(2) != p.D ||
      (p.float32 ? p.dh % 4 || p.dh > 512 : p.dh % 64 || p.dh > 1024) || at::autocast::is_autocast_enabled(at::kCUDA))
    return false;
  bool records = recording(*p.cell, x, nullptr);
  if (records && !train) return false;
  for (PyObject *h : g_engine.global_hooks)
    if (h && PyDict_Size(h)) return false;
  PyObject *cell = submodule(layer, g_names.slstm_cell), *conv1d = submodule(layer, g_names.conv1d);
  PyObject *conv = conv1d ? submodule(conv1d, g_names.conv) : nullptr;
  PyObject *norm = submodule(layer, g_names.group_norm), *dropout = submodule(layer, g_names.dropout);
  if (!cell || !conv || !norm || !dropout || has_hooks(cell) || (!train && has_hooks(dropout))) return false;
  {
    PyRef fused(attribute(layer, g_names.fused_pre_ops));
    if (fused.o != Py_True) return false;
    PyRef training(attribute(dropout, g_names.training)), rate(attribute(dropout, g_names.p));
    const double dp = PyFloat_AsDouble(rate.o);
    if (PyErr_Occurred()) { PyErr_Clear(); return false; }
    if (!train && training.o == Py_True && dp != 0.0) return false;
    PyRef keep(attribute(cell, g_names.keep_state_fp32)), eps(attribute(norm, g_names.eps));
    p.keep_state = keep.o == Py_True;
    p.eps = PyFloat_AsDouble(eps.o);
    if (PyErr_Occurred()) throw PythonError{};
    p.cell_config.o = attribute(cell, g_names.config);
  }
  OutShape shape;
  if (!input_is_bsgnh(p.cell_config.o) || !out_shape(p.cell_config.o, shape) || shape != OutShape::BNSH) return false;
  if (!parameter(conv, g_names.weight, x, p.conv_w) || !p.conv_w.defined() || !parameter(conv, g_names.bias, x, p.conv_b) ||
      (!train && !parameter(norm, g_names.weight, x, p.norm_w)))
    return false;
  // (the module called fgate feeds the i slot, igate the f slot)
  PyObject *gates[4] = {g_names.fgate, g_names.igate, g_names.zgate, g_names.ogate};
  for (int g = 0; g < 4; ++g) {
    PyObject *gate = submodule(layer, gates[g]);
    if (!gate || !parameter(gate, g_names.weight, x, p.gate[g]) || !p.gate[g].defined() || p.gate[g].numel() != p.NH * p.dh * p.dh) return false;
  }
  for (const at::Tensor *t : {&p.conv_w, &p.conv_b, &p.norm_w, &p.gate[0], &p.gate[1], &p.gate[2], &p.gate[3]})
    records |= at::GradMode::is_enabled() && t->defined() && t->requires_grad();
  p.K = p.conv_w.numel() / p.D;
  return p.K >= 2 && p.K <= 4 && records == train;
}

void run_conv(const LayerParts &p, const at::Tensor &x, const void *taps, int64_t taps_stride, const at::Tensor *mask, void *out, void *ring, void *stream, void *x_out = nullptr) {
  xs_conv_args a{};
  a.B = (int32_t)x.size(0); a.T = (int32_t)x.size(1); a.D = (int32_t)p.D; a.K = (int32_t)p.K;
  a.dtype = XS_BF16;
  a.x = x.data_ptr(); a.x_stride_b = x.stride(0); a.x_stride_t = x.stride(1);
  a.conv_state = taps; a.conv_state_stride_b = taps && x.size(0) > 1 ? taps_stride : 0;
  a.weight = p.conv_w.data_ptr(); a.bias = p.conv_b.defined() ? p.conv_b.data_ptr() : nullptr;
  a.reset = mask ? (const uint8_t *)mask->data_ptr() : nullptr; a.reset_stride_b = mask ? mask->stride(0) : 0;
  a.out = out; a.ring_out = ring; a.stream = stream;
  launched(x_out ? g_engine.conv_token(&a, x_out) : g_engine.conv(&a));
}
void run_gates(const LayerParts &p, const at::Tensor &x, const void *x_conv, void *out, void *stream) {
  xs_gates_args a{};
  a.M = (int32_t)(x.size(0) * x.size(1)); a.NH = (int32_t)p.NH; a.dh = (int32_t)p.dh;
  a.dtype = XS_BF16;
  a.x = x.data_ptr(); a.x_stride_row = p.D; a.x_conv = x_conv; a.x_conv_stride_row = p.D;
  for (int g = 0; g < 4; ++g) a.w[g] = p.gate[g].data_ptr();
  a.out = out; a.out_stride_row = 4 * p.D; a.stream = stream;
  launched(g_engine.gates(&a));
}
void run_norm(const LayerParts &p, const at::Tensor &h, int64_t B, int64_t T, void *out, void *stream) {
  xs_norm_args a{};
  a.B = (int32_t)B; a.T = (int32_t)T; a.NH = (int32_t)p.NH; a.dh = (int32_t)p.dh;
  a.dtype = XS_BF16; a.eps = (float)p.eps;
  a.x = h.data_ptr(); a.x_stride_b = p.D; a.x_stride_h = p.dh; a.x_stride_t = B * p.D;  // [T,B,H] memory
  a.weight = p.norm_w.defined() ? p.norm_w.data_ptr() : nullptr;
  a.out = out; a.stream = stream;
  launched(g_engine.norm(&a));
}

// the float32 kernels' argument block, with what a pass in either direction needs; x: contiguous
xs_layer_args float32_args(const LayerParts &p, const at::Tensor &x, const at::Tensor &x_conv, const at::Tensor *mask) {
  xs_layer_args a{};
  a.B = (int32_t)x.size(0); a.T = (int32_t)x.size(1); a.NH = (int32_t)p.NH; a.dh = (int32_t)p.dh; a.K = (int32_t)p.K;
  a.eps = (float)p.eps;
  auto ptr = [](const at::Tensor &t) { return t.defined() ? (const float *)t.data_ptr() : nullptr; };
  a.x = ptr(x); a.x_stride_b = x.stride(0); a.x_stride_t = x.stride(1);
  a.conv_w = ptr(p.conv_w); a.conv_b = ptr(p.conv_b); a.norm_w = ptr(p.norm_w);
  for (int g = 0; g < 4; ++g) a.gate_w[g] = ptr(p.gate[g]);
  a.reset = mask ? (const uint8_t *)mask->data_ptr() : nullptr; a.reset_stride_b = mask ? mask->stride(0) : 0;
  a.x_conv = (float *)x_conv.data_ptr();
  a.stream = stream_of(x.device());
  return a;
}

// (the kernels around the cell record no graph in inference calls)
bool wants_gradient(const at::Tensor &t) { return at::GradMode::is_enabled() && t.requires_grad(); }

// the taps in front of the first token: a [B,n,D] tensor of which the last K-1 inputs count
bool taps_of(const LayerParts &p, const at::Tensor &t, int64_t B, const void *&taps, int64_t &stride) {
  const int64_t n = t.dim() == 3 ? t.size(1) : 0;
  const int64_t esz = p.float32 ? 4 : 2;
  if (t.scalar_type() != (p.float32 ? at::kFloat : at::kBFloat16) || n < p.K - 1 || t.size(0) != B || t.size(2) != p.D || t.stride(2) != 1 ||
      t.stride(1) != p.D || t.stride(0) * esz % 16 || !t.is_cuda() || !aligned(t.data_ptr(), 16))
    return false;
  if (B > 1 && t.stride(0) < (p.K - 1) * p.D) return false;  // (rows that share memory, one state for all of them: laid out by the general path)
  stride = t.stride(0);
  taps = (const char *)t.data_ptr() + (n - (p.K - 1)) * p.D * esz;
  return true;
}

bool overlap(const void *a, int64_t a_bytes, const at::Tensor &b) {  // (b: contiguous)
  const char *pa = (const char *)a, *pb = (const char *)b.data_ptr();
  return a && pa < pb + b.nbytes() && pb < pa + a_bytes;
}

PyObject *states_dict(PyObject *conv_state, const at::Tensor &state) {
  PyRef s(THPVariable_Wrap(state)), d(PyDict_New());
  if (!s.o || !d.o || !conv_state || PyDict_SetItem(d.o, g_names.conv_state, conv_state) || PyDict_SetItem(d.o, g_names.slstm_state, s.o)) throw PythonError{};
  return d.release();
}
PyObject *first_of(PyObject *o) {  // a state that may come in a tuple or list of one
  if (PyTuple_Check(o)) return PyTuple_GET_SIZE(o) ? PyTuple_GET_ITEM(o, 0) : Py_None;
  if (PyList_Check(o)) return PyList_GET_SIZE(o) ? PyList_GET_ITEM(o, 0) : Py_None;
  return o;
}

// layer_step(layer, cell path, x, conv_state, slstm_state, slstm_state_out, conv_state_out, h_out, h_prev, out[, x_out])
//   -> (out, {"conv_state": (ring,), "slstm_state": state}) or None.  x_out: a buffer that x is left in as well
PyObject *layer_step_(PyObject *const *args) {
  const at::Tensor *xp = tensor_of(args[2]), *statep = tensor_of(args[4]), *ring_out, *out_given, *x_out;
  CellPath &c = *((CellPathObject *)args[1])->c;
  StepBuffers buffers;
  if (!xp || !statep || !c.plan || !step_buffers(args[5], args[7], args[8], buffers) || !optional_tensor(args[6], ring_out) ||
      !optional_tensor(args[9], out_given) || !optional_tensor(args[10], x_out))
    Py_RETURN_NONE;
  const at::Tensor &x = *xp, &state = *statep;
  LayerParts p;
  if (!collect(args[0], args[1], x, p) || p.float32 || !step_fits(c, x, state, buffers) || !aligned(x.data_ptr(), 16)) Py_RETURN_NONE;
  const int64_t B = x.size(0);
  if (B < 1) Py_RETURN_NONE;
  const void *taps = nullptr;
  int64_t taps_stride = 0;
  at::Tensor before;  // (held: it may come in a list, which another thread may change)
  PyObject *prev = absent(args[3]) ? nullptr : first_of(args[3]);
  if (!absent(prev)) {
    const at::Tensor *t = tensor_of(prev);
    if (!t || wants_gradient(*t) || t->dim() != 3 || (t->size(1) != p.K && t->size(1) != p.K - 1) || !taps_of(p, *t, B, taps, taps_stride)) Py_RETURN_NONE;  // (the general path asserts)
    before = *t;
  }
  const auto opts = x.options();
  if (ring_out && (ring_out->scalar_type() != at::kBFloat16 || ring_out->dim() != 3 || ring_out->size(0) != B || ring_out->size(1) != p.K ||
                   ring_out->size(2) != p.D || !ring_out->is_contiguous()))
    Py_RETURN_NONE;
  if (out_given && (out_given->scalar_type() != at::kBFloat16 || out_given->numel() != B * p.D || !out_given->is_contiguous())) Py_RETURN_NONE;
  if (x_out && x_out->data_ptr() == x.data_ptr()) x_out = nullptr;
  if (x_out && (x_out->scalar_type() != at::kBFloat16 || x_out->sizes() != x.sizes() || !x_out->is_contiguous() || x_out->device() != x.device() ||
                !aligned(x_out->data_ptr(), 16) || overlap(x.data_ptr(), x.nbytes(), *x_out)))
    Py_RETURN_NONE;
  c10::OptionalDeviceGuard guard(x.device());
  Step step(c);
  at::Tensor ring, out, state_out;
  {
    WithoutGil no_gil;
    void *stream = stream_of(x.device());
    ring = ring_out ? *ring_out : at::empty({B, p.K, p.D}, opts);
    out = out_given ? *out_given : at::empty({B, 1, p.D}, opts);
    step.fill(opts, state, buffers, nullptr);
    // (one kernel: its workgroups read a head's inputs while others write their units' results.  The parts have read x and the
    // taps before the step writes h and the state, so buffers that share memory go to them)
    const int64_t taps_bytes = taps ? 2 * ((B - 1) * taps_stride + (p.K - 1) * p.D) : 0;
    const bool shared = overlap(x.data_ptr(), x.nbytes(), ring) || overlap(x.data_ptr(), x.nbytes(), step.h) || overlap(x.data_ptr(), x.nbytes(), step.state) ||
                        overlap(taps, taps_bytes, step.h) || overlap(taps, taps_bytes, step.state) || (x_out && overlap(taps, taps_bytes, *x_out));
    if (g_engine.own_parts && !shared && g_engine.layer_step_fits((int32_t)B, (int32_t)p.NH, (int32_t)p.dh, (int32_t)p.K)) {
      xs_layer_step_args a{};
      a.cell = step.a;
      a.x = x.data_ptr();
      a.conv_state = taps; a.conv_state_stride_b = taps && B > 1 ? taps_stride : 0;
      a.conv_w = p.conv_w.data_ptr(); a.conv_b = p.conv_b.defined() ? p.conv_b.data_ptr() : nullptr;
      a.ring_out = ring.data_ptr(); a.x_out = x_out ? x_out->data_ptr() : nullptr; a.K = (int32_t)p.K;
      for (int g = 0; g < 4; ++g) a.gate_w[g] = p.gate[g].data_ptr();
      launched(g_engine.layer_step(&a));
    } else {
      at::Tensor wx = at::empty({B, 1, 4 * p.D}, opts), x_conv = at::empty({B, 1, p.D}, opts);
      const bool with_x = x_out && !overlap(taps, taps_bytes, *x_out);
      run_conv(p, x, taps, taps_stride, nullptr, x_conv.data_ptr(), ring.data_ptr(), stream, with_x ? x_out->data_ptr() : nullptr);
      run_gates(p, x, x_conv.data_ptr(), wx.data_ptr(), stream);
      step.launch(wx);
      if (x_out && !with_x) {
        at::NoGradGuard no_grad;
        x_out->copy_(x);
      }
    }
    run_norm(p, step.h, B, 1, out.data_ptr(), stream);
    state_out = p.keep_state ? step.state : step.state.to(at::kBFloat16);
  }
  step.leave(p.keep_state);
  PyRef po(THPVariable_Wrap(out)), pr(THPVariable_Wrap(ring)), tuple(nullptr);
  if (!po.o || !pr.o) throw PythonError{};
  tuple.o = PyTuple_Pack(1, pr.o);
  PyRef states(states_dict(tuple.o, state_out));
  return PyTuple_Pack(2, po.o, states.o);
}

// layer_forward(layer, cell path, x, conv_state, slstm_state, return_last_state, reset_mask) -> the layer's result or None
PyObject *layer_forward_(PyObject *const *args) {
  const at::Tensor *xp = tensor_of(args[2]), *state, *mask_in;
  if (!xp || !optional_tensor(args[4], state) || !optional_tensor(args[6], mask_in)) Py_RETURN_NONE;
  const at::Tensor &x_in = *xp;
  LayerParts p;
  if (x_in.dim() != 3 || x_in.size(1) < 2 || !collect(args[0], args[1], x_in, p)) Py_RETURN_NONE;
  const int64_t B = x_in.size(0), T = x_in.size(1);
  if (!sequence_fits(*p.cell, x_in, B, T, state, mask_in) || recording(*p.cell, x_in, state)) Py_RETURN_NONE;
  const void *taps = nullptr;
  int64_t taps_stride = 0;
  at::Tensor before;  // (held: it may come in a list, which another thread may change)
  PyObject *prev = absent(args[3]) ? nullptr : first_of(args[3]);
  if (!absent(prev)) {
    const at::Tensor *t = tensor_of(prev);
    if (!t || wants_gradient(*t) || !taps_of(p, *t, B, taps, taps_stride)) Py_RETURN_NONE;
    before = *t;
  }
  const bool last = args[5] == Py_True;
  if (last && T < p.K - 1) Py_RETURN_NONE;
  c10::OptionalDeviceGuard guard(x_in.device());
  if (!have_word(*p.cell, x_in.device())) Py_RETURN_NONE;
  Sequence s(*p.cell, x_in.device(), B);
  at::Tensor out, tail, state_out;
  {
    WithoutGil no_gil;
    at::Tensor mask;
    if (mask_in) mask = mask_bytes(*mask_in);
    const at::Tensor *maskp = mask_in ? &mask : nullptr;
    const at::Tensor x = p.float32 ? laid_out(x_in) : x_in.contiguous();  // (bf16: a misaligned x is refused, as by the kernels' own entry points)
    void *stream = stream_of(x.device());
    at::Tensor wx = at::empty({B, T, 4 * p.D}, x.options()), x_conv = at::empty({B, T, p.D}, x.options());
    out = x_conv;  // (its last reader has been launched in front of the norm)
    if (p.float32) {
      xs_layer_args a = float32_args(p, x, x_conv, maskp);
      a.conv_state = (const float *)taps; a.conv_state_stride_b = taps && B > 1 ? taps_stride : 0;
      a.wx = (float *)wx.data_ptr();
      launched(g_engine.layer_front(&a));
      s.run(wx, state, maskp, OutShape::SBH);
      a.h = (const float *)s.h.data_ptr(); a.out = (float *)out.data_ptr();
      launched(g_engine.layer_norm(&a));
    } else {
      run_conv(p, x, taps, taps_stride, maskp, x_conv.data_ptr(), nullptr, stream);
      run_gates(p, x, x_conv.data_ptr(), wx.data_ptr(), stream);
      s.run(wx, state, maskp, OutShape::SBH);
      run_norm(p, s.h, B, T, out.data_ptr(), stream);
    }
    if (last) {
      // the last K-1 inputs: a tensor of their own where the call continued a state (x may be reused for the next chunk)
      tail = x_in.narrow(1, T - (p.K - 1), p.K - 1);
      if (taps) tail = tail.clone();
      state_out = p.keep_state || p.float32 ? s.state : s.state.to(at::kBFloat16);
    }
  }
  s.leave();
  PyRef po(THPVariable_Wrap(out));
  if (!po.o) throw PythonError{};
  if (!last) return po.release();
  PyRef pt(THPVariable_Wrap(tail));
  PyRef states(states_dict(pt.o, state_out));
  return PyTuple_Pack(2, po.o, states.o);
}

// ---- training of a float32 layer: one node of the autograd graph for everything between x and the cell's output
struct PythonObject {  // a reference that is given back with the GIL held
  PyObject *o;
  explicit PythonObject(PyObject *p) : o(p) { Py_INCREF(o); }
  ~PythonObject() {
    if (!Py_IsInitialized()) return;
    PyGILState_STATE gil = PyGILState_Ensure();
    Py_DECREF(o);
    PyGILState_Release(gil);
  }
  PythonObject(const PythonObject &) = delete;
  PythonObject &operator=(const PythonObject &) = delete;
};

struct LayerBackward : public torch::autograd::Node {
  // the inputs in the order of the gradients: x, convolution weight and bias, the four gate weights, R, b, state
  enum { X, CONV_W, CONV_B, GATE, R = GATE + 4, BIAS, STATE, INPUTS };
  SavedVariable inputs[INPUTS], x_conv, h, coef;
  bool given[INPUTS] = {};
  std::shared_ptr<Share> share;  // the coefficients'
  ReverseInputs in;  // (its saved tensors are filled in when the backward runs)
  int64_t K = 0;
  at::ScalarType r_dtype = at::kFloat, b_dtype = at::kFloat, s_dtype = at::kFloat;
  std::unique_ptr<PythonObject> recorded_backward;  // (sLSTMLayer._gradients_with_graph, the cell's config)

  std::string name() const override { return "sLSTMLayerBackward"; }
  void release_variables() override {
    std::unique_ptr<PythonObject> last;  // (given back behind the lock: that may run Python code)
    std::lock_guard<std::mutex> lock(mutex_);
    for (SavedVariable &v : inputs) v.reset_data();
    for (SavedVariable *v : {&x_conv, &h, &coef}) v->reset_data();
    in.mask.reset();
    share.reset();
    last = std::move(recorded_backward);
  }

  // A backward that is itself recorded (create_graph): the layer's operations once more, one by one, and their gradients
  variable_list with_graph(PyObject *function_and_config, const at::Tensor (&t)[INPUTS], const ReverseInputs &call, const variable_list &grads) {
    struct Gil { PyGILState_STATE g = PyGILState_Ensure(); ~Gil() { PyGILState_Release(g); } } gil;
    PyRef held(function_and_config);
    auto wrapped = [](const at::Tensor &v) {
      if (v.defined()) return THPVariable_Wrap(v);
      Py_INCREF(Py_None);
      return Py_None;
    };
    PyRef list(PyTuple_New(INPUTS)), d_out(wrapped(grads[0])), d_state(wrapped(grads[1])), mask(wrapped(call.mask));
    PyRef reports(PyCapsule_New(new Reports{call.word, call.calls}, kReports, [](PyObject *o) { delete (Reports *)PyCapsule_GetPointer(o, kReports); }));
    if (list.o)
      for (int i = 0; i < INPUTS; ++i) PyTuple_SET_ITEM(list.o, i, wrapped(t[i]));
    PyRef result(list.o && reports.o && held.o ? PyObject_CallFunctionObjArgs(PyTuple_GET_ITEM(held.o, 0), PyTuple_GET_ITEM(held.o, 1), list.o, mask.o, d_out.o, d_state.o,
                                                                              reports.o, nullptr) : nullptr);
    variable_list out(INPUTS);
    if (!result.o || !PyTuple_Check(result.o) || PyTuple_GET_SIZE(result.o) != INPUTS) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "the gradients of the layer are missing");
      python_error e;
      e.persist();
      throw e;
    }
    for (int i = 0; i < INPUTS; ++i)
      if (const at::Tensor *g = tensor_of(PyTuple_GET_ITEM(result.o, i))) out[i] = *g;
    return out;
  }

  variable_list apply(variable_list &&grads) override {
    at::Tensor t[INPUTS], xc;
    ReverseInputs call;
    PyObject *function_and_config = nullptr;
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (int i = 0; i < INPUTS; ++i)
        if (given[i]) t[i] = inputs[i].unpack();
      call = in;
      call.h = h.unpack(shared_from_this());
      call.coef = coef.unpack();
      xc = x_conv.unpack();
      if (at::GradMode::is_enabled() && recorded_backward) {
        PyGILState_STATE gil = PyGILState_Ensure();
        function_and_config = recorded_backward->o;
        Py_INCREF(function_and_config);
        PyGILState_Release(gil);
      }
    }
    c10::OptionalDeviceGuard guard(call.h.device());
    if (at::GradMode::is_enabled()) return with_graph(function_and_config, t, call, grads);
    at::NoGradGuard no_grad;
    call.h = laid_out(call.h, OutShape::BNSH, call);
    call.coef = laid_out(call.coef);
    xc = laid_out(xc);
    for (int i = CONV_W; i <= R; ++i)
      if (given[i]) t[i] = laid_out(t[i]);
    call.r = t[R];
    if (given[STATE]) call.state = laid_out(t[STATE]);
    const int64_t B = in.B, T = in.T, D = in.NH * in.dh;
    int64_t sb, st;
    const at::Tensor d = output_gradient(call, OutShape::BNSH, grads[0], sb, st);
    CellGradients g = run_reverse(call, d, sb, st, grads[1]);
    const auto f32 = call.h.options();
    const at::Tensor x = laid_out(t[X]);
    LayerParts p;
    p.NH = in.NH; p.dh = in.dh; p.D = D; p.K = K;
    p.conv_w = t[CONV_W]; p.conv_b = t[CONV_B];
    for (int i = 0; i < 4; ++i) p.gate[i] = t[GATE + i];
    xs_layer_args a = float32_args(p, x, xc, call.mask.defined() ? &call.mask : nullptr);
    variable_list out(INPUTS);
    out[R] = g.d_r.to(r_dtype);
    out[BIAS] = g.d_bias.to(b_dtype);
    if (given[STATE]) out[STATE] = g.d_s0.to(s_dtype);
    bool any = false;  // (what is frozen costs nothing)
    for (int i = X; i < R; ++i)
      if (given[i] && task_should_compute_output(i)) {
        out[i] = at::empty(t[i].sizes(), f32);
        any = true;
      }
    if (!any) return out;
    at::Tensor d_x_conv;
    if (out[X].defined() || out[CONV_W].defined() || out[CONV_B].defined()) d_x_conv = at::empty({B, T, D}, f32);
    const at::Tensor scratch = at::empty({(int64_t)g_engine.layer_scratch((int32_t)B, (int32_t)T, (int32_t)in.NH, (int32_t)in.dh, (int32_t)K)}, f32);
    auto ptr = [](const at::Tensor &v) { return v.defined() ? (float *)v.data_ptr() : nullptr; };
    a.scratch = ptr(scratch);
    a.d_wx = ptr(g.d_wx); a.d_x = ptr(out[X]);
    a.d_x_conv = ptr(d_x_conv);
    a.d_conv_w = ptr(out[CONV_W]); a.d_conv_b = ptr(out[CONV_B]);
    for (int i = 0; i < 4; ++i) a.d_gate_w[i] = ptr(out[GATE + i]);
    const int rc = g_engine.layer_front_backward(&a);
    if (rc != XS_OK) engine_failed_in_backward(rc);
    return out;
  }
};

// layer_train(layer, cell path, x, slstm_state, reset_mask, bytes of coefficients that a device may hold) -> (the cell's output,
// state) with their place in the graph, or None.  The caller has looked at the modules (sLSTMLayer._plain_modules)
PyObject *layer_train_(PyObject *const *args) {
  const at::Tensor *xp = tensor_of(args[2]), *state, *mask_in;
  if (!xp || !optional_tensor(args[3], state) || !optional_tensor(args[4], mask_in)) Py_RETURN_NONE;
  const at::Tensor &x_in = *xp;
  LayerParts p;
  if (x_in.dim() != 3 || x_in.size(1) < 2 || x_in.scalar_type() != at::kFloat || !collect(args[0], args[1], x_in, p, true)) Py_RETURN_NONE;
  CellPath &c = *p.cell;
  const int64_t B = x_in.size(0), T = x_in.size(1);
  const at::Tensor *rp, *bp;
  if (!sequence_fits(c, x_in, B, T, state, mask_in) || !g_engine.coef_floats(1, 1, (int32_t)p.NH, (int32_t)p.dh, XS_F32) || !c.weights(rp, bp))
    Py_RETURN_NONE;
  const at::Tensor given[LayerBackward::INPUTS] = {x_in, p.conv_w, p.conv_b, p.gate[0], p.gate[1], p.gate[2], p.gate[3], *rp, *bp, state ? *state : at::Tensor()};
  for (const at::Tensor &t : given)
    if (t.defined() && t._fw_grad(0).defined()) Py_RETURN_NONE;  // (forward mode: the general path refuses it)
  PyRef cut(PyObject_GetAttr(p.cell_config.o, g_names.cut)), clip(PyObject_GetAttr(p.cell_config.o, g_names.clipval));
  if (!cut.o || !clip.o) throw PythonError{};
  const int cut_on = PyObject_IsTrue(cut.o);
  const double clipval = clip.o == Py_None ? 0.0 : PyFloat_AsDouble(clip.o);
  const int64_t limit = PyLong_AsLongLong(args[5]);
  if (PyErr_Occurred()) throw PythonError{};
  c10::OptionalDeviceGuard guard(x_in.device());
  if (!have_word(c, x_in.device())) Py_RETURN_NONE;
  std::shared_ptr<Share> share = Share::take(x_in.device().index(), 4 * (int64_t)g_engine.coef_floats((int32_t)B, (int32_t)T, (int32_t)p.NH, (int32_t)p.dh, XS_F32), limit);
  if (!share) Py_RETURN_NONE;
  Sequence s(c, x_in.device(), B);
  PyRef function(attribute(args[0], g_names.gradients_with_graph)), pair(PyTuple_Pack(2, function.o, p.cell_config.o));
  if (!pair.o) throw PythonError{};
  auto recorded_backward = std::make_unique<PythonObject>(pair.o);
  {
    WithoutGil no_gil;
    at::Tensor x_conv;
    {
      at::NoGradGuard no_grad;
      at::Tensor mask;
      if (mask_in) mask = mask_bytes(*mask_in);
      const at::Tensor *maskp = mask_in ? &mask : nullptr;
      const at::Tensor x = x_in.is_contiguous() && aligned(x_in.data_ptr(), 16) ? x_in.detach() : x_in.clone(at::MemoryFormat::Contiguous);
      const at::Tensor wx = at::empty({B, T, 4 * p.D}, x.options());
      x_conv = at::empty({B, T, p.D}, x.options());
      xs_layer_args a = float32_args(p, x, x_conv, maskp);
      a.wx = (float *)wx.data_ptr();
      launched(g_engine.layer_front(&a));
      s.run(wx, state, maskp, OutShape::BNSH, true);
    }
    auto node = std::shared_ptr<LayerBackward>(new LayerBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(given[0], given[1], given[2], given[3], given[4], given[5], given[6], given[7], given[8], given[9]));
    for (int i = 0; i < LayerBackward::INPUTS; ++i)
      if ((node->given[i] = given[i].defined())) node->inputs[i] = SavedVariable(given[i], false);
    node->x_conv = SavedVariable(x_conv, false);
    node->coef = SavedVariable(s.coef, false);
    node->share = std::move(share);
    node->K = p.K;
    node->r_dtype = rp->scalar_type(); node->b_dtype = bp->scalar_type();
    if (state) node->s_dtype = state->scalar_type();
    node->in.mask = s.mask; node->in.word = s.word; node->in.calls = c.calls;
    node->in.B = B; node->in.T = T; node->in.NH = p.NH; node->in.dh = p.dh;
    node->in.cut = cut_on != 0; node->in.clip = clipval;
    node->recorded_backward = std::move(recorded_backward);
    torch::autograd::set_history(s.h, node);
    torch::autograd::set_history(s.state, node);
    node->h = SavedVariable(s.h, true);
  }
  s.leave();
  PyRef ph(THPVariable_Wrap(s.h)), ps(THPVariable_Wrap(s.state));
  if (!ph.o || !ps.o) throw PythonError{};
  return PyTuple_Pack(2, ph.o, ps.o);
}

template <PyObject *(*F)(PyObject *const *), int N, int OPTIONAL = 0>
PyObject *layer_call(PyObject *, PyObject *const *given, Py_ssize_t n) {
  if (n < N || n > N + OPTIONAL) { PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n); return nullptr; }
  PyObject *args[N + OPTIONAL] = {};  // (what is not given: null)
  std::copy(given, given + n, args);
  if (!PyObject_TypeCheck(args[1], g_cell_type)) Py_RETURN_NONE;
  try {
    return F(args);
  } catch (const PythonError &) {
    return nullptr;
  } catch (const EngineFailed &e) {
    PyErr_SetString(g_engine.error, e.what.c_str());
    return nullptr;
  } catch (...) {  // (out of memory and the like: as the type that torch raises for it)
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

// keep(device, bytes, limit) -> a share of what the device may hold, given back when the object goes, or None beyond the limit
void share_gone(PyObject *capsule) { delete (std::shared_ptr<Share> *)PyCapsule_GetPointer(capsule, "share"); }
PyObject *keep(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 3) { PyErr_SetString(PyExc_TypeError, "keep(device, bytes, limit)"); return nullptr; }
  const long long device = PyLong_AsLongLong(args[0]), bytes = PyLong_AsLongLong(args[1]), limit = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  std::shared_ptr<Share> share = Share::take((int)device, bytes, limit);
  if (!share) Py_RETURN_NONE;
  return PyCapsule_New(new std::shared_ptr<Share>(std::move(share)), "share", share_gone);
}
// kept(device) -> the bytes that are held now
PyObject *kept(PyObject *, PyObject *const *args, Py_ssize_t n) {
  const long long device = n == 1 ? PyLong_AsLongLong(args[0]) : -1;
  if (PyErr_Occurred()) return nullptr;
  if (device < 0 || device >= 64) { PyErr_SetString(PyExc_ValueError, "kept(device)"); return nullptr; }
  return PyLong_FromLongLong(g_kept_bytes[device].load());
}

// bind(addresses: dict name -> int, EngineError, the two dicts of global module hooks)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 4 || !PyDict_Check(args[0])) { PyErr_SetString(PyExc_TypeError, "bind(addresses, error, hooks, pre_hooks)"); return nullptr; }
  auto get = [&](const char *name, auto &fn) {
    PyObject *v = PyDict_GetItemString(args[0], name);
    fn = v ? (std::decay_t<decltype(fn)>)PyLong_AsVoidPtr(v) : nullptr;
    return fn != nullptr;
  };
  if (!get("xs_slstm_step", g_engine.step) || !get("xs_slstm_forward_watched", g_engine.forward) ||
      !get("xs_slstm_workspace_bytes", g_engine.workspace_bytes) || !get("xs_last_error", g_engine.last_error) ||
      !get("xs_causal_conv_silu", g_engine.conv) || !get("xs_causal_conv_silu_token", g_engine.conv_token) || !get("xs_headwise_gates", g_engine.gates) || !get("xs_headwise_group_norm", g_engine.norm) ||
      !get("xs_slstm_train_coef_floats", g_engine.coef_floats) || !get("xs_slstm_train_exchange_bytes", g_engine.exchange_bytes) ||
      !get("xs_slstm_train_forward", g_engine.train_forward) || !get("xs_slstm_train_backward", g_engine.train_backward) ||
      !get("xs_slstm_backward_params", g_engine.backward_params) || !get("xs_layer_front", g_engine.layer_front) ||
      !get("xs_layer_step_fits", g_engine.layer_step_fits) || !get("xs_layer_step", g_engine.layer_step) ||
      !get("xs_layer_norm", g_engine.layer_norm) || !get("xs_layer_scratch_floats", g_engine.layer_scratch) ||
      !get("xs_layer_front_backward", g_engine.layer_front_backward)) {
    PyErr_SetString(PyExc_KeyError, "an entry point of the engine is missing");
    return nullptr;
  }
  // (whoever binds other entry points for the parts of a layer's step that the one kernel stands for, to watch them or to stand in for
  // them, has them called; the norm behind it is called either way)
  static const Engine first = g_engine;
  g_engine.own_parts = g_engine.step == first.step && g_engine.conv == first.conv && g_engine.gates == first.gates;
  for (int i = 1; i < 4; ++i) Py_INCREF(args[i]);
  g_engine.error = args[1];
  for (int i = 0; i < 2; ++i) g_engine.global_hooks[i] = PyDict_Check(args[2 + i]) ? args[2 + i] : nullptr;
  Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {
    {"bind", (PyCFunction)(void *)bind, METH_FASTCALL, nullptr},
    {"keep", (PyCFunction)(void *)keep, METH_FASTCALL, nullptr},
    {"kept", (PyCFunction)(void *)kept, METH_FASTCALL, nullptr},
    {"layer_step", (PyCFunction)(void *)layer_call<layer_step_, 10, 1>, METH_FASTCALL, nullptr},
    {"layer_forward", (PyCFunction)(void *)layer_call<layer_forward_, 7>, METH_FASTCALL, nullptr},
    {"layer_train", (PyCFunction)(void *)layer_call<layer_train_, 6>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_xlstm_host", "native host path of the cell's and the layer's frequent calls", -1, module_methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__xlstm_host(void) {
  auto s = [](const char *v) { return PyUnicode_InternFromString(v); };
  g_names = Names{s("_recurrent_kernel_"), s("_bias_"), s("weight"), s("bias"), s("conv_state"), s("slstm_state"), s("input_shape"), s("output_shape"),
                  s("keep_state_fp32"), s("config"), s("_modules"), s("_parameters"), s("_forward_hooks"), s("_forward_pre_hooks"), s("training"), s("p"),
                  s("eps"), s("conv1d"), s("conv"), s("fgate"), s("igate"), s("zgate"), s("ogate"), s("group_norm"), s("slstm_cell"), s("dropout"),
                  s("fused_pre_ops"), s("BSGNH"), s("gradient_recurrent_cut"), s("gradient_recurrent_clipval"), s("_gradients_with_graph")};
  PyObject *m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  g_cell_type = (PyTypeObject *)PyType_FromSpec(&cell_spec);
  if (!g_cell_type || PyModule_AddObject(m, "CellPath", (PyObject *)g_cell_type)) return nullptr;
  Py_INCREF(g_cell_type);
  return m;
}
