// Host side of the Buffer operators and of the expert FFN: argument checks, output allocation and launches of one
// call in native code (module moonep_amd._host).
//
// An operator of a small batch is bound by the host: through Python and ctypes a decode step
// (8 tokens, dispatch + combine) took 63 us for 22 us of GPU work -- nine allocations, fifteen
// shape checks and four launches, a microsecond or more each.  Here a plan's eight tensors take four
// allocations past the dispatcher, and the checks cost nanoseconds.
//
// Every function returns None, with nothing launched, when the call is not the plain case it
// handles (a failed check, a world with host threads, ...): the Python body of the operator
// then runs and raises what it always raised, or does the rarer work.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <initializer_list>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/moonep_hip.h"

namespace {

struct Names {
  PyObject *dst, *etc, *zfr, *stats, *dup_groups, *dup_loffs, *dup_counts, *N, *R, *E, *NvS, *K, *no_map, *record;
} nm;

// what a Buffer keeps from one call to the next
struct Ctx {
  int S, H, K, E, R, epn, NvS, rank, tp;
  int64_t N, wslot_stride;
  at::Tensor hidden_buf, meta_buf, hidden_local, weights_local, scratch;
  c10::Stream comm = c10::Stream(c10::Stream::UNSAFE, c10::Device(c10::kCPU), 0);
  hipStream_t comm_raw = nullptr;
  hipEvent_t order = nullptr;
  // A call's ordering and its launches belong together.  comm_used: something may be on the communication stream.
  // coming: callers of comes_to_comm whose work is not all there.  beside_open: the last asynchronous call that stayed on its
  // caller's stream, beside_on, until the communication stream is ordered behind it; beside, where it is recorded
  // (beside_kept), lies behind that call.  several: such calls came from more than one stream.
  std::mutex order_mutex;
  bool comm_used = false, beside_open = false, beside_kept = false, several = false;
  int coming = 0;
  hipEvent_t beside = nullptr;
  hipStream_t beside_on = nullptr;
  hipError_t keep_beside() {
    hipError_t e = beside ? hipSuccess : hipEventCreateWithFlags(&beside, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(beside, beside_on);
    beside_kept = e == hipSuccess;
    return e;
  }
  PyObject *plan_type = nullptr, *hidden_local_py = nullptr, *no_map_token = nullptr, *event_type = nullptr,
           *comm_py = nullptr, *empty = nullptr;
  PyObject *current_stream = nullptr, *caller_py = nullptr;  // torch's function; what it answered for the stream caller_id
  c10::StreamId caller_id = 0;
  PyObject *py_N = nullptr, *py_R = nullptr, *py_E = nullptr, *py_NvS = nullptr, *py_K = nullptr;
  ~Ctx() {
    for (PyObject* o : {plan_type, hidden_local_py, no_map_token, event_type, comm_py, empty, py_N, py_R, py_E,
                        py_NvS, py_K, current_stream, caller_py})
      Py_XDECREF(o);
    if (order) (void)hipEventDestroy(order);
    if (beside) (void)hipEventDestroy(beside);
  }
};

const char* kCapsule = "moonep_amd._host.Ctx";

void free_ctx(PyObject* cap) { delete (Ctx*)PyCapsule_GetPointer(cap, kCapsule); }

Ctx* ctx_of(PyObject* cap) { return (Ctx*)PyCapsule_GetPointer(cap, kCapsule); }

// the C ABI's return code as the exception the Python binding raises
bool failed(int rc, const char* what) {
  if (rc == 0) return false;
  PyErr_Format(PyExc_RuntimeError, "%s failed: %s (code %d)", what, mep_strerror(rc), rc);
  return true;
}

const char* const kOrdering = "ordering the communication stream";

const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

bool is(const at::Tensor& t, at::ScalarType dt, const Ctx& c) {
  return t.scalar_type() == dt && t.device() == c.hidden_buf.device() && t.is_contiguous();
}

bool shape(const at::Tensor& t, std::initializer_list<int64_t> s) {
  return t.sizes() == c10::IntArrayRef(s.begin(), s.size());
}

bool aligned(const void* p) { return ((uintptr_t)p & 15) == 0; }

// a dense tensor of `sizes` at element `offset` of a storage
at::Tensor view_of(const at::Tensor& base, caffe2::TypeMeta dtype, int64_t offset, c10::IntArrayRef sizes) {
  at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(base.storage()), base.key_set(), dtype);
  c10::TensorImpl* impl = t.unsafeGetTensorImpl();
  impl->set_storage_offset(offset);
  impl->set_sizes_contiguous(sizes);
  return t;
}

PyObject* new_none() { Py_RETURN_NONE; }

// Other Python threads run meanwhile: an allocation may wait for the device and a launch for a place
// in a full queue.  Nothing of Python may be touched inside.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// hipErrorNotReady is an answer: nobody is to find it as the last error
hipError_t asked(hipError_t e) {
  if (e == hipErrorNotReady) (void)hipGetLastError();
  return e;
}

// Queries while another thread captures a stream, in whatever mode
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// The most that an asynchronous call moves and stays on its caller's stream.  A crossing to the communication
// stream and back takes 22 us of the GPU, and on the host some 40 a call: an event's record and the wait of
// another stream for it, 16 us while the event has not come, and a record for every tensor that is freed after use on a
// stream that is not its own.  Up to this size the call itself is no longer than the crossing.  us a pass of dispatch and
// combine, each waited for, H = 2048, K = 8, on the communication stream -> on the caller's, the default one, alone and with a
// product of 60, 115 and 370 us of the caller's own behind each call, which the communication stream works beside: 8 tokens
// 102 -> 30, 160 -> 131, 205 -> 204, 642 -> 643; 512 97 -> 29, 153 -> 135, 207 -> 208, 655 -> 651; 1536 (48 MiB of copies) 100 -> 36, 158 ->
// 148, 223 -> 223, 670 -> 663; H = 7168 the same.  From another stream, whose calls record an event each: 8 tokens alone 36, with the
// products 137, 211 and 649.  Synchronous calls alone: 8 tokens 16, 512 21, 1536 29.
constexpr int64_t kBeside = (int64_t)64 << 20;

// ---- asynchronous calls: the work goes to the communication stream, small calls' while that is idle to the caller's
struct Async {
  Ctx& c;
  bool on, here = false, ordered = false;
  hipStream_t stream;
  std::unique_lock<std::mutex> lock;
  // moved: bytes that the call reads or writes, whichever is more
  Async(Ctx& ctx, bool async, int64_t moved = INT64_MAX) : c(ctx), on(async) {
    if (on && !c.comm_raw) {  // asked for by the first asynchronous call: the answer makes the stream exist
      PyObject* o = PyObject_GetAttrString(c.comm_py, "cuda_stream");
      c.comm_raw = o ? (hipStream_t)PyLong_AsVoidPtr(o) : nullptr;
      Py_XDECREF(o);
      if (PyErr_Occurred()) throw python_error();
    }
    here = on && moved <= kBeside && !external();
    stream = on ? c.comm_raw : callers();
  }
  // A stream that torch did not make (its id is its handle) may end before the memory that is recorded on it, which the
  // allocator then still touches it for, and before the calls that are to come behind its own: another of the
  // same handle may have taken its place.  Nothing is kept by it.
  bool external() const {
    const c10::hip::HIPStream s = c10::hip::getCurrentHIPStream(c.hidden_buf.device().index());
    return s.stream() && s.id() == (c10::StreamId)(intptr_t)s.stream();
  }
  hipStream_t callers() const { return c10::hip::getCurrentHIPStream(c.hidden_buf.device().index()).stream(); }
  // `on_stream` behind the last call that stayed on its caller's stream
  static hipError_t behind(Ctx& c, hipStream_t on_stream) {
    if (!c.beside_open || c.beside_on == on_stream) return hipSuccess;
    const RelaxedCapture relaxed;
    hipError_t e = hipSuccess;
    if (!c.beside_kept) {
      c.several = true;
      if ((e = c.keep_beside()) != hipSuccess) return e;
    }
    e = asked(hipEventQuery(c.beside));
    return e == hipErrorNotReady ? hipStreamWaitEvent(on_stream, c.beside, 0) : e;
  }
  // after the caller's work; the allocator must not reuse what the stream still works on
  int begin(std::initializer_list<const at::Tensor*> used) {
    if (!on) return MEP_OK;
    hipStream_t main = callers();
    lock = std::unique_lock<std::mutex>(c.order_mutex);
    if (here && c.coming) here = false;  // the stream may be idle until another thread's launches
    if (here && c.comm_used) {
      const RelaxedCapture relaxed;
      const hipError_t e = asked(hipStreamQuery(c.comm_raw));
      if (e != hipSuccess && e != hipErrorNotReady) return (int)e;
      here = e == hipSuccess;
      c.comm_used = !here;
    }
    // on the caller's stream, too: a tensor may have been allocated on another (one of the same costs a look-up)
    const c10::StreamId callers_id = c10::hip::getCurrentHIPStream(c.hidden_buf.device().index()).id();
    const c10::Stream user = here ? c10::Stream(c10::Stream::UNSAFE, c.comm.device(), callers_id) : c.comm;
    const c10::StorageImpl* seen[24];
    int n = 0;
    for (const at::Tensor* t : used) {
      if (!t || !t->defined()) continue;
      const c10::StorageImpl* s = t->storage().unsafeGetStorageImpl();
      bool dup = false;
      for (int i = 0; i < n; ++i) dup |= seen[i] == s;
      if (dup) continue;
      if (n < 24) seen[n++] = s;
      t->record_stream(user);
    }
    if (here) {
      stream = main;
      const hipError_t e = behind(c, main);
      ordered = e == hipSuccess;
      return (int)e;
    }
    c.comm_used = true;
    hipError_t e = c.order ? hipSuccess : hipEventCreateWithFlags(&c.order, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(c.order, main);
    if (e == hipSuccess) e = hipStreamWaitEvent(c.comm_raw, c.order, 0);
    if (e == hipSuccess && c.beside_on != main) e = behind(c, c.comm_raw);
    if (e == hipSuccess) c.beside_open = false;
    return (int)e;
  }
  // the call's work is on its stream, or the part of it in front of the launch that failed
  int launched(int rc) {
    if (here && ordered) {
      c.beside_on = stream;
      c.beside_kept = false;
      // The default stream is there as long as the process and never under capture: behind its calls the event may be
      // recorded when a call of another stream asks, for the first time then, since the later the more lies in front of it.
      // (A record takes 4.5 us of the stream.)
      const hipError_t e = !stream && !c.several ? hipSuccess : c.keep_beside();
      c.beside_open = e == hipSuccess;
      if (rc == MEP_OK) rc = (int)e;
    }
    if (lock.owns_lock()) lock.unlock();
    return rc;
  }
  // the caller's stream as a Python object (4 us when torch makes a new one for every event)
  PyObject* caller() {
    const c10::hip::HIPStream s = c10::hip::getCurrentHIPStream(c.hidden_buf.device().index());
    if (!c.caller_py || c.caller_id != s.id()) {
      PyObject* o = PyObject_CallFunction(c.current_stream, "i", (int)s.device_index());
      if (!o) return nullptr;
      Py_XSETREF(c.caller_py, o);
      c.caller_id = s.id();
    }
    return c.caller_py;
  }
  // a new reference to the completion event
  PyObject* end() {
    PyObject* ev = PyObject_CallNoArgs(c.event_type);
    if (!ev) return nullptr;
    PyObject* on_stream = here ? caller() : c.comm_py;
    PyObject* r = on_stream ? PyObject_CallMethodOneArg(ev, nm.record, on_stream) : nullptr;
    if (!r) { Py_DECREF(ev); return nullptr; }
    Py_DECREF(r);
    return ev;
  }
};

// an ordering event is shared by a Buffer's calls: under stream capture the Python body makes its own
bool capturing(const Ctx& c) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  hipStream_t s = c10::hip::getCurrentHIPStream(c.hidden_buf.device().index()).stream();
  return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

// ---- plans -------------------------------------------------------------------------------
struct Plan {
  at::Tensor dst, etc, zfr, stats, dup_groups, dup_loffs, dup_counts;
};

const at::Tensor* attr_tensor(PyObject* plan, PyObject* name, std::vector<PyObject*>& hold) {
  PyObject* o = PyObject_GetAttr(plan, name);
  if (!o) { PyErr_Clear(); return nullptr; }
  hold.push_back(o);
  return tensor(o);
}

bool attr_is(PyObject* plan, PyObject* name, int64_t want) {
  PyObject* o = PyObject_GetAttr(plan, name);
  if (!o) { PyErr_Clear(); return false; }
  const long long v = PyLong_Check(o) ? PyLong_AsLongLong(o) : -1;
  Py_DECREF(o);
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  return v == want;
}

// the tensors of a caller's plan, checked as a dispatch checks them; false: let Python look
bool read_plan(const Ctx& c, PyObject* plan, Plan* p) {
  if ((PyObject*)Py_TYPE(plan) != c.plan_type) return false;
  if (!attr_is(plan, nm.N, c.N) || !attr_is(plan, nm.R, c.R) || !attr_is(plan, nm.K, c.K) ||
      !attr_is(plan, nm.NvS, c.NvS))
    return false;
  std::vector<PyObject*> hold;
  hold.reserve(8);
  const at::Tensor* t[7];
  PyObject* names[7] = {nm.dst, nm.etc, nm.zfr, nm.stats, nm.dup_groups, nm.dup_loffs, nm.dup_counts};
  bool ok = true;
  for (int i = 0; i < 7; ++i) {
    t[i] = attr_tensor(plan, names[i], hold);
    ok = ok && t[i] && is(*t[i], at::kInt, c);
  }
  ok = ok && shape(*t[0], {c.N}) && shape(*t[1], {c.R, c.epn}) && shape(*t[2], {2 * c.epn, 2}) &&
       shape(*t[3], {2}) && shape(*t[4], {c.NvS, 3}) && shape(*t[5], {c.NvS}) && shape(*t[6], {2});
  if (ok) *p = Plan{*t[0], *t[1], *t[2], *t[3], *t[4], *t[5], *t[6]};
  for (PyObject* o : hold) Py_DECREF(o);
  return ok;
}

// a MoonEPCommPlan whose tensors are already known to be right (its __post_init__ checks nothing new)
PyObject* wrap_plan(const Ctx& c, const Plan& p) {
  PyTypeObject* type = (PyTypeObject*)c.plan_type;
  PyObject* plan = type->tp_new(type, c.empty, nullptr);
  if (!plan) return nullptr;
  auto set = [&](PyObject* name, PyObject* value, bool own) {  // the slots themselves: the class is frozen
    const int rc = value ? PyObject_GenericSetAttr(plan, name, value) : -1;
    if (own) Py_XDECREF(value);
    return rc == 0;
  };
  PyObject* counts = THPVariable_Wrap(p.dup_counts);
  bool ok = counts != nullptr;
  // the other ranks' routing is unknown: the plan has no duplicate map of this world
  if (ok && c.R > 1) ok = PyObject_SetAttr(counts, nm.no_map, c.no_map_token) == 0;
  ok = ok && set(nm.dst, THPVariable_Wrap(p.dst), true) && set(nm.etc, THPVariable_Wrap(p.etc), true) &&
       set(nm.zfr, THPVariable_Wrap(p.zfr), true) && set(nm.stats, THPVariable_Wrap(p.stats), true) &&
       set(nm.dup_groups, THPVariable_Wrap(p.dup_groups), true) &&
       set(nm.dup_loffs, THPVariable_Wrap(p.dup_loffs), true) && set(nm.dup_counts, counts, false) &&
       set(nm.N, c.py_N, false) && set(nm.R, c.py_R, false) && set(nm.E, c.py_E, false) &&
       set(nm.NvS, c.py_NvS, false) && set(nm.K, c.py_K, false);
  Py_XDECREF(counts);
  if (!ok) { Py_DECREF(plan); return nullptr; }
  return plan;
}

// A dense tensor of its own from the allocator that meta_buf came from, past the dispatcher (a call
// of it 1.4 us, this 0.7: dispatch + combine of 8 tokens, host time 12.6 -> 11.8 us).
struct New {
  const at::Tensor& like;
  c10::Allocator* from;
  explicit New(const Ctx& c) : like(c.meta_buf), from(c.meta_buf.storage().allocator()) {
    // at::empty looks after the device, and after what a tensor of an inference mode may be used for
    if (c10::hip::current_device() != like.device().index() || like.is_inference() || c10::InferenceMode::is_enabled())
      from = nullptr;
  }
  at::Tensor operator()(at::ScalarType type, std::initializer_list<int64_t> s) const {
    const c10::IntArrayRef sizes(s.begin(), s.size());
    if (!from) return at::empty(sizes, like.options().dtype(type));
    const caffe2::TypeMeta dtype = c10::scalarTypeToTypeMeta(type);
    const size_t bytes = (size_t)c10::multiply_integers(sizes) * dtype.itemsize();
    at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(
        c10::Storage(c10::make_intrusive<c10::StorageImpl>(c10::StorageImpl::use_byte_size_t(), bytes, from->allocate(bytes),
                                                           from, /*resizable=*/true)),
        like.key_set(), dtype);
    t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
    return t;
  }
  at::Tensor operator()(std::initializer_list<int64_t> s) const { return (*this)(at::kInt, s); }
};

// A fresh plan and its cu_seqlens.  The small tensors are views of one block of a few KB (64-byte
// starts), those that grow with the tokens own their memory, so that what a caller keeps holds
// nothing large besides.  (Dispatch + combine of 8 tokens, host time: all eight in one block 16.9 us, so 17.5, each
// on its own 18.2.)
void new_plan(const Ctx& c, const New& make, Plan* p, at::Tensor* cu) {
  int64_t at_int = 0;
  auto take = [&](int64_t n) { const int64_t o = at_int; at_int += (n + 15) & ~(int64_t)15; return o; };
  const int64_t o_cu = take(2 * c.epn), o_etc = take((int64_t)c.R * c.epn), o_zfr = take(4 * c.epn), o_stats = take(2),
                o_counts = take(2);
  const at::Tensor block = make({at_int});
  auto v = [&](int64_t o, std::initializer_list<int64_t> s) {
    return view_of(block, block.dtype(), o, c10::IntArrayRef(s.begin(), s.size()));
  };
  *p = Plan{make({c.N}), v(o_etc, {c.R, c.epn}), v(o_zfr, {2 * c.epn, 2}), v(o_stats, {2}), make({c.NvS, 3}),
            make({c.NvS}), v(o_counts, {2})};
  *cu = v(o_cu, {2 * c.epn});
}

template <class T>
T* ptr(const at::Tensor& t) { return t.defined() ? (T*)t.data_ptr() : nullptr; }

// ---- dispatch(ctx, hidden, weights, topk, tpe, plan, async, zero_copy, weights_zero_copy) ----
PyObject* py_dispatch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) { PyErr_SetString(PyExc_TypeError, "dispatch takes 9 arguments"); return nullptr; }
  Ctx* cp = ctx_of(args[0]);
  if (!cp) return nullptr;
  Ctx& c = *cp;
  const at::Tensor* hidden = tensor(args[1]);
  const at::Tensor* w = args[2] == Py_None ? nullptr : tensor(args[2]);
  if (!hidden || !is(*hidden, at::kBFloat16, c) || !shape(*hidden, {c.S, c.H}) || !aligned(hidden->data_ptr()))
    return new_none();
  if (args[2] != Py_None && (!w || !is(*w, at::kFloat, c) || !shape(*w, {c.S, c.K}))) return new_none();
  const bool async = args[6] == Py_True, zero_copy = args[7] == Py_True, w_zero_copy = args[8] == Py_True;
  if (async && capturing(c)) return new_none();
  const bool fresh = args[5] == Py_None;
  const at::Tensor *topk = nullptr, *tpe = nullptr;
  Plan plan;
  at::Tensor cu;
  if (fresh) {
    topk = tensor(args[3]);
    tpe = tensor(args[4]);
    if (!topk || !is(*topk, at::kInt, c) || topk->dim() == 3 || topk->numel() != c.N) return new_none();
    if (!tpe || !is(*tpe, at::kInt, c) || tpe->dim() != 2 || !shape(*tpe, {c.R, c.E})) return new_none();
  } else if (!read_plan(c, args[5], &plan)) {
    return new_none();
  }
  const int64_t row = (int64_t)c.H * 2, padded = std::min((int64_t)c.NvS, c.N + 2 * c.epn * (int64_t)(c.tp - 1));
  Async as(c, async, padded * row + (zero_copy ? 0 : c.NvS * row));
  at::Tensor out, w_out;
  const char* what = kOrdering;
  int rc;
  {
    NoGil other_threads;
    const New make(c);
    if (fresh) new_plan(c, make, &plan, &cu);
    out = zero_copy ? c.hidden_local : make(at::kBFloat16, {c.NvS, c.H});
    at::Tensor w_local = view_of(c.weights_local, caffe2::TypeMeta::Make<float>(), c.weights_local.storage_offset(), {c.NvS});
    if (w) w_out = w_zero_copy ? w_local : make(at::kFloat, {c.NvS});
    rc = as.begin({hidden, w, &out, &w_out, &plan.dst, &plan.etc, &plan.zfr, &plan.stats, &plan.dup_groups,
                   &plan.dup_loffs, &plan.dup_counts, topk, tpe, &cu});
    if (rc == MEP_OK && fresh && !async) {
      what = "mep_dispatch_fresh";
      rc = mep_dispatch_fresh(ptr<int>(*tpe), ptr<int>(*topk), hidden->data_ptr(), w ? ptr<float>(*w) : nullptr, c.rank, c.S,
                              c.H, c.K, c.E, c.R, c.tp, c.NvS, ptr<int>(plan.dst), ptr<int>(cu), ptr<int>(plan.etc),
                              ptr<int>(plan.zfr), ptr<int>(plan.stats), ptr<int>(plan.dup_counts),
                              c.hidden_buf.data_ptr(), c.NvS, w ? ptr<float>(c.meta_buf) : nullptr, c.wslot_stride,
                              ptr<void>(c.scratch), c.scratch.defined() ? c.scratch.nbytes() : 0, as.stream);
    } else if (rc == MEP_OK) {
      // what is on the communication stream runs beside kernels that hold CUs, GEMMs all of them: two launches even of a
      // small call (has_all_cus in planner.hip has the figures), and the same two where it stays on its caller's
      // stream (one there: 8 tokens 30 -> 27 us a pass)
      what = "mep_plan";
      if (fresh)
        rc = mep_plan_fresh(ptr<int>(*tpe), ptr<int>(*topk), c.rank, c.S, c.K, c.E, c.R, c.tp, c.NvS,
                            ptr<int>(plan.dst), ptr<int>(cu), ptr<int>(plan.etc), ptr<int>(plan.zfr),
                            ptr<int>(plan.stats), ptr<int>(plan.dup_counts), ptr<void>(c.scratch),
                            c.scratch.defined() ? c.scratch.nbytes() : 0, hidden->data_ptr(), hidden->nbytes(), as.stream);
    }
    if (rc == MEP_OK && !(fresh && !async)) {
      what = "mep_dispatch";
      rc = mep_dispatch(hidden->data_ptr(), w ? ptr<float>(*w) : nullptr, ptr<int>(plan.dst), ptr<int>(plan.zfr),
                        c.hidden_buf.data_ptr(), c.NvS, w ? ptr<float>(c.meta_buf) : nullptr, c.wslot_stride,
                        c.rank, c.S, c.H, c.K, c.R, c.epn, c.NvS, c.tp, MEP_DISPATCH_WRITE_DUPS, as.stream);
    }
    const bool copy_w = w && !w_zero_copy;
    if (rc == MEP_OK && (!zero_copy || copy_w)) {
      what = "mep_copy_shard";
      rc = mep_copy_shard(zero_copy ? nullptr : out.data_ptr(), zero_copy ? nullptr : c.hidden_local.data_ptr(),
                          zero_copy ? 0 : out.nbytes(), copy_w ? w_out.data_ptr() : nullptr,
                          copy_w ? w_local.data_ptr() : nullptr, copy_w ? (size_t)c.NvS : 0, as.stream);
    }
    rc = as.launched(rc);
  }
  if (failed(rc, what)) return nullptr;
  PyObject* event = nullptr;
  if (async && !(event = as.end())) return nullptr;
  PyObject* res = PyTuple_New(async ? 5 : 4);
  PyObject* py_out;
  if (zero_copy) { py_out = c.hidden_local_py; Py_INCREF(py_out); }
  else py_out = THPVariable_Wrap(out);
  PyObject* py_plan;
  if (fresh) py_plan = wrap_plan(c, plan);
  else { py_plan = args[5]; Py_INCREF(py_plan); }
  if (!res || !py_out || !py_plan) { Py_XDECREF(res); Py_XDECREF(py_out); Py_XDECREF(py_plan); Py_XDECREF(event); return nullptr; }
  PyTuple_SET_ITEM(res, 0, py_out);
  PyTuple_SET_ITEM(res, 1, w ? THPVariable_Wrap(w_out) : new_none());
  PyTuple_SET_ITEM(res, 2, fresh ? THPVariable_Wrap(cu) : new_none());
  PyTuple_SET_ITEM(res, 3, py_plan);
  if (async) PyTuple_SET_ITEM(res, 4, event);
  return res;
  END_HANDLE_TH_ERRORS
}

// ---- combine(ctx, plan, hidden, weights, async, zero_copy, weights_zero_copy) ----------------
PyObject* py_combine(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) { PyErr_SetString(PyExc_TypeError, "combine takes 7 arguments"); return nullptr; }
  Ctx* cp = ctx_of(args[0]);
  if (!cp) return nullptr;
  Ctx& c = *cp;
  Plan plan;
  const at::Tensor* hidden = tensor(args[2]);
  const at::Tensor* w = args[3] == Py_None ? nullptr : tensor(args[3]);
  if (!read_plan(c, args[1], &plan)) return new_none();
  if (!hidden || !is(*hidden, at::kBFloat16, c) || !shape(*hidden, {c.NvS, c.H}) || !aligned(hidden->data_ptr()))
    return new_none();
  if (args[3] != Py_None && (!w || !is(*w, at::kFloat, c) || !shape(*w, {c.NvS}))) return new_none();
  const bool async = args[4] == Py_True, zero_copy = args[5] == Py_True, w_zero_copy = args[6] == Py_True;
  const bool copy_h = hidden->data_ptr() != c.hidden_local.data_ptr();
  const bool copy_w = w && w->data_ptr() != c.weights_local.data_ptr();
  if ((zero_copy && copy_h) || (w_zero_copy && copy_w)) return new_none();
  if (async && capturing(c)) return new_none();
  Async as(c, async, (c.N + (copy_h ? c.NvS : 0)) * (int64_t)c.H * 2);  // what it reads is more than what it writes
  at::Tensor out, out_w;
  const char* what = kOrdering;
  int rc;
  {
    NoGil other_threads;
    const New make(c);
    out = make(at::kBFloat16, {c.S, c.H});
    if (w) out_w = make(at::kFloat, {c.S, c.K});
    rc = as.begin({&out, &plan.dst, &plan.etc, &plan.zfr, &plan.stats, &plan.dup_groups, &plan.dup_loffs,
                   &plan.dup_counts, hidden, w, &out_w});
    if (rc == MEP_OK && (copy_h || copy_w)) {
      what = "mep_copy_shard";
      rc = mep_copy_shard(copy_h ? c.hidden_local.data_ptr() : nullptr, copy_h ? hidden->data_ptr() : nullptr,
                          copy_h ? hidden->nbytes() : 0, copy_w ? c.weights_local.data_ptr() : nullptr,
                          copy_w ? w->data_ptr() : nullptr, copy_w ? (size_t)c.NvS : 0, as.stream);
    }
    if (rc == MEP_OK) {
      what = "mep_combine";
      rc = mep_combine(c.hidden_buf.data_ptr(), c.NvS, w ? ptr<float>(c.meta_buf) : nullptr, c.wslot_stride,
                       ptr<int>(plan.dst), out.data_ptr(), w ? ptr<float>(out_w) : nullptr, c.S, c.H, c.K, c.R, c.NvS,
                       MEP_COMBINE_TWO_LEVEL, as.stream);
    }
    rc = as.launched(rc);
  }
  if (failed(rc, what)) return nullptr;
  PyObject* event = async ? as.end() : new_none();
  if (!event) return nullptr;
  PyObject* res = PyTuple_New(3);
  if (!res) { Py_DECREF(event); return nullptr; }
  PyTuple_SET_ITEM(res, 0, THPVariable_Wrap(out));
  PyTuple_SET_ITEM(res, 1, w ? THPVariable_Wrap(out_w) : new_none());
  PyTuple_SET_ITEM(res, 2, event);
  return res;
  END_HANDLE_TH_ERRORS
}

// ---- weights and gradients: (this rank's tensor, all-rank pool) pairs ------------------------
// dense [epn, ...] and [R, epn, ...], blocks of the pool 16-byte aligned and inside the storage
bool pair_ok(const Ctx& c, const at::Tensor* local, const at::Tensor* pool) {
  if (!local || !pool || local->device() != c.hidden_buf.device() || pool->device() != c.hidden_buf.device())
    return false;
  const int64_t d = local->dim();
  if (d < 2 || local->scalar_type() != pool->scalar_type() || !local->is_contiguous() || pool->dim() != d + 1)
    return false;
  if (local->size(0) != c.epn || pool->size(0) != c.R) return false;
  int64_t dense = 1;
  for (int64_t i = d; i >= 1; --i) {
    if (pool->size(i) != local->size(i - 1) || pool->stride(i) != dense) return false;
    dense *= pool->size(i);
  }
  const int64_t width = pool->element_size(), stride = pool->stride(0);
  if (dense <= 0 || stride < dense || (stride * width) % 16 != 0 || stride * width >= ((int64_t)1 << 40)) return false;
  if (!aligned(pool->data_ptr()) || !aligned(local->data_ptr())) return false;
  return (pool->storage_offset() + stride * (c.R - 1) + dense) * width <= (int64_t)pool->storage().nbytes();
}

bool matrix_ok(const at::Tensor& t) { return t.dim() == 3 && t.size(1) % 128 == 0 && t.size(2) % 128 == 0; }

// plan.experts_to_copy, or undefined
at::Tensor slot_table(const Ctx& c, PyObject* plan) {
  at::Tensor etc;
  if ((PyObject*)Py_TYPE(plan) != c.plan_type) return etc;
  PyObject* o = PyObject_GetAttr(plan, nm.etc);
  if (!o) { PyErr_Clear(); return etc; }
  const at::Tensor* t = tensor(o);
  if (t && is(*t, at::kInt, c) && shape(*t, {c.R, c.epn})) etc = *t;
  Py_DECREF(o);
  return etc;
}

// prefetch(ctx, plan, async, 3 x local, 3 x pool, 3 x local scale, 3 x scale pool) -> True | event
PyObject* py_prefetch(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15) { PyErr_SetString(PyExc_TypeError, "prefetch takes 15 arguments"); return nullptr; }
  Ctx* cp = ctx_of(args[0]);
  if (!cp) return nullptr;
  Ctx& c = *cp;
  const bool async = args[2] == Py_True;
  at::Tensor etc = slot_table(c, args[1]);
  if (!etc.defined() || (async && capturing(c))) return new_none();
  const void* src[6];
  void* dst[6];
  int64_t stride[6], bytes[6];
  const at::Tensor* t[12] = {};
  int given = 0;
  for (int i = 9; i < 15; ++i) given += args[i] != Py_None;
  if (given != 0 && given != 6) return new_none();
  const int m = given ? 6 : 3;
  for (int i = 0; i < m; ++i) {
    const bool scale = i >= 3;
    const at::Tensor* l = tensor(args[(scale ? 9 : 3) + i % 3]);
    const at::Tensor* p = tensor(args[(scale ? 12 : 6) + i % 3]);
    if (!pair_ok(c, l, p)) return new_none();
    const at::ScalarType dt = l->scalar_type();
    if (!scale) {
      if (!matrix_ok(*l)) return new_none();
      if (dt != at::kBFloat16 && dt != at::kChar && dt != at::kByte) return new_none();
      if (i > 0 && dt != t[0]->scalar_type()) return new_none();
      if (given && dt != at::kByte) return new_none();
    } else if (dt != at::kByte) {
      return new_none();
    }
    t[i] = l; t[6 + i] = p;
    src[i] = l->data_ptr(); dst[i] = p->data_ptr();
    stride[i] = p->stride(0) * p->element_size();
    bytes[i] = (int64_t)(l->nbytes() / c.epn);
    if (scale && bytes[i] % (128 * 128) != 0) return new_none();
  }
  Async as(c, async);
  const char* what = kOrdering;
  int rc;
  {
    NoGil other_threads;
    rc = as.begin({&etc, t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], t[9], t[10], t[11]});
    if (rc == MEP_OK) {
      what = "mep_prefetch";
      rc = mep_prefetch(m, src, dst, stride, bytes, ptr<int>(etc), c.rank, c.epn, c.R, as.stream);
    }
    rc = as.launched(rc);
  }
  if (failed(rc, what)) return nullptr;
  if (async) return as.end();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// reduce_grad(ctx, plan, async, 3 x local, 3 x pool) -> True | event
PyObject* py_reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) { PyErr_SetString(PyExc_TypeError, "reduce_grad takes 9 arguments"); return nullptr; }
  Ctx* cp = ctx_of(args[0]);
  if (!cp) return nullptr;
  Ctx& c = *cp;
  const bool async = args[2] == Py_True;
  at::Tensor etc = slot_table(c, args[1]);
  if (!etc.defined() || (async && capturing(c))) return new_none();
  const at::Tensor *l[3], *p[3];
  for (int i = 0; i < 3; ++i) {
    l[i] = tensor(args[3 + i]);
    p[i] = tensor(args[6 + i]);
    if (!pair_ok(c, l[i], p[i]) || l[i]->scalar_type() != at::kFloat || !matrix_ok(*l[i])) return new_none();
  }
  Async as(c, async);
  float *lp[3], *pp[3];
  int64_t stride[3], elems[3];
  for (int i = 0; i < 3; ++i) {
    lp[i] = ptr<float>(*l[i]); pp[i] = ptr<float>(*p[i]);
    stride[i] = p[i]->stride(0); elems[i] = l[i]->size(1) * l[i]->size(2);
  }
  const char* what = kOrdering;
  int rc;
  {
    NoGil other_threads;
    rc = as.begin({&etc, l[0], l[1], l[2], p[0], p[1], p[2]});
    if (rc == MEP_OK) {
      what = "mep_grad_reduce";
      rc = mep_grad_reduce_batch(3, lp, pp, stride, elems, ptr<int>(etc), c.rank, 1, c.epn, c.R, 0, as.stream);
    }
    rc = as.launched(rc);
  }
  if (failed(rc, what)) return nullptr;
  if (async) return as.end();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// ---- the expert FFN --------------------------------------------------------------------------
struct Ffn {
  const at::Tensor *rows, *slots = nullptr, *cu, *gate, *up, *down;
  int n, M, H, Hp, G;  // ranks, rows and groups of a rank
  bool many;           // every tensor has a leading rank dimension
  at::TensorOptions bf16, f32;
  hipStream_t stream;
  // shape of a tensor with `s` per rank
  c10::SmallVector<int64_t, 5> per_rank(std::initializer_list<int64_t> s) const {
    c10::SmallVector<int64_t, 5> v;
    if (many) v.push_back(n);
    v.append(s.begin(), s.end());
    return v;
  }
  bool of(const at::Tensor& t, std::initializer_list<int64_t> s) const { return t.sizes() == c10::IntArrayRef(per_rank(s)); }
  at::Tensor make(std::initializer_list<int64_t> s, const at::TensorOptions& o) const { return at::empty(per_rank(s), o); }
};

bool dense(const at::Tensor* t, at::ScalarType dt, const at::Tensor& like) {
  return t && t->scalar_type() == dt && t->device() == like.device() && t->is_contiguous() && aligned(t->data_ptr());
}

// args: rows, slots, cu, gate, up, down, token_padding
bool read_ffn(PyObject* const* args, Ffn* f) {
  f->rows = tensor(args[0]);
  if (!f->rows || !f->rows->is_cuda() || !dense(f->rows, at::kBFloat16, *f->rows)) return false;
  const at::Tensor& x = *f->rows;
  if (x.dim() != 2 && x.dim() != 3) return false;
  f->many = x.dim() == 3;
  const int d = f->many;
  f->cu = tensor(args[2]); f->gate = tensor(args[3]); f->up = tensor(args[4]); f->down = tensor(args[5]);
  if (!f->cu || f->cu->scalar_type() != at::kInt || !f->cu->is_contiguous() || f->cu->dim() != 1 + d ||
      f->cu->device() != x.device())
    return false;
  if (!dense(f->gate, at::kBFloat16, x) || !dense(f->up, at::kBFloat16, x) || !dense(f->down, at::kBFloat16, x)) return false;
  const int64_t n = d ? x.size(0) : 1, M = x.size(d), H = x.size(d + 1), G = f->cu->size(d);
  if (f->gate->dim() != 3 + d || M % 128 != 0 || H % 256 != 0 || n <= 0 || M <= 0 || n * M > INT32_MAX ||
      H > (1 << 20) || G <= 0)
    return false;
  const int64_t Hp = f->gate->size(1 + d);
  if (Hp % 128 != 0 || Hp <= 0 || Hp > (1 << 20)) return false;
  f->n = (int)n; f->M = (int)M; f->H = (int)H; f->Hp = (int)Hp; f->G = (int)G;
  if (d && f->cu->size(0) != n) return false;
  if (!f->of(*f->gate, {G, Hp, H}) || !f->of(*f->up, {G, Hp, H}) || !f->of(*f->down, {G, H, Hp})) return false;
  if (args[1] != Py_None) {
    f->slots = tensor(args[1]);
    if (!dense(f->slots, at::kFloat, x) || f->slots->numel() != n * M) return false;
  }
  if (!PyLong_CheckExact(args[6])) return false;
  const long tp = PyLong_AsLong(args[6]);
  if (tp <= 0 || tp % 128 != 0) { PyErr_Clear(); return false; }
  if (x.device().index() != c10::hip::current_device()) return false;
  f->bf16 = x.options(); f->f32 = x.options().dtype(at::kFloat);
  f->stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  return true;
}

// ffn_forward(rows, slots, cu, gate, up, down, token_padding, train) -> y | (y, (gate_pre, up_pre))
PyObject* py_ffn_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) { PyErr_SetString(PyExc_TypeError, "ffn_forward takes 8 arguments"); return nullptr; }
  Ffn f;
  if (!read_ffn(args, &f)) return new_none();
  const bool train = args[7] == Py_True;
  at::Tensor y, gp, up;
  int rc;
  {
    NoGil other_threads;
    y = f.make({f.M, f.H}, f.bf16);
    at::Tensor act = f.make({f.M, f.Hp}, f.bf16);
    if (train) { gp = f.make({f.M, f.Hp}, f.bf16); up = f.make({f.M, f.Hp}, f.bf16); }
    rc = mep_ffn_forward(f.rows->data_ptr(), f.slots ? ptr<float>(*f.slots) : nullptr, ptr<int>(*f.cu), f.G,
                         f.gate->data_ptr(), f.up->data_ptr(), f.down->data_ptr(), act.data_ptr(),
                         ptr<void>(gp), ptr<void>(up), y.data_ptr(), f.n, f.M, f.H, f.Hp, f.stream);
  }
  if (failed(rc, "mep_ffn_forward")) return nullptr;
  if (!train) return THPVariable_Wrap(y);
  return Py_BuildValue("(N(NN))", THPVariable_Wrap(y), THPVariable_Wrap(gp), THPVariable_Wrap(up));
  END_HANDLE_TH_ERRORS
}

// ffn_backward(rows, slots, cu, gate, up, down, token_padding, dy, gate_pre, up_pre, skip_unused,
//              own, from_slots): own and from_slots are tuples of three fp32 tensors for the
//              weight gradients of the lower and the upper half of the groups, or None
//   -> (drows, dslots, dgate, dup, ddown), the last three None where own is given
// Both take several ranks' tensors with a leading rank dimension (the backward with own given).
PyObject* py_ffn_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13) { PyErr_SetString(PyExc_TypeError, "ffn_backward takes 13 arguments"); return nullptr; }
  Ffn f;
  if (!read_ffn(args, &f)) return new_none();
  const at::Tensor *dy = tensor(args[7]), *gp = tensor(args[8]), *up = tensor(args[9]);
  if (!dense(dy, at::kBFloat16, *f.rows) || !dense(gp, at::kBFloat16, *f.rows) || !dense(up, at::kBFloat16, *f.rows) ||
      !f.of(*dy, {f.M, f.H}) || !f.of(*gp, {f.M, f.Hp}) || !f.of(*up, {f.M, f.Hp}))
    return new_none();
  const bool skip = args[10] == Py_True, given = args[11] != Py_None;
  if (f.Hp % 256 != 0 || f.G % 2 != 0 || (f.many && !given)) return new_none();
  float *w[3], *w2[3];
  at::Tensor dw[3];
  for (int i = 0; i < 3; ++i) {
    const int64_t a = i < 2 ? f.Hp : f.H, b = i < 2 ? f.H : f.Hp;
    if (given) {
      if (!PyTuple_Check(args[11]) || PyTuple_GET_SIZE(args[11]) != 3 || !PyTuple_Check(args[12]) ||
          PyTuple_GET_SIZE(args[12]) != 3)
        return new_none();
      const at::Tensor *o = tensor(PyTuple_GET_ITEM(args[11], i)), *s = tensor(PyTuple_GET_ITEM(args[12], i));
      if (!dense(o, at::kFloat, *f.rows) || !dense(s, at::kFloat, *f.rows) || !f.of(*o, {f.G / 2, a, b}) ||
          !f.of(*s, {f.G / 2, a, b}))
        return new_none();
      w[i] = ptr<float>(*o); w2[i] = ptr<float>(*s);
    }
  }
  at::Tensor drows, dslots;
  int rc;
  {
    NoGil other_threads;
    for (int i = 0; i < 3 && !given; ++i) {
      const int64_t a = i < 2 ? f.Hp : f.H, b = i < 2 ? f.H : f.Hp;
      dw[i] = at::empty({f.G, a, b}, f.f32);
      w[i] = ptr<float>(dw[i]); w2[i] = w[i] + (int64_t)(f.G / 2) * a * b;
    }
    drows = f.make({f.M, f.H}, f.bf16);
    at::Tensor dh = f.make({f.M, f.Hp}, f.bf16), dg = f.make({f.M, f.Hp}, f.bf16), du = f.make({f.M, f.Hp}, f.bf16),
               hs = f.make({f.M, f.Hp}, f.bf16);
    if (f.slots) dslots = f.make({f.M}, f.f32);
    rc = mep_ffn_backward(dy->data_ptr(), f.rows->data_ptr(), f.slots ? ptr<float>(*f.slots) : nullptr,
                          ptr<int>(*f.cu), f.G, f.gate->data_ptr(), f.up->data_ptr(), f.down->data_ptr(),
                          gp->data_ptr(), up->data_ptr(), dh.data_ptr(), dg.data_ptr(), du.data_ptr(),
                          hs.data_ptr(), ptr<float>(dslots), drows.data_ptr(), w, w2, f.G / 2, f.n, f.M, f.H, f.Hp,
                          skip ? f.G / 2 : f.G, f.stream);
  }
  if (failed(rc, "mep_ffn_backward")) return nullptr;
  auto give = [](const at::Tensor& t) { return t.defined() ? THPVariable_Wrap(t) : new_none(); };
  return Py_BuildValue("(NNNNN)", give(drows), give(dslots), give(dw[0]), give(dw[1]), give(dw[2]));
  END_HANDLE_TH_ERRORS
}

// ---- context(ctx dict, plan type, no-map token, comm stream, event type) ----------------------
PyObject* py_context(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !PyDict_Check(args[0])) { PyErr_SetString(PyExc_TypeError, "context takes 5 arguments"); return nullptr; }
  PyObject* d = args[0];
  bool ok = true;
  auto num = [&](const char* key) -> int64_t {
    PyObject* o = PyDict_GetItemString(d, key);  // borrowed
    const int64_t v = o ? PyLong_AsLongLong(o) : -1;
    ok = ok && o && !PyErr_Occurred();
    return v;
  };
  auto tens = [&](const char* key) -> at::Tensor {
    PyObject* o = PyDict_GetItemString(d, key);
    const at::Tensor* t = o ? tensor(o) : nullptr;
    return t ? *t : at::Tensor();
  };
  auto cptr = std::make_unique<Ctx>();
  Ctx& c = *cptr;
  c.S = (int)num("S"); c.H = (int)num("H"); c.K = (int)num("K"); c.E = (int)num("E"); c.R = (int)num("R");
  c.NvS = (int)num("NvS"); c.rank = (int)num("rank"); c.tp = (int)num("token_padding");
  c.N = (int64_t)c.S * c.K;
  c.wslot_stride = num("meta_chunk_padded");
  if (!ok) { PyErr_Clear(); return new_none(); }
  c.epn = c.E / c.R;
  c.hidden_buf = tens("hidden_buf"); c.meta_buf = tens("meta_buf");
  c.hidden_local = tens("hidden_buf_local"); c.weights_local = tens("weights_buf_local");
  c.scratch = tens("plan_scratch");
  // the launches below address the weight slots at the start of a meta chunk and shards NvS rows apart
  if (!c.hidden_buf.defined() || !c.meta_buf.defined() || !c.hidden_local.defined() || !c.weights_local.defined() ||
      num("WEIGHTS_OFF") != 0 || num("NvS_padded") != c.NvS || c.H % 8 != 0)
    return new_none();
  auto keep = [](PyObject* o) { Py_INCREF(o); return o; };
  c.plan_type = keep(args[1]);
  c.no_map_token = keep(args[2]);
  c.comm_py = keep(args[3]);
  c.event_type = keep(args[4]);
  c.hidden_local_py = keep(PyDict_GetItemString(d, "hidden_buf_local"));
  c.empty = PyTuple_New(0);
  c.py_N = PyLong_FromLongLong(c.N); c.py_R = PyLong_FromLong(c.R); c.py_E = PyLong_FromLong(c.E);
  c.py_NvS = PyLong_FromLong(c.NvS); c.py_K = PyLong_FromLong(c.K);
  auto stream_num = [&](const char* key) -> int64_t {
    PyObject* o = PyObject_GetAttrString(args[3], key);
    const int64_t v = o ? PyLong_AsLongLong(o) : 0;
    Py_XDECREF(o);
    return v;
  };
  c.comm = c10::Stream::unpack3(stream_num("stream_id"), (c10::DeviceIndex)stream_num("device_index"),
                                (c10::DeviceType)stream_num("device_type"));
  PyObject* cuda = PyImport_ImportModule("torch.cuda");
  c.current_stream = cuda ? PyObject_GetAttrString(cuda, "current_stream") : nullptr;
  Py_XDECREF(cuda);
  if (PyErr_Occurred()) return nullptr;
  PyObject* cap = PyCapsule_New(cptr.get(), kCapsule, free_ctx);
  if (cap) cptr.release();
  return cap;
  END_HANDLE_TH_ERRORS
}

// comes_to_comm(ctx): the communication stream, which the caller is about to use behind its own stream, behind the last
// call that stayed on another; until the caller's leaves_comm(ctx) that stream counts as busy
PyObject* py_comes_to_comm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Ctx* cp = n == 1 ? ctx_of(args[0]) : nullptr;
  if (!cp) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "comes_to_comm takes a context"); return nullptr; }
  Ctx& c = *cp;
  Async as(c, true);
  const bool captured = capturing(c);
  hipError_t e = hipSuccess;
  {
    NoGil other_threads;
    std::lock_guard<std::mutex> lock(c.order_mutex);
    c.comm_used = true;
    if (c.beside_open && captured) {  // a stream under capture cannot wait for what was not captured
      const RelaxedCapture relaxed;
      if (!c.beside_kept) e = c.keep_beside();
      if (e == hipSuccess) e = hipEventSynchronize(c.beside);
    } else if (c.beside_on != as.callers()) {
      e = Async::behind(c, c.comm_raw);
    }
    if (e == hipSuccess) {
      c.beside_open = false;
      ++c.coming;
    }
  }
  if (failed((int)e, kOrdering)) return nullptr;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// leaves_comm(ctx): all that the caller of comes_to_comm had for the communication stream is on it
PyObject* py_leaves_comm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Ctx* c = n == 1 ? ctx_of(args[0]) : nullptr;
  if (!c) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "leaves_comm takes a context"); return nullptr; }
  {
    NoGil other_threads;
    std::lock_guard<std::mutex> lock(c->order_mutex);
    --c->coming;
  }
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define MEP_FAST(f) (PyCFunction)(void (*)(void)) f, METH_FASTCALL, nullptr
PyMethodDef kMethods[] = {{"context", MEP_FAST(py_context)},
                          {"dispatch", MEP_FAST(py_dispatch)},
                          {"combine", MEP_FAST(py_combine)},
                          {"prefetch", MEP_FAST(py_prefetch)},
                          {"reduce_grad", MEP_FAST(py_reduce)},
                          {"comes_to_comm", MEP_FAST(py_comes_to_comm)},
                          {"leaves_comm", MEP_FAST(py_leaves_comm)},
                          {"ffn_forward", MEP_FAST(py_ffn_forward)},
                          {"ffn_backward", MEP_FAST(py_ffn_backward)},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "native host side of the Buffer operators", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  auto s = [](const char* t) { return PyUnicode_InternFromString(t); };
  nm = Names{s("dst"), s("experts_to_copy"), s("zero_fill_ranges"), s("remote_stats"), s("dup_groups"),
             s("dup_loffs"), s("dup_counts"), s("N"), s("R"), s("E"), s("NvS"), s("K"), s("_no_dup_map_in"),
             s("record")};
  return PyModule_Create(&kModule);
}
