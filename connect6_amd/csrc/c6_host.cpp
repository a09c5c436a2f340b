// The host side of a call, natively: argument checks, output tensors, the launch.
//
// A call on few boards is bound by what the host does between two launches, and most of that was
// Python around the C ABI: walking the module's parameters to see whether the packed weights are
// still current (20 tensors), three to six torch.empty calls, a device context, 20-odd ctypes
// conversions.  Measured per call of the B = 1 forward plus mask_logits: 68 us in Python, about 36
// with this.  The kernels are reached through the C ABI's own entry points, whose
// addresses connect6_amd/_lib.py hands over (`bind`), so this module links against no GPU library.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/torch.h>

#include <array>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/connect6_amd.h"

namespace {

struct Abi {
  decltype(&c6_forward) forward;
  decltype(&c6_forward_cascade) forward_cascade;
  decltype(&c6_forward_boards) forward_boards;
  decltype(&c6_forward_boards_cascade) forward_boards_cascade;
  decltype(&c6_cascade_workspace_bytes) cascade_workspace_bytes;
  decltype(&c6_mask_logits) mask_logits;
  decltype(&c6_softmax_sample) softmax_sample;
  decltype(&c6_env_step) env_step;
  decltype(&c6_canonical_input) canonical_input;
  decltype(&c6_forward_generic_packed) forward_generic_packed;
  decltype(&c6_team_bytes) team_bytes;
  decltype(&c6_forward_team) forward_team;
  decltype(&c6_forward_boards_team) forward_boards_team;
  decltype(&c6_stream_capturing) stream_capturing;
  decltype(&c6_forward_cascade_team) forward_cascade_team;
  decltype(&c6_forward_boards_cascade_team) forward_boards_cascade_team;
  decltype(&c6_generic_pack) generic_pack;
} abi;

PyObject *fail(PyObject *type, const std::string &what) {
  PyErr_SetString(type, what.c_str());
  return nullptr;
}

// A tensor argument; anything else is a TypeError (thrown: see HANDLE_TH_ERRORS).
const at::Tensor &tensor(PyObject *o) {
  if (!THPVariable_Check(o)) throw torch::TypeError(std::string("expected a tensor, got ") + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
// ... or null for None
const at::Tensor *tensor_or_null(PyObject *o) { return o == Py_None ? nullptr : &tensor(o); }

std::string shape_text(const at::Tensor &t) {
  std::string s = "(";
  for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
  return s + (t.dim() == 1 ? ",)" : ")");
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return C6_DT_F32;
    case at::kBFloat16: return C6_DT_BF16;
    case at::kHalf: return C6_DT_F16;
    default: return -1;
  }
}
at::ScalarType type_of_code(int code) {
  return code == C6_DT_BF16 ? at::kBFloat16 : (code == C6_DT_F16 ? at::kHalf : at::kFloat);
}

template <class T> T *ptr(const at::Tensor &t) { return t.defined() ? static_cast<T *>(t.data_ptr()) : nullptr; }

at::Tensor fresh(at::IntArrayRef shape, at::ScalarType type, const at::Device &dev) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(dev));
}

// A tensor on a device, contiguous, of a type (or as it is: no trip through the dispatcher then).
bool ready(const at::Tensor &t, const at::Device &dev) { return t.layout() == at::kStrided && t.device() == dev && t.is_contiguous(); }
at::Tensor on(const at::Tensor &t, const at::Device &dev) { return ready(t, dev) ? t : t.to(dev).contiguous(); }
at::Tensor on(const at::Tensor &t, const at::Device &dev, at::ScalarType type) {
  return ready(t, dev) && t.scalar_type() == type ? t : t.to(dev, type).contiguous();
}

PyObject *wrap(const at::Tensor &t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

// (rc, tensors ...): the caller turns a nonzero rc into the exception for it
template <size_t N> PyObject *answer(int rc, const std::array<at::Tensor, N> &ts) {
  PyObject *out = PyTuple_New(N + 1);
  if (out == nullptr) return nullptr;
  PyTuple_SET_ITEM(out, 0, PyLong_FromLong(rc));
  for (size_t i = 0; i < N; ++i) PyTuple_SET_ITEM(out, i + 1, wrap(ts[i]));
  return out;
}

bool is_cascade(int prec) { return prec == C6_PREC_BF16C || prec == C6_PREC_BF16C6; }

at::Tensor cascade_workspace(int64_t boards, const at::Device &dev) {
  size_t bytes = 0;
  if (abi.cascade_workspace_bytes(boards, &bytes) != C6_OK) return {};
  return fresh({(int64_t)(bytes / 4)}, at::kInt, dev);
}

// Buffers of a call that shares a board between workgroups (c6_forward_team); `work` stays undefined
// where the call is not one.
struct Team {
  at::Tensor work, flags;
  uint32_t tag = 0;
};

// The tag of a call behind one that took `last` and last + 1, or 1 where the flag words have to be cleared for it: a word
// that says which XCD a workgroup is on holds a tag's low 28 bits, and one in a slot that few calls use may be as old as
// the words.  A cascade's second pass takes the next tag, so a call counts two.
constexpr uint32_t kTagsEnd = 1u << 28;
constexpr uint32_t next_tag(uint32_t last) { return last == 0 || last > kTagsEnd - 4 ? 1 : last + 2; }
PyObject *team_tag(PyObject *, PyObject *last) {
  const unsigned long v = PyLong_AsUnsignedLong(last);
  return PyErr_Occurred() ? nullptr : PyLong_FromUnsignedLong(next_tag((uint32_t)v));
}

// The flag words are kept per stream, with the last call's tag: calls on one stream follow
// one another, so a tag counted up per call is one that no word holds.  Sixteen streams at most; the
// one that has waited longest gives its words back.  (Only under the interpreter's lock.)  Inside a
// graph capture the words are the graph's own, cleared in the graph: a replay has the same tag.
Team team_buffers(int prec, int64_t boards, const at::Device &dev, void *stream) {
  struct Kept {
    int device;
    void *stream;
    at::Tensor flags;
    uint32_t tag;
    uint64_t used;
  };
  static std::vector<Kept> &kept = *new std::vector<Kept>;   // (never destroyed: the device is gone at exit)
  static uint64_t clock = 0;
  constexpr size_t kMost = 16;
  Team t;
  size_t bytes = 0, flag_bytes = 0;
  if (abi.team_bytes(prec, boards, &bytes, &flag_bytes) != C6_OK || bytes == 0) return t;
  t.work = fresh({(int64_t)bytes}, at::kByte, dev);
  const auto zeros = [&](int64_t words) { return at::zeros({words}, at::TensorOptions().dtype(at::kInt).device(dev)); };
  if (abi.stream_capturing(stream)) {
    t.flags = zeros((int64_t)(flag_bytes / 4));
    t.tag = 1;
    return t;
  }
  Kept *k = nullptr;
  for (Kept &e : kept)
    if (e.device == dev.index() && e.stream == stream) k = &e;
  if (k == nullptr) {
    if (kept.size() == kMost) {
      size_t oldest = 0;
      for (size_t i = 1; i < kept.size(); ++i)
        if (kept[i].used < kept[oldest].used) oldest = i;
      kept.erase(kept.begin() + (long)oldest);
    }
    kept.push_back(Kept{dev.index(), stream, {}, 0, 0});
    k = &kept.back();
  }
  if (!k->flags.defined() || (size_t)k->flags.nbytes() < flag_bytes) k->tag = 0;
  t.tag = next_tag(k->tag);
  if (t.tag == 1) k->flags = zeros((int64_t)(flag_bytes / 4));
  k->tag = t.tag;
  k->used = ++clock;
  t.flags = k->flags;
  return t;
}

// Uniform draws as the kernels read them: fp32 on the device, one per board.
bool take_draws(const at::Tensor *u, int64_t total, const at::Device &dev, at::Tensor &out) {
  out = on(*u, dev, at::kFloat);
  if (out.dim() == 1 && out.size(0) == total) return true;
  fail(PyExc_ValueError, "u must have shape (" + std::to_string(total) + ",), got " + shape_text(out));
  return false;
}

// ---- is the packed copy of a module's parameters still current? --------------------------------
struct ParamKey {
  const void *impl, *data;
  int64_t version;
  int32_t dtype, pad;
};

bool walk_parameters(PyObject *module, std::string &key, PyObject *&first) {
  static PyObject *params_name = PyUnicode_InternFromString("_parameters");
  static PyObject *modules_name = PyUnicode_InternFromString("_modules");
  static PyObject *dict_name = PyUnicode_InternFromString("__dict__");
  PyObject *dict = PyObject_GetAttr(module, dict_name);
  if (dict == nullptr) return false;
  bool ok = true;
  PyObject *k, *v;
  Py_ssize_t pos = 0;
  PyObject *params = PyDict_GetItem(dict, params_name);
  while (params != nullptr && PyDict_Check(params) && PyDict_Next(params, &pos, &k, &v)) {
    if (!THPVariable_Check(v)) continue;
    const at::Tensor &t = THPVariable_Unpack(v);
    if (first == nullptr) first = v;
    // (inference tensors carry no version counter; load_state_dict and refresh_weights bump the epoch)
    const ParamKey e{t.unsafeGetTensorImpl(), t.has_storage() ? t.data_ptr() : nullptr,
                     t.is_inference() ? -1 : (int64_t)t._version(), (int32_t)t.scalar_type(), 0};
    key.append(reinterpret_cast<const char *>(&e), sizeof(e));
  }
  pos = 0;
  PyObject *children = PyDict_GetItem(dict, modules_name);
  while (ok && children != nullptr && PyDict_Check(children) && PyDict_Next(children, &pos, &k, &v))
    if (v != Py_None) ok = walk_parameters(v, key, first);
  Py_DECREF(dict);
  return ok;
}

// parameters(module) -> (key, first parameter or None): the key changes whenever a parameter of the
// module or of a module in it is replaced, moved, retyped or modified in place
PyObject *parameters(PyObject *, PyObject *module) {
  std::string key;
  key.reserve(24 * sizeof(ParamKey));
  PyObject *first = nullptr;
  if (!walk_parameters(module, key, first)) return nullptr;
  PyObject *bytes = PyBytes_FromStringAndSize(key.data(), (Py_ssize_t)key.size());
  if (bytes == nullptr) return nullptr;
  PyObject *out = PyTuple_Pack(2, bytes, first != nullptr ? first : Py_None);
  Py_DECREF(bytes);
  return out;
}

// forward(x, packed, prec, groups, boards_per_group, want_logits, want_value, mask_mode, legal, fill, u,
//         temperature, want_logprob, threshold, logits dtype code, stream[, input code])
// input code: that of an fp32 input which counts as rounded to a 16-bit type (C6_DT_F32_AS_...), or 0
//   -> (rc, logits, value, actions, logprob, cascade: boards evaluated twice as an int32[1])
PyObject *forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 16 && n != 17) return fail(PyExc_TypeError, "forward takes 16 or 17 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor x = tensor(a[0]).contiguous();
  const at::Tensor &packed = tensor(a[1]);
  const int prec = (int)PyLong_AsLong(a[2]);
  const int64_t groups = PyLong_AsLongLong(a[3]), per = PyLong_AsLongLong(a[4]), total = groups * per;
  const bool want_logits = PyObject_IsTrue(a[5]) == 1, want_value = PyObject_IsTrue(a[6]) == 1,
             want_logprob = PyObject_IsTrue(a[12]) == 1;
  const int mask_mode = (int)PyLong_AsLong(a[7]);
  const at::Tensor *legal_in = tensor_or_null(a[8]), *u_in = tensor_or_null(a[10]);
  const float fill = (float)PyFloat_AsDouble(a[9]), temperature = (float)PyFloat_AsDouble(a[11]);
  const float threshold = (float)PyFloat_AsDouble(a[13]);
  const int logits_code = (int)PyLong_AsLong(a[14]);
  void *stream = PyLong_AsVoidPtr(a[15]);
  const int as_code = n > 16 ? (int)PyLong_AsLong(a[16]) : 0;
  if (PyErr_Occurred()) return nullptr;
  const at::Device dev = x.device();
  const int x_code = as_code != 0 && x.scalar_type() == at::kFloat ? as_code : dtype_code(x.scalar_type());
  if (x_code < 0)
    return fail(PyExc_ValueError, std::string("unsupported tensor dtype ") + c10::toString(x.scalar_type()) +
                                      "; expected float32, bfloat16 or float16");
  at::Tensor legal, u, logits, value, actions, logprob, ws;
  if (u_in != nullptr && !take_draws(u_in, total, dev, u)) return nullptr;
  if (legal_in != nullptr) {
    if (legal_in->dim() != 2 || legal_in->size(0) != total || legal_in->size(1) != C6_ACTIONS)
      return fail(PyExc_ValueError, "legal mask must have shape (" + std::to_string(total) + ", 361), got " +
                                        shape_text(*legal_in));
    if (legal_in->scalar_type() != at::kBool && legal_in->scalar_type() != at::kByte)
      return fail(PyExc_ValueError, "legal mask must be a bool or uint8 tensor");
    legal = on(*legal_in, dev);
  }
  const c10::DeviceGuard guard(dev);
  if (want_logits) logits = fresh({total, C6_ACTIONS}, type_of_code(logits_code), dev);
  if (want_value) value = fresh({total}, at::kFloat, dev);
  if (u_in != nullptr) {
    actions = fresh({total}, at::kLong, dev);
    if (want_logprob) logprob = fresh({total}, at::kFloat, dev);
  }
  const size_t stride = (size_t)packed.numel() / (size_t)(groups > 1 ? groups : 1);
  const uint8_t *legal_ptr = static_cast<const uint8_t *>(legal.defined() ? legal.data_ptr() : nullptr);
  int rc;
  if (is_cascade(prec)) {
    ws = cascade_workspace(total, dev);
    const Team t = team_buffers(prec, total, dev, stream);
    rc = t.work.defined()
             ? abi.forward_cascade_team(
                   x.data_ptr(), x_code, groups, per, packed.data_ptr(), stride, prec, ptr<void>(logits), logits_code,
                   ptr<float>(value), mask_mode, legal_ptr, fill, ptr<float>(u), temperature, ptr<int64_t>(actions),
                   ptr<float>(logprob), threshold, ptr<void>(ws), ws.defined() ? ws.nbytes() : 0, t.work.data_ptr(),
                   t.work.nbytes(), t.flags.data_ptr(), t.flags.nbytes(), t.tag, 0, stream)
             : abi.forward_cascade(x.data_ptr(), x_code, groups, per, packed.data_ptr(), stride, prec, ptr<void>(logits),
                             logits_code, ptr<float>(value), mask_mode, legal_ptr, fill, ptr<float>(u), temperature,
                             ptr<int64_t>(actions), ptr<float>(logprob), threshold, ptr<void>(ws),
                             ws.defined() ? ws.nbytes() : 0, stream);
  } else if (const Team t = team_buffers(prec, total, dev, stream); t.work.defined()) {
    rc = abi.forward_team(x.data_ptr(), x_code, groups, per, packed.data_ptr(), stride, prec, ptr<float>(logits),
                          ptr<float>(value), mask_mode, legal_ptr, fill, ptr<float>(u), temperature,
                          ptr<int64_t>(actions), ptr<float>(logprob), t.work.data_ptr(), t.work.nbytes(),
                          t.flags.data_ptr(), t.flags.nbytes(), t.tag, 0, stream);
  } else {
    rc = abi.forward(x.data_ptr(), x_code, groups, per, packed.data_ptr(), stride, prec, ptr<float>(logits),
                     ptr<float>(value), mask_mode, legal_ptr, fill, ptr<float>(u), temperature,
                     ptr<int64_t>(actions), ptr<float>(logprob), stream);
  }
  return answer<5>(rc, {logits, value, actions, logprob, ws.defined() ? ws.narrow(0, 0, 1) : ws});
  END_HANDLE_TH_ERRORS
}

// forward_boards(boards, player, stones_left, index, view, packed, prec, want_logits, mask_mode, fill, u,
//                temperature, threshold, stream) -> as forward; the state tensors are checked by the caller
PyObject *forward_boards(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 14) return fail(PyExc_TypeError, "forward_boards takes 14 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor &boards_in = tensor(a[0]);
  const at::Device dev = boards_in.device();
  const int64_t states = boards_in.size(0);
  const at::Tensor boards = boards_in.contiguous();
  const at::Tensor player = on(tensor(a[1]), dev);
  const at::Tensor left = on(tensor(a[2]), dev);
  const at::Tensor *index_in = tensor_or_null(a[3]), *u_in = tensor_or_null(a[10]);
  const int view = (int)PyLong_AsLong(a[4]);
  const at::Tensor &packed = tensor(a[5]);
  const int prec = (int)PyLong_AsLong(a[6]);
  const bool want_logits = PyObject_IsTrue(a[7]) == 1;
  const int mask_mode = (int)PyLong_AsLong(a[8]);
  const float fill = (float)PyFloat_AsDouble(a[9]), temperature = (float)PyFloat_AsDouble(a[11]);
  const float threshold = (float)PyFloat_AsDouble(a[12]);
  void *stream = PyLong_AsVoidPtr(a[13]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor index, u, logits, actions, logprob, ws;
  if (index_in != nullptr) index = on(*index_in, dev);
  const int64_t total = index.defined() ? index.numel() : states;
  if (u_in != nullptr && !take_draws(u_in, total, dev, u)) return nullptr;
  const c10::DeviceGuard guard(dev);
  if (want_logits) logits = fresh({total, C6_ACTIONS}, at::kFloat, dev);
  const at::Tensor value = fresh({total}, at::kFloat, dev);
  if (u_in != nullptr) {
    actions = fresh({total}, at::kLong, dev);
    logprob = fresh({total}, at::kFloat, dev);
  }
  int rc;
  if (is_cascade(prec)) {
    ws = cascade_workspace(total, dev);
    const Team t = team_buffers(prec, total, dev, stream);
    rc = t.work.defined()
             ? abi.forward_boards_cascade_team(
                   ptr<int8_t>(boards), ptr<int8_t>(player), ptr<int8_t>(left), states, ptr<int64_t>(index), view, total,
                   packed.data_ptr(), prec, ptr<void>(logits), C6_DT_F32, ptr<float>(value), mask_mode, fill,
                   ptr<float>(u), temperature, ptr<int64_t>(actions), ptr<float>(logprob), threshold, ptr<void>(ws),
                   ws.defined() ? ws.nbytes() : 0, t.work.data_ptr(), t.work.nbytes(), t.flags.data_ptr(),
                   t.flags.nbytes(), t.tag, 0, stream)
             : abi.forward_boards_cascade(ptr<int8_t>(boards), ptr<int8_t>(player), ptr<int8_t>(left), states,
                                    ptr<int64_t>(index), view, total, packed.data_ptr(), prec, ptr<void>(logits),
                                    C6_DT_F32, ptr<float>(value), mask_mode, fill, ptr<float>(u), temperature,
                                    ptr<int64_t>(actions), ptr<float>(logprob), threshold, ptr<void>(ws),
                                    ws.defined() ? ws.nbytes() : 0, stream);
  } else if (const Team t = team_buffers(prec, total, dev, stream); t.work.defined()) {
    rc = abi.forward_boards_team(ptr<int8_t>(boards), ptr<int8_t>(player), ptr<int8_t>(left), states,
                                 ptr<int64_t>(index), view, total, packed.data_ptr(), prec, ptr<float>(logits),
                                 ptr<float>(value), mask_mode, fill, ptr<float>(u), temperature, ptr<int64_t>(actions),
                                 ptr<float>(logprob), t.work.data_ptr(), t.work.nbytes(), t.flags.data_ptr(),
                                 t.flags.nbytes(), t.tag, 0, stream);
  } else {
    rc = abi.forward_boards(ptr<int8_t>(boards), ptr<int8_t>(player), ptr<int8_t>(left), states, ptr<int64_t>(index),
                            view, total, packed.data_ptr(), prec, ptr<float>(logits), ptr<float>(value), mask_mode,
                            fill, ptr<float>(u), temperature, ptr<int64_t>(actions), ptr<float>(logprob), stream);
  }
  return answer<5>(rc, {logits, value, actions, logprob, ws.defined() ? ws.narrow(0, 0, 1) : ws});
  END_HANDLE_TH_ERRORS
}

// Names as Python objects, made once: a look into a dictionary by a C string makes one each time.
PyObject *interned(const char *name) { return PyUnicode_InternFromString(name); }
PyObject *index_name(int i) {
  static std::vector<PyObject *> &names = *new std::vector<PyObject *>;   // (under the interpreter's lock)
  while ((int)names.size() <= i) names.push_back(interned(std::to_string(names.size()).c_str()));
  return names[(size_t)i];
}
std::string path_text(std::initializer_list<PyObject *> path) {
  std::string name;
  for (PyObject *part : path) name += (name.empty() ? "" : ".") + std::string(PyUnicode_AsUTF8(part));
  return name;
}

// A tensor of a module by the path of its name ("convs", "3", "weight"), as state_dict() finds it: null where
// there is none (no Python error set).
const at::Tensor *module_tensor(PyObject *module, std::initializer_list<PyObject *> path) {
  static PyObject *dict_name = interned("__dict__"), *parameters_name = interned("_parameters"),
                  *modules_name = interned("_modules"), *buffers_name = interned("_buffers");
  const at::Tensor *found = nullptr;
  PyObject *at = module;   // (borrowed: the module above holds it)
  for (size_t i = 0; i < path.size() && at != nullptr; ++i) {
    PyObject *dict = PyObject_GetAttr(at, dict_name);
    at = nullptr;
    if (dict == nullptr) break;
    PyObject *name = path.begin()[i];
    const bool last = i + 1 == path.size();
    for (PyObject *kind : {last ? parameters_name : modules_name, buffers_name}) {
      PyObject *of = PyDict_GetItem(dict, kind);
      PyObject *v = of != nullptr && PyDict_Check(of) ? PyDict_GetItem(of, name) : nullptr;
      if (v == nullptr || v == Py_None) continue;
      if (!last) at = v;
      else if (THPVariable_Check(v)) found = &THPVariable_Unpack(v);
      break;
    }
    Py_DECREF(dict);
  }
  PyErr_Clear();
  return found;
}

struct GenericCall {
  at::Tensor x, legal, logits, value;
  int x_code = -1, layers = 0, prec = 0, mask_mode = 0;
  const int *kernels = nullptr, *channels = nullptr;
  int64_t b = 0, board = 0;
  float fill = 0.0f;
  void *stream = nullptr;
};
// arguments x, architecture, precision, want_value, mask_mode, legal, fill, stream; the outputs
bool generic_call(GenericCall &c, PyObject *x, PyObject *arch_bytes, PyObject *prec, PyObject *want_value,
                  PyObject *mask_mode, PyObject *legal, PyObject *fill, PyObject *stream) {
  c.x = tensor(x).contiguous();
  char *arch = nullptr;
  Py_ssize_t bytes = 0;
  if (PyBytes_AsStringAndSize(arch_bytes, &arch, &bytes) != 0) return false;
  c.layers = (int)(bytes / (2 * sizeof(int)));
  c.kernels = reinterpret_cast<const int *>(arch);
  c.channels = c.kernels + c.layers;
  c.prec = (int)PyLong_AsLong(prec);
  c.mask_mode = (int)PyLong_AsLong(mask_mode);
  c.fill = (float)PyFloat_AsDouble(fill);
  c.stream = PyLong_AsVoidPtr(stream);
  const at::Tensor *legal_in = tensor_or_null(legal);
  if (PyErr_Occurred()) return false;
  const at::Device dev = c.x.device();
  c.b = c.x.size(0);
  c.board = c.x.size(3);
  c.x_code = dtype_code(c.x.scalar_type());
  if (c.x_code < 0) {
    fail(PyExc_ValueError, std::string("unsupported tensor dtype ") + c10::toString(c.x.scalar_type()) +
                               "; expected float32, bfloat16 or float16");
    return false;
  }
  if (legal_in != nullptr) {
    if (legal_in->dim() != 2 || legal_in->size(0) != c.b || legal_in->size(1) != c.board * c.board) {
      fail(PyExc_ValueError, "legal mask must have shape (" + std::to_string(c.b) + ", " +
                                 std::to_string(c.board * c.board) + "), got " + shape_text(*legal_in));
      return false;
    }
    c.legal = on(*legal_in, dev);
  }
  const c10::DeviceGuard guard(dev);
  c.logits = fresh({c.b, c.board * c.board}, at::kFloat, dev);
  if (PyObject_IsTrue(want_value) == 1) c.value = fresh({c.b}, at::kFloat, dev);
  return true;
}
int generic_launch(const GenericCall &c, const at::Tensor &packed, int64_t groups) {
  return abi.forward_generic_packed(
      c.x.data_ptr(), c.x_code, groups, c.b / groups, (int)c.board, c.layers, c.kernels, c.channels, packed.data_ptr(),
      (size_t)(packed.numel() / groups), c.prec, ptr<float>(c.logits), ptr<float>(c.value), c.mask_mode,
      static_cast<const uint8_t *>(c.legal.defined() ? c.legal.data_ptr() : nullptr), c.fill, c.stream);
}

// forward_generic(x, packed, groups, architecture, prec, want_value, mask_mode, legal, fill, stream[, input code])
//   -> (rc, logits, value).  architecture: bytes of the C ints kernels[layers], channels[layers]
PyObject *forward_generic(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 10 && n != 11) return fail(PyExc_TypeError, "forward_generic takes 10 or 11 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor &packed = tensor(a[1]);
  const int64_t groups = PyLong_AsLongLong(a[2]);
  const int as_code = n > 10 ? (int)PyLong_AsLong(a[10]) : 0;
  if (PyErr_Occurred()) return nullptr;
  GenericCall c;
  if (!generic_call(c, a[0], a[3], a[4], a[5], a[6], a[7], a[8], a[9])) return nullptr;
  if (as_code != 0 && c.x.scalar_type() == at::kFloat) c.x_code = as_code;
  const c10::DeviceGuard guard(c.x.device());
  return answer<2>(generic_launch(c, packed, groups), {c.logits, c.value});
  END_HANDLE_TH_ERRORS
}

// forward_generic_module(module, x, packed bytes, architecture, prec, mask_mode, legal, fill, stream)
//   -> (rc, logits, value).  The module's parameters as they are now, packed by a launch in front of the
//   forward's: an edit that no version counter shows (p.data) counts, as it does where a layer reads them.
PyObject *forward_generic_module(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 9) return fail(PyExc_TypeError, "forward_generic_module takes 9 arguments");
  HANDLE_TH_ERRORS
  const int64_t bytes = PyLong_AsLongLong(a[2]);
  if (PyErr_Occurred()) return nullptr;
  GenericCall c;
  if (!generic_call(c, a[1], a[3], a[4], Py_True, a[5], a[6], a[7], a[8])) return nullptr;
  const at::Device dev = c.x.device();
  const c10::DeviceGuard guard(dev);
  static PyObject *convs = interned("convs"), *weight = interned("weight"), *bias_name = interned("bias"),
                  *policy = interned("policy_output"), *value = interned("value_output");
  std::vector<at::Tensor> keep;   // (copies, where a parameter is not fp32, contiguous and on the device)
  bool ok = true;
  const auto take = [&](std::initializer_list<PyObject *> path, int64_t count, bool required) -> const float * {
    const at::Tensor *t = ok ? module_tensor(a[0], path) : nullptr;
    if (t == nullptr) {
      if (ok && required) ok = fail(PyExc_KeyError, "missing parameter " + path_text(path)) != nullptr;
      return nullptr;
    }
    if (t->numel() != count) {
      ok = fail(PyExc_ValueError, path_text(path) + " has " + std::to_string(t->numel()) +
                                      " elements, the network's layers need " + std::to_string(count)) != nullptr;
      return nullptr;
    }
    // (as it is, where it is what the launch reads: the module holds it)
    if (t->layout() == at::kStrided && t->scalar_type() == at::kFloat && t->device() == dev && t->is_contiguous() &&
        !t->is_neg() && t->has_storage())
      return ptr<float>(*t);
    keep.push_back(t->detach().to(dev, at::kFloat).contiguous());
    return ptr<float>(keep.back());
  };
  std::vector<const float *> w((size_t)c.layers), bias((size_t)c.layers);
  int64_t cin = 3;
  for (int l = 0; l < c.layers; ++l) {
    w[(size_t)l] = take({convs, index_name(l), weight}, cin * c.channels[l] * c.kernels[l] * c.kernels[l], true);
    bias[(size_t)l] = take({convs, index_name(l), bias_name}, c.channels[l], false);
    cin = c.channels[l];
  }
  const float *pol_w = take({policy, weight}, cin, true), *pol_b = take({policy, bias_name}, 1, false);
  const float *val_w = take({value, weight}, cin, false), *val_b = take({value, bias_name}, 1, false);
  if (!ok) return nullptr;
  if (val_w == nullptr) return fail(PyExc_ValueError, "missing parameter value_output.weight: no value without it");
  const at::Tensor packed = fresh({bytes}, at::kByte, dev);
  int rc = abi.generic_pack(1, (int)c.board, c.layers, c.kernels, c.channels, w.data(), bias.data(), pol_w, pol_b, val_w,
                            val_b, c.prec, packed.data_ptr(), (size_t)bytes, c.stream);
  if (rc == C6_OK) rc = generic_launch(c, packed, 1);
  return answer<2>(rc, {c.logits, c.value});
  END_HANDLE_TH_ERRORS
}

// mask_logits(logits, legal, stream) -> (rc, masked); the fill is the lowest finite value of the type
PyObject *mask_logits(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 3) return fail(PyExc_TypeError, "mask_logits takes 3 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor src = tensor(a[0]).contiguous();
  const at::Tensor &legal_in = tensor(a[1]);
  void *stream = PyLong_AsVoidPtr(a[2]);
  if (PyErr_Occurred()) return nullptr;
  const at::Device dev = src.device();
  const int code = dtype_code(src.scalar_type());
  if (code < 0)
    return fail(PyExc_ValueError, std::string("unsupported tensor dtype ") + c10::toString(src.scalar_type()) +
                                      "; expected float32, bfloat16 or float16");
  const at::Tensor legal = on(legal_in, dev);
  // bit patterns of -(largest finite value): fp32, bf16, fp16
  const uint32_t fill = code == C6_DT_F32 ? 0xFF7FFFFFu : (code == C6_DT_BF16 ? 0xFF7Fu : 0xFBFFu);
  const c10::DeviceGuard guard(dev);
  const at::Tensor out = fresh(src.sizes(), src.scalar_type(), dev);
  const int rc = abi.mask_logits(src.data_ptr(), static_cast<const uint8_t *>(legal.data_ptr()), code, src.size(0),
                                 fill, out.data_ptr(), stream);
  return answer<1>(rc, {out});
  END_HANDLE_TH_ERRORS
}

// sample(logits, legal, temperature, u, want_logprob, stream) -> (rc, actions, logprob)
PyObject *sample(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 6) return fail(PyExc_TypeError, "sample takes 6 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor src = on(tensor(a[0]), tensor(a[0]).device(), at::kFloat);
  const at::Tensor *legal_in = tensor_or_null(a[1]);
  const float temperature = (float)PyFloat_AsDouble(a[2]);
  const at::Device dev = src.device();
  const int64_t b = src.size(0);
  void *stream = PyLong_AsVoidPtr(a[5]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor legal, u, logprob;
  if (legal_in != nullptr) legal = on(*legal_in, dev);
  if (!take_draws(&tensor(a[3]), b, dev, u)) return nullptr;
  const c10::DeviceGuard guard(dev);
  const at::Tensor actions = fresh({b}, at::kLong, dev);
  if (PyObject_IsTrue(a[4]) == 1) logprob = fresh({b}, at::kFloat, dev);
  const int rc = abi.softmax_sample(ptr<float>(src), static_cast<const uint8_t *>(ptr<void>(legal)), ptr<float>(u),
                                    temperature, b, ptr<int64_t>(actions), ptr<float>(logprob), stream);
  return answer<2>(rc, {actions, logprob});
  END_HANDLE_TH_ERRORS
}

// env_step(boards, player, stones_left, empty_count, move_count, actions, view, win_length, stream)
//   -> (rc, reward, done, winner, sign, lengths)
PyObject *env_step(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 9) return fail(PyExc_TypeError, "env_step takes 9 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor &boards = tensor(a[0]);
  const at::Device dev = boards.device();
  const int64_t num = boards.size(0);
  const at::Tensor &actions = tensor(a[5]);
  const int view = (int)PyLong_AsLong(a[6]), win = (int)PyLong_AsLong(a[7]);
  void *stream = PyLong_AsVoidPtr(a[8]);
  if (PyErr_Occurred()) return nullptr;
  const c10::DeviceGuard guard(dev);
  const at::Tensor reward = fresh({num}, at::kFloat, dev), done = fresh({num}, at::kBool, dev),
                   winner = fresh({num}, at::kChar, dev), sign = fresh({num}, at::kChar, dev),
                   lengths = fresh({num}, at::kShort, dev);
  const int rc = abi.env_step(ptr<int8_t>(boards), ptr<int8_t>(tensor(a[1])),
                              ptr<int8_t>(tensor(a[2])), ptr<int16_t>(tensor(a[3])),
                              ptr<int16_t>(tensor(a[4])), ptr<int64_t>(actions), view, num,
                              (int)boards.size(1), win, ptr<float>(reward), static_cast<uint8_t *>(done.data_ptr()),
                              ptr<int8_t>(winner), ptr<int8_t>(sign), ptr<int16_t>(lengths), stream);
  return answer<5>(rc, {reward, done, winner, sign, lengths});
  END_HANDLE_TH_ERRORS
}

// canonical_input(boards, player, stones_left, stream) -> (rc, planes); rc is kBadState where the state is not what
// VectorConnect6 holds (the caller says what is wrong)
constexpr int kBadState = -1000;
bool state_ok(const at::Tensor &boards, const at::Tensor &player, const at::Tensor &left) {
  if (!boards.is_cuda() || boards.dim() != 3 || boards.size(1) != boards.size(2)) return false;
  for (const at::Tensor *t : {&boards, &player, &left})
    if (t->scalar_type() != at::kChar || t->device() != boards.device()) return false;
  return player.dim() == 1 && player.size(0) == boards.size(0) && left.dim() == 1 && left.size(0) == boards.size(0);
}
PyObject *canonical_input(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 4) return fail(PyExc_TypeError, "canonical_input takes 4 arguments");
  HANDLE_TH_ERRORS
  if (!state_ok(tensor(a[0]), tensor(a[1]), tensor(a[2]))) return answer<1>(kBadState, {at::Tensor()});
  const at::Tensor boards = tensor(a[0]).contiguous(), player = tensor(a[1]).contiguous(),
                   left = tensor(a[2]).contiguous();
  void *stream = PyLong_AsVoidPtr(a[3]);
  if (PyErr_Occurred()) return nullptr;
  const at::Device dev = boards.device();
  const int64_t num = boards.size(0), size = boards.size(2);
  const c10::DeviceGuard guard(dev);
  const at::Tensor out = fresh({num, 3, size, size}, at::kFloat, dev);
  const int rc = abi.canonical_input(ptr<int8_t>(boards), ptr<int8_t>(player), ptr<int8_t>(left), num, (int)size,
                                     ptr<float>(out), stream);
  return answer<1>(rc, {out});
  END_HANDLE_TH_ERRORS
}

// bind(addresses): the C ABI's entry points, in the order of `Abi`
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
  constexpr Py_ssize_t kEntries = sizeof(Abi) / sizeof(void *);
  if (n != kEntries) return fail(PyExc_TypeError, "bind takes one address per entry point");
  std::array<void *, kEntries> addr;
  for (Py_ssize_t i = 0; i < kEntries; ++i) addr[i] = PyLong_AsVoidPtr(a[i]);
  if (PyErr_Occurred()) return nullptr;
  std::memcpy(&abi, addr.data(), sizeof(abi));
  Py_RETURN_NONE;
}

#define C6_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {C6_FAST(bind),        C6_FAST(forward),        C6_FAST(forward_boards),
                         C6_FAST(mask_logits), C6_FAST(sample),         C6_FAST(env_step),
                         C6_FAST(canonical_input), C6_FAST(forward_generic), C6_FAST(forward_generic_module),
                         {"parameters", parameters, METH_O, nullptr},
                         {"team_tag", team_tag, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_c6_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__c6_host(void) { return PyModule_Create(&module_def); }
