// Python extension module arcticinference_amd._host_ext: the host layer of torch_forwards.cpp as plain functions
// of positional arguments, one per operator schema of py_custom_ops.py, which binds them to the CUDA dispatch key and calls them directly
// for eager GPU calls.  The per-layer tensor lists of the bulk write are read in place from the Python list
// (borrowed references, no copy into a vector): at 40 layers that is 160 tensors per call, and what a serving
// process pays on every engine step.  A failed check raises RuntimeError, as TORCH_CHECK does in the reference.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <string>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "torch_host.hpp"

namespace {

namespace py = pybind11;
using arctic_host::OptTensor;

// By the object's own type: a proxy or a mock that calls itself a Tensor holds none, and the question must not raise.
bool is_tensor(PyObject *o) { return PyObject_TypeCheck(o, (PyTypeObject *)THPVariableClass); }

// ---- functions of positional arguments, called by Python's vector call -----------------------------------------
// A call of an operator costs as much in the conversion of its arguments as in its checks, so these take what Python
// hands over without a tuple, tensors by reference (0.2 to 0.3 us a call less than through pybind's dispatch).
// What they accept is what pybind's casters of the same types do.
struct Refused {
  const char *wanted;
};
template <typename T>
struct From;
template <>
struct From<const at::Tensor &> {
  static const at::Tensor &get(PyObject *o) {
    if (!is_tensor(o)) throw Refused{"a Tensor"};
    return THPVariable_Unpack(o);
  }
};
template <>
struct From<const OptTensor &> {
  static OptTensor get(PyObject *o) {
    if (o == Py_None) return c10::nullopt;
    if (!is_tensor(o)) throw Refused{"a Tensor or None"};
    return THPVariable_Unpack(o);
  }
};
template <>
struct From<double> {
  static double get(PyObject *o) {
    if (PyFloat_CheckExact(o)) return PyFloat_AS_DOUBLE(o);
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw Refused{"a float"};
    return v;
  }
};
template <>
struct From<int64_t> {
  static int64_t get(PyObject *o) {
    if (PyFloat_Check(o)) throw Refused{"an int"};
    long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      // neither an int nor an index, but a number that int() takes (numpy's float32, a tensor of one float, a Decimal)
      PyErr_Clear();
      const py::object number = py::reinterpret_steal<py::object>(PyNumber_Check(o) ? PyNumber_Long(o) : nullptr);
      if (number) v = PyLong_AsLongLong(number.ptr());
      if (!number || (v == -1 && PyErr_Occurred())) throw Refused{"an int"};
    }
    return v;
  }
};
template <>
struct From<bool> {
  static bool get(PyObject *o) {
    if (o == Py_True || o == Py_False) return o == Py_True;
    if (o == Py_None) return false;
    const PyNumberMethods *number = Py_TYPE(o)->tp_as_number;
    const int v = number && number->nb_bool ? number->nb_bool(o) : -1;
    if (v < 0) throw Refused{"a bool"};
    return v != 0;
  }
};
template <>
struct From<const std::string &> {
  static std::string get(PyObject *o) {
    Py_ssize_t n = 0;
    const char *text = PyUnicode_Check(o) ? PyUnicode_AsUTF8AndSize(o, &n) : nullptr;
    if (!text && PyBytes_Check(o)) text = PyBytes_AS_STRING(o), n = PyBytes_GET_SIZE(o);
    if (!text && PyByteArray_Check(o)) text = PyByteArray_AS_STRING(o), n = PyByteArray_GET_SIZE(o);
    if (!text) throw Refused{"a str"};
    return std::string(text, (size_t)n);
  }
};
template <>
struct From<const py::handle &> {
  static py::handle get(PyObject *o) { return o; }
};

PyObject *to_python(const at::Tensor &t) { return THPVariable_Wrap(t); }
PyObject *to_python(const std::tuple<at::Tensor, at::Tensor> &t) {
  py::object first = py::reinterpret_steal<py::object>(to_python(std::get<0>(t))),
             second = py::reinterpret_steal<py::object>(to_python(std::get<1>(t)));
  if (!first || !second) return nullptr;
  return PyTuple_Pack(2, first.ptr(), second.ptr());
}

template <auto kFunction, typename R, typename... Args, size_t... I>
PyObject *call_with(R (*)(Args...), PyObject *const *args, std::index_sequence<I...>) {
  if constexpr (std::is_void_v<R>) {
    kFunction(From<Args>::get(args[I])...);
    Py_RETURN_NONE;
  } else {
    return to_python(kFunction(From<Args>::get(args[I])...));
  }
}
template <typename R, typename... Args>
constexpr Py_ssize_t arity(R (*)(Args...)) {
  return sizeof...(Args);
}
template <auto kFunction>
PyObject *fast_call(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  constexpr Py_ssize_t kArity = arity(kFunction);
  if (n != kArity) return PyErr_Format(PyExc_TypeError, "%zd arguments are needed, %zd were given", kArity, n);
  try {
    return call_with<kFunction>(kFunction, args, std::make_index_sequence<(size_t)kArity>());
  } catch (const Refused &r) {
    PyErr_Clear();
    return PyErr_Format(PyExc_TypeError, "incompatible function arguments: %s is needed where something else was given",
                        r.wanted);
  } catch (py::error_already_set &e) {
    e.restore();
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}
template <auto kFunction>
void def(py::module_ &m, const char *name) {
  static PyMethodDef method = {name, (PyCFunction)(void *)fast_call<kFunction>, METH_FASTCALL, nullptr};
  const py::object module_name = m.attr("__name__");
  py::object function = py::reinterpret_steal<py::object>(PyCFunction_NewEx(&method, nullptr, module_name.ptr()));
  if (!function) throw py::error_already_set();
  m.add_object(name, function);
}

// Whether `o`, or the first element of the list or tuple `o`, is a tensor on a GPU: what decides whether a call goes
// straight to the functions below.  A tensor subclass may answer for its device in Python, and raise there.
PyObject *on_gpu(PyObject *, PyObject *o) {
  HANDLE_TH_ERRORS
  if (PyList_Check(o) && PyList_GET_SIZE(o)) o = PyList_GET_ITEM(o, 0);
  else if (PyTuple_Check(o) && PyTuple_GET_SIZE(o)) o = PyTuple_GET_ITEM(o, 0);
  return PyBool_FromLong(is_tensor(o) && THPVariable_Unpack(o).is_cuda());
  END_HANDLE_TH_ERRORS
}

// A Python list or tuple of tensors, read in place.
class TensorSequence {
 public:
  TensorSequence(const py::handle &obj, const char *what) {
    fast_ = py::reinterpret_steal<py::object>(PySequence_Fast(obj.ptr(), what));
    if (!fast_) throw py::error_already_set();
    count_ = PySequence_Fast_GET_SIZE(fast_.ptr());
    items_ = PySequence_Fast_ITEMS(fast_.ptr());
    for (Py_ssize_t i = 0; i < count_; ++i)
      TORCH_CHECK(is_tensor(items_[i]), what, ": element ", (int64_t)i, " is not a Tensor");
  }
  int64_t size() const { return (int64_t)count_; }
  const at::Tensor &operator[](int64_t i) const { return THPVariable_Unpack(items_[i]); }

 private:
  py::object fast_;
  PyObject **items_ = nullptr;
  Py_ssize_t count_ = 0;
};

struct PyLayerLists {
  const TensorSequence *list[4];
};
const at::Tensor &py_layer_get(const void *ctx, int list, int64_t l) { return (*((const PyLayerLists *)ctx)->list[list])[l]; }
const at::Tensor &py_list_get(const void *ctx, int64_t i) { return (*(const TensorSequence *)ctx)[i]; }

void bulk(const at::Tensor &keys, const at::Tensor &values, const py::handle &key_caches, const py::handle &value_caches,
          const at::Tensor &slot_mapping, const std::string &kv_cache_dtype, const py::handle &k_scales,
          const py::handle &v_scales, int64_t num_heads, int64_t head_size, const arctic_host::SelectRows *select) {
  const TensorSequence kc(key_caches, "key_caches must be a list of Tensors"),
      vc(value_caches, "value_caches must be a list of Tensors"), ks(k_scales, "k_scales must be a list of Tensors"),
      vs(v_scales, "v_scales must be a list of Tensors");
  const PyLayerLists lists = {{&kc, &vc, &ks, &vs}};
  const arctic_host::LayerLists layers = {{kc.size(), vc.size(), ks.size(), vs.size()}, py_layer_get, &lists};
  arctic_host::bulk_write(keys, values, layers, slot_mapping, kv_cache_dtype, num_heads, head_size, select);
}

void reshape_and_cache_flash_bulk(const at::Tensor &keys, const at::Tensor &values, const py::handle &key_caches,
                                  const py::handle &value_caches, const at::Tensor &slot_mapping,
                                  const std::string &kv_cache_dtype, const py::handle &k_scales,
                                  const py::handle &v_scales, int64_t num_heads, int64_t head_size) {
  bulk(keys, values, key_caches, value_caches, slot_mapping, kv_cache_dtype, k_scales, v_scales, num_heads, head_size,
       nullptr);
}

void reshape_and_cache_flash_bulk_select(const at::Tensor &keys, const at::Tensor &values, const py::handle &key_caches,
                                         const py::handle &value_caches, const at::Tensor &slot_mapping,
                                         const std::string &kv_cache_dtype, const py::handle &k_scales,
                                         const py::handle &v_scales, int64_t num_heads, int64_t head_size,
                                         const at::Tensor &logits_indices, const at::Tensor &k_out,
                                         const at::Tensor &v_out) {
  const arctic_host::SelectRows select = {logits_indices, k_out, v_out};
  bulk(keys, values, key_caches, value_caches, slot_mapping, kv_cache_dtype, k_scales, v_scales, num_heads, head_size,
       &select);
}

// The per-layer tensors of a bulk write, checked once and held, for a caller that writes the same layers on every
// step (SwiftKV's caller rebuilds its four lists of views on every engine step, llama_swiftkv.py:594-615, which costs
// it more host time than the write).  The object keeps an alias of every tensor, so the addresses in its tables stay
// allocated and the geometry it checked cannot change under it; it must be rebuilt when the pool is (the caller
// knows: its kv_cache objects are new ones then).
class PreparedLayers {
 public:
  PreparedLayers(const py::handle &key_caches, const py::handle &value_caches, const py::handle &k_scales,
                 const py::handle &v_scales) {
    const TensorSequence kc(key_caches, "key_caches must be a list of Tensors"),
        vc(value_caches, "value_caches must be a list of Tensors"), ks(k_scales, "k_scales must be a list of Tensors"),
        vs(v_scales, "v_scales must be a list of Tensors");
    const TensorSequence *lists[4] = {&kc, &vc, &ks, &vs};
    for (const TensorSequence *list : lists)
      for (int64_t i = 0; i < list->size(); ++i) held_.push_back((*list)[i].alias());
    // the tables are made from the held aliases, not from the caller's objects
    offsets_[0] = 0;
    for (int k = 0; k < 4; ++k) offsets_[k + 1] = offsets_[k] + lists[k]->size();
    const arctic_host::LayerLists layers = {
        {kc.size(), vc.size(), ks.size(), vs.size()},
        [](const void *ctx, int list, int64_t l) -> const at::Tensor & {
          const PreparedLayers *self = (const PreparedLayers *)ctx;
          return self->held_[(size_t)(self->offsets_[list] + l)];
        },
        this};
    checked_ = arctic_host::check_layers(layers);
  }
  int64_t num_layers() const { return checked_.num_layers; }
  void write(const at::Tensor &keys, const at::Tensor &values, const at::Tensor &slot_mapping,
             const std::string &kv_cache_dtype, int64_t num_heads, int64_t head_size) const {
    arctic_host::bulk_write(keys, values, checked_, slot_mapping, kv_cache_dtype, num_heads, head_size, nullptr);
  }
  void write_select(const at::Tensor &keys, const at::Tensor &values, const at::Tensor &slot_mapping,
                    const std::string &kv_cache_dtype, int64_t num_heads, int64_t head_size,
                    const at::Tensor &logits_indices, const at::Tensor &k_out, const at::Tensor &v_out) const {
    const arctic_host::SelectRows select = {logits_indices, k_out, v_out};
    arctic_host::bulk_write(keys, values, checked_, slot_mapping, kv_cache_dtype, num_heads, head_size, &select);
  }

 private:
  std::vector<at::Tensor> held_;
  int64_t offsets_[5];
  arctic_host::CheckedLayers checked_;
};

void reshape_and_cache_flash_fp4(const at::Tensor &key, const at::Tensor &value, const at::Tensor &key_cache,
                                 const at::Tensor &value_cache, const at::Tensor &slot_mapping,
                                 const std::string &kv_cache_dtype, const at::Tensor &k_scale, const at::Tensor &v_scale,
                                 const at::Tensor &key_scale_cache, const at::Tensor &value_scale_cache) {
  (void)kv_cache_dtype, (void)k_scale, (void)v_scale;   // accepted and unused, as in the reference
  arctic_host::cache_write_fp4(key, value, key_cache, value_cache, slot_mapping, key_scale_cache, value_scale_cache);
}

at::Tensor speculator_ln_cuda(const at::Tensor &input, const OptTensor &weight, const OptTensor &bias, double eps) {
  return arctic_host::add_ln_act("speculator_ln", input, c10::nullopt, c10::nullopt, weight, bias, 0.0, eps, "none", 1.0);
}

at::Tensor speculator_add_ln_act_cuda(const at::Tensor &input, const OptTensor &z, const OptTensor &weight,
                                      const OptTensor &bias, double alpha, double eps, const std::string &activation,
                                      double out_scale) {
  return arctic_host::add_ln_act("speculator_add_ln_act", input, z, c10::nullopt, weight, bias, alpha, eps, activation,
                                 out_scale);
}

at::Tensor speculator_embed_add_ln_act_cuda(const at::Tensor &input, const at::Tensor &emb_weight,
                                            const at::Tensor &token_ids, const OptTensor &weight, const OptTensor &bias,
                                            double alpha, double eps, const std::string &activation, double out_scale) {
  return arctic_host::add_ln_act("speculator_embed_add_ln_act", input, emb_weight, token_ids, weight, bias, alpha, eps,
                                 activation, out_scale);
}

using TwoTensors = std::tuple<at::Tensor, at::Tensor>;

TwoTensors sum_lstm_cuda(const at::Tensor &states_4d, const at::Tensor &z4_4d, const OptTensor &prev_cell_d,
                         const OptTensor &w_cell, const OptTensor &b_cell, const OptTensor &w_state,
                         const OptTensor &b_state, double alpha, double eps_cell, double eps_state, bool use_fast_gelu) {
  return arctic_host::sum_lstm(states_4d, z4_4d, c10::nullopt, prev_cell_d, w_cell, b_cell, w_state, b_state, alpha,
                               eps_cell, eps_state, use_fast_gelu, false);
}

TwoTensors sum_lstm_zero_cell_cuda(const at::Tensor &states_4d, const at::Tensor &z4_4d, const OptTensor &w_cell,
                                   const OptTensor &b_cell, const OptTensor &w_state, const OptTensor &b_state,
                                   double alpha, double eps_cell, double eps_state, bool use_fast_gelu) {
  return arctic_host::sum_lstm(states_4d, z4_4d, c10::nullopt, c10::nullopt, w_cell, b_cell, w_state, b_state, alpha,
                               eps_cell, eps_state, use_fast_gelu, false);
}

TwoTensors sum_lstm_shared_z_cuda(const at::Tensor &states_4d, const at::Tensor &z_d, const OptTensor &prev_cell_d,
                                  const OptTensor &w_cell, const OptTensor &b_cell, const OptTensor &w_state,
                                  const OptTensor &b_state, double alpha, double eps_cell, double eps_state,
                                  bool use_fast_gelu) {
  return arctic_host::sum_lstm(states_4d, z_d, c10::nullopt, prev_cell_d, w_cell, b_cell, w_state, b_state, alpha,
                               eps_cell, eps_state, use_fast_gelu, true);
}

TwoTensors sum_lstm_embedded_cuda(const at::Tensor &states_4d, const at::Tensor &emb_weight, const at::Tensor &token_ids,
                                  const OptTensor &prev_cell_d, const OptTensor &w_cell, const OptTensor &b_cell,
                                  const OptTensor &w_state, const OptTensor &b_state, double alpha, double eps_cell,
                                  double eps_state, bool use_fast_gelu) {
  return arctic_host::sum_lstm(states_4d, emb_weight, token_ids, prev_cell_d, w_cell, b_cell, w_state, b_state, alpha,
                               eps_cell, eps_state, use_fast_gelu, true);
}

void move(const char *fn, const py::handle &sources, const at::Tensor &indices, const py::handle &outs, bool scatter) {
  const TensorSequence src(sources, "sources must be a list of Tensors"), dst(outs, "outs must be a list of Tensors");
  const arctic_host::TensorList s = {src.size(), py_list_get, &src}, d = {dst.size(), py_list_get, &dst};
  arctic_host::move_rows(fn, s, indices, d, scatter);
}
void gather_rows(const py::handle &sources, const at::Tensor &indices, const py::handle &outs) {
  move("gather_rows", sources, indices, outs, false);
}
void scatter_rows(const py::handle &sources, const at::Tensor &indices, const py::handle &outs) {
  move("scatter_rows", sources, indices, outs, true);
}

at::Tensor speculator_argmax_cuda(const at::Tensor &logits, int64_t max_index) {
  return arctic_host::argmax_clamp(logits, max_index);
}

}  // namespace

PYBIND11_MODULE(_host_ext, m) {
  m.doc() = "C++ host layer of the arctic_inference operators over libarctic_mi355x.so";
  def<&reshape_and_cache_flash_bulk>(m, "reshape_and_cache_flash_bulk");
  def<&reshape_and_cache_flash_bulk_select>(m, "reshape_and_cache_flash_bulk_select");
  def<&reshape_and_cache_flash_fp4>(m, "reshape_and_cache_flash_fp4");
  def<&speculator_ln_cuda>(m, "speculator_ln_cuda");
  def<&speculator_add_ln_act_cuda>(m, "speculator_add_ln_act_cuda");
  def<&speculator_embed_add_ln_act_cuda>(m, "speculator_embed_add_ln_act_cuda");
  def<&sum_lstm_cuda>(m, "sum_lstm_cuda");
  def<&sum_lstm_zero_cell_cuda>(m, "sum_lstm_zero_cell_cuda");
  def<&sum_lstm_shared_z_cuda>(m, "sum_lstm_shared_z_cuda");
  def<&sum_lstm_embedded_cuda>(m, "sum_lstm_embedded_cuda");
  def<&gather_rows>(m, "gather_rows");
  def<&scatter_rows>(m, "scatter_rows");
  def<&speculator_argmax_cuda>(m, "speculator_argmax_cuda");
  static PyMethodDef method = {"on_gpu", on_gpu, METH_O, nullptr};
  m.add_object("on_gpu", py::reinterpret_steal<py::object>(PyCFunction_New(&method, nullptr)));
  py::class_<PreparedLayers>(m, "BulkKVLayers")
      .def(py::init<const py::handle &, const py::handle &, const py::handle &, const py::handle &>(),
           py::arg("key_caches"), py::arg("value_caches"), py::arg("k_scales"), py::arg("v_scales"))
      .def_property_readonly("num_layers", &PreparedLayers::num_layers)
      .def("write", &PreparedLayers::write)
      .def("write_select", &PreparedLayers::write_select);
}
