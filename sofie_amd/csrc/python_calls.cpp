// Calls of the C-ABI from Python: `call(name, *args)` of a Runtime as one native method that converts the arguments and calls the entry
// point itself.
//
// A launch costs the host about 2.1 us in the HIP runtime; a ctypes call around it took another 0.7 - 1.2 us (one converter object
// per argument, two Python frames), which is what a program of small kernels then waits for.  Here an argument is a type test and
// a load: 0.1 - 0.2 us a call.  What this file does not know (another kind of argument, a wrong count, a status that is not 0) goes
// to the Python path of the same name, which converts, raises and reports as before.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include "sofie_hip.h"
#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

namespace {

// ---- what ctypes objects look like ----------------------------------------------------------------------------------------
// Where a ctypes instance keeps the address of its value, and where a byref() object keeps the address and the object it was
// made from.  Not part of any interface, so learned from sample objects when the module is loaded; an offset that the samples
// do not agree on stays 0, and such arguments take the Python path.
struct CtypesLayout {
   Py_ssize_t data = 0;                    // instance -> void * of its value
   Py_ssize_t ref_address = 0, ref_obj = 0; // byref() object -> void *, PyObject *
   // Other parameters that ctypes has already converted (c_int.from_param) have the same type as a byref() object.  The two words behind the
   // object's head, the second of which begins with a letter, tell them apart.
   void *ref_kind = nullptr;
   char ref_letter = 0;
   PyTypeObject *void_p = nullptr, *size_t_ = nullptr, *float_ = nullptr, *array = nullptr, *ref = nullptr;
} g_layout;

PyObject *new_reference(PyObject *o)
{
   Py_INCREF(o);
   return o;
}
void *word_at(PyObject *o, Py_ssize_t offset) { return *(void **)((char *)o + offset); }
constexpr Py_ssize_t REF_KIND = sizeof(PyObject), REF_LETTER = REF_KIND + (Py_ssize_t)sizeof(void *);
bool is_reference(PyObject *o) { return word_at(o, REF_KIND) == g_layout.ref_kind && ((const char *)o)[REF_LETTER] == g_layout.ref_letter; }

// ---- one argument ---------------------------------------------------------------------------------------------------------
// `want`: the structure type a typed pointer asks for, or null.  False: not an argument this file converts.
template <class T>
bool take(PyObject *o, PyTypeObject *want, T &out)
{
   if constexpr (std::is_pointer_v<T>) {
      if (o == Py_None)
         return out = nullptr, true;
      PyTypeObject *t = Py_TYPE(o);
      if (t == g_layout.ref && g_layout.ref_address) {
         if (!is_reference(o))
            return false;
         PyObject *of = (PyObject *)word_at(o, g_layout.ref_obj);
         if (want && (!of || Py_TYPE(of) != want))
            return false;
         return out = (T)word_at(o, g_layout.ref_address), true;
      }
      if (want || !g_layout.data)
         return false;
      if (t == g_layout.void_p)
         return out = (T) * (void **)word_at(o, g_layout.data), true;
      if (PyType_IsSubtype(t, g_layout.array))
         return out = (T)word_at(o, g_layout.data), true;
      return false;
   } else if constexpr (std::is_floating_point_v<T>) {
      if (PyFloat_CheckExact(o))
         return out = (T)PyFloat_AS_DOUBLE(o), true;
      if (Py_TYPE(o) == g_layout.float_ && g_layout.data)
         return out = (T) * (float *)word_at(o, g_layout.data), true;
      return false;
   } else {
      static_assert(std::is_integral_v<T>);
      if (PyLong_Check(o)) {
         int overflow = 0;
         const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
         return out = (T)v, !overflow;
      }
      // a parameter of another type, of the same size though it be, refuses a c_size_t
      if (std::is_same_v<T, size_t> && Py_TYPE(o) == g_layout.size_t_ && g_layout.data)
         return out = (T) * (size_t *)word_at(o, g_layout.data), true;
      return false;
   }
}

// ---- one entry point ------------------------------------------------------------------------------------------------------
enum { NOT_TAKEN = -1 };
struct Entry;
typedef int (*Thunk)(const Entry &, sofie_hip_ctx *, PyObject *const *);
struct Entry {
   void *function = nullptr;
   Thunk thunk = nullptr;
   Py_ssize_t count = 0; // arguments behind the context
   std::vector<PyTypeObject *> want;
};

template <class... A, std::size_t... I>
int call_as(int (*fn)(sofie_hip_ctx *, A...), const Entry &e, sofie_hip_ctx *ctx, PyObject *const *args, std::index_sequence<I...>)
{
   std::tuple<std::decay_t<A>...> v;
   if (!(take(args[I], e.want[I], std::get<I>(v)) && ...))
      return NOT_TAKEN;
   int status;
   Py_BEGIN_ALLOW_THREADS
   status = fn(ctx, std::get<I>(v)...);
   Py_END_ALLOW_THREADS
   return status;
}

template <class F>
struct ThunkOf;
template <class... A>
struct ThunkOf<int(sofie_hip_ctx *, A...)> {
   static constexpr Py_ssize_t count = sizeof...(A);
   static int run(const Entry &e, sofie_hip_ctx *ctx, PyObject *const *args)
   {
      return call_as<A...>((int (*)(sofie_hip_ctx *, A...))e.function, e, ctx, args, std::index_sequence_for<A...>());
   }
};

struct Known {
   const char *name;
   Thunk thunk;
   Py_ssize_t count;
};
#define KNOWN(f) {#f, ThunkOf<decltype(f)>::run, ThunkOf<decltype(f)>::count}
// every entry point that a pass of a model is made of; the others (set-up, statistics) take the Python path
const Known kKnown[] = {
   KNOWN(sofie_hip_gemm_f32),
   KNOWN(sofie_hip_gemm_chain_f32),
   KNOWN(sofie_hip_gemm_i8),
   KNOWN(sofie_hip_gemm_i8_noalloc),
   KNOWN(sofie_hip_gemm_fp8),
   KNOWN(sofie_hip_transpose_i8),
   KNOWN(sofie_hip_transpose_f32),
   KNOWN(sofie_hip_strided_gather_f32),
   KNOWN(sofie_hip_copy_rows),
   KNOWN(sofie_hip_copy),
   KNOWN(sofie_hip_fill_zero),
   KNOWN(sofie_hip_upload),
   KNOWN(sofie_hip_download),
   KNOWN(sofie_hip_sync),
   KNOWN(sofie_hip_quantize_fp8),
   KNOWN(sofie_hip_quantize_linear),
   KNOWN(sofie_hip_dequantize_linear_i8),
   KNOWN(sofie_hip_dequantize_linear_i32),
   KNOWN(sofie_hip_unary_f32),
   KNOWN(sofie_hip_unary_chain_f32),
   KNOWN(sofie_hip_add_f32),
   KNOWN(sofie_hip_binary_f32),
   KNOWN(sofie_hip_conv_f32),
   KNOWN(sofie_hip_conv3d_f32),
   KNOWN(sofie_hip_conv_i8),
   KNOWN(sofie_hip_global_avg_pool_f32),
   KNOWN(sofie_hip_global_avg_pool_i8),
   KNOWN(sofie_hip_pool_f32),
   KNOWN(sofie_hip_pool3d_f32),
   KNOWN(sofie_hip_plane_sums_to_average),
   KNOWN(sofie_hip_plane_sums_take_average),
   KNOWN(sofie_hip_softmax_f32),
   KNOWN(sofie_hip_reduce_f32),
   KNOWN(sofie_hip_layernorm_f32),
   KNOWN(sofie_hip_batchnorm_f32),
};

PyObject *g_entries = nullptr; // name -> index into g_table
std::vector<Entry> g_table;

// ---- the method -----------------------------------------------------------------------------------------------------------
// Runtime.call: a method, so that what a caller keeps of it (rt.call, held over a loop) keeps the Runtime, and its context with it, alive;
// and the context is read from the Runtime at each call, so that one that was closed in between is refused.
PyObject *g_ctx_name = nullptr; // "ctx"
PyObject *g_slow = nullptr;     // slow(runtime, status or None, name, *args): converts anything, raises

PyObject *slow_call(PyObject *self, PyObject *const *args, Py_ssize_t n, PyObject *kwnames, PyObject *status)
{
   PyObject *all = PyTuple_New(n + 2), *kw = nullptr, *r = nullptr;
   if (!all)
      return nullptr;
   PyTuple_SET_ITEM(all, 0, new_reference(self));
   PyTuple_SET_ITEM(all, 1, new_reference(status));
   for (Py_ssize_t i = 0; i < n; i++)
      PyTuple_SET_ITEM(all, i + 2, new_reference(args[i]));
   bool good = true;
   if (kwnames) {
      kw = PyDict_New();
      good = kw != nullptr;
      for (Py_ssize_t i = 0; good && i < PyTuple_GET_SIZE(kwnames); i++)
         good = PyDict_SetItem(kw, PyTuple_GET_ITEM(kwnames, i), args[n + i]) == 0;
   }
   if (good)
      r = PyObject_Call(g_slow, all, kw);
   Py_XDECREF(kw);
   Py_DECREF(all);
   return r;
}

PyObject *call_method(PyObject *self, PyObject *const *args, Py_ssize_t n, PyObject *kwnames)
{
   if (n >= 1 && !kwnames && PyUnicode_CheckExact(args[0])) {
      PyObject *index = PyDict_GetItemWithError(g_entries, args[0]);
      if (index) {
         const Entry &e = g_table[(size_t)PyLong_AsSsize_t(index)];
         if (e.count == n - 1) {
            PyObject *held = PyObject_GetAttr(self, g_ctx_name);
            if (!held)
               return nullptr;
            sofie_hip_ctx *ctx = nullptr;
            const int status = take(held, nullptr, ctx) ? e.thunk(e, ctx, args + 1) : (int)NOT_TAKEN;
            Py_DECREF(held);
            if (status == SOFIE_HIP_OK)
               Py_RETURN_NONE;
            if (status != NOT_TAKEN) {
               PyObject *s = PyLong_FromLong(status);
               if (!s)
                  return nullptr;
               PyObject *r = slow_call(self, args, n, nullptr, s);
               Py_DECREF(s);
               return r;
            }
         }
      } else if (PyErr_Occurred())
         return nullptr;
   }
   return slow_call(self, args, n, kwnames, Py_None);
}

PyMethodDef g_call = {"call", (PyCFunction)(void (*)(void))call_method, METH_FASTCALL | METH_KEYWORDS,
                      "call(name, *args): the entry point of that name on this context; raises SofieHipError where it fails"};

// method(type, slow): the method `call` of that type
PyObject *make_method(PyObject *, PyObject *args)
{
   PyObject *type, *slow;
   if (!PyArg_ParseTuple(args, "O!O", &PyType_Type, &type, &slow))
      return nullptr;
   Py_XDECREF(g_slow);
   g_slow = new_reference(slow);
   return PyDescr_NewMethod((PyTypeObject *)type, &g_call);
}

// entry(name, address of the function, tuple of the structure types its typed pointers ask for (None: any)) -> whether it is taken
PyObject *add_entry(PyObject *, PyObject *args)
{
   PyObject *name, *address, *want;
   if (!PyArg_ParseTuple(args, "UOO!", &name, &address, &PyTuple_Type, &want))
      return nullptr;
   const char *text = PyUnicode_AsUTF8(name);
   if (!text)
      return nullptr;
   for (const Known &k : kKnown)
      if (strcmp(text, k.name) == 0 && PyTuple_GET_SIZE(want) == k.count) {
         Entry e;
         e.function = PyLong_AsVoidPtr(address);
         if (!e.function)
            return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "%s has no address", text);
         e.thunk = k.thunk;
         e.count = k.count;
         for (Py_ssize_t i = 0; i < k.count; i++) {
            PyObject *t = PyTuple_GET_ITEM(want, i);
            e.want.push_back(PyType_Check(t) ? (PyTypeObject *)new_reference(t) : nullptr);
         }
         PyObject *index = PyLong_FromSize_t(g_table.size());
         if (!index)
            return nullptr;
         g_table.push_back(std::move(e));
         const int bad = PyDict_SetItem(g_entries, name, index);
         Py_DECREF(index);
         if (bad)
            return nullptr;
         Py_RETURN_TRUE;
      }
   Py_RETURN_FALSE;
}

// The one offset in every object of `objects` at which the word of the same position in `words` stands; 0 if there is none or they differ.
Py_ssize_t offset_of(const std::vector<PyObject *> &objects, const std::vector<void *> &words)
{
   for (Py_ssize_t off = (Py_ssize_t)sizeof(PyObject); off + (Py_ssize_t)sizeof(void *) <= Py_TYPE(objects[0])->tp_basicsize; off += (Py_ssize_t)sizeof(void *)) {
      bool all = true;
      for (size_t i = 0; i < objects.size(); i++)
         all = all && off + (Py_ssize_t)sizeof(void *) <= Py_TYPE(objects[i])->tp_basicsize && word_at(objects[i], off) == words[i];
      if (all)
         return off;
   }
   return 0;
}

// layout(c_void_p, c_size_t, c_float, Array, type of byref(), [(instance, address)], [(byref object, address, object)])
PyObject *learn_layout(PyObject *, PyObject *args)
{
   PyObject *types[5], *instances, *refs;
   if (!PyArg_ParseTuple(args, "O!O!O!O!O!O!O!", &PyType_Type, &types[0], &PyType_Type, &types[1], &PyType_Type, &types[2], &PyType_Type, &types[3], &PyType_Type, &types[4],
                         &PyList_Type, &instances, &PyList_Type, &refs))
      return nullptr;
   std::vector<PyObject *> objects;
   std::vector<void *> words, owners;
   for (Py_ssize_t i = 0; i < PyList_GET_SIZE(instances); i++) {
      PyObject *o, *a;
      if (!PyArg_ParseTuple(PyList_GET_ITEM(instances, i), "OO", &o, &a))
         return nullptr;
      objects.push_back(o);
      words.push_back(PyLong_AsVoidPtr(a));
   }
   g_layout.data = objects.size() >= 2 ? offset_of(objects, words) : 0;
   objects.clear();
   words.clear();
   for (Py_ssize_t i = 0; i < PyList_GET_SIZE(refs); i++) {
      PyObject *o, *a, *of;
      if (!PyArg_ParseTuple(PyList_GET_ITEM(refs, i), "OOO", &o, &a, &of))
         return nullptr;
      objects.push_back(o);
      words.push_back(PyLong_AsVoidPtr(a));
      owners.push_back(of);
   }
   g_layout.ref_address = objects.size() >= 2 ? offset_of(objects, words) : 0;
   g_layout.ref_obj = objects.size() >= 2 ? offset_of(objects, owners) : 0;
   if (!objects.empty()) {
      g_layout.ref_kind = word_at(objects[0], REF_KIND);
      g_layout.ref_letter = ((const char *)objects[0])[REF_LETTER];
   }
   bool alike = g_layout.ref_address > REF_LETTER && g_layout.ref_obj > REF_LETTER;
   for (PyObject *o : objects)
      alike = alike && is_reference(o);
   if (!alike)
      g_layout.ref_address = 0;
   if (PyErr_Occurred())
      return nullptr;
   PyTypeObject **to[5] = {&g_layout.void_p, &g_layout.size_t_, &g_layout.float_, &g_layout.array, &g_layout.ref};
   for (int i = 0; i < 5; i++)
      *to[i] = (PyTypeObject *)new_reference(types[i]);
   return PyBool_FromLong(g_layout.data && g_layout.ref_address);
}

PyMethodDef g_methods[] = {{"method", make_method, METH_VARARGS, "method(type, slow): what Runtime.call is"},
                           {"entry", add_entry, METH_VARARGS, "entry(name, address, wanted types): an entry point of the library"},
                           {"layout", learn_layout, METH_VARARGS, "layout(...): where ctypes objects keep their addresses"},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_calls", "Calls of the C-ABI", -1, g_methods};

} // namespace

PyMODINIT_FUNC PyInit__calls(void)
{
   g_entries = PyDict_New();
   g_ctx_name = PyUnicode_InternFromString("ctx");
   if (!g_entries || !g_ctx_name)
      return nullptr;
   return PyModule_Create(&g_module);
}
