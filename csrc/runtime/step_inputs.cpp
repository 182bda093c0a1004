// A decode step's inputs, written from the sequences into the pinned image that one copy takes to the device
// (engine/runner.py: _Staging).  Bound by the walk over the sequences' block lists: 50 sequences of 210 blocks took 180 us
// as a Python loop with a numpy assignment per field, of a step of 1240.
#include <pybind11/pybind11.h>
#include <pybind11/numpy.h>

#include <cstdint>

namespace py = pybind11;

namespace {

struct Names {
  PyObject *n_tokens, *prompt_len, *inflight, *tok, *block_ids, *state_slot, *preemptions, *params, *temperature, *top_p,
      *top_k, *seed;
  Names() {
    auto in = [](const char* s) { return PyUnicode_InternFromString(s); };
    n_tokens = in("n_tokens"), prompt_len = in("prompt_len"), inflight = in("inflight"), tok = in("_tok");
    block_ids = in("block_ids"), state_slot = in("state_slot"), preemptions = in("preemptions"), params = in("params");
    temperature = in("temperature"), top_p = in("top_p"), top_k = in("top_k"), seed = in("seed");
  }
};

py::object attr(PyObject* o, PyObject* name) {
  PyObject* v = PyObject_GetAttr(o, name);
  if (v == nullptr) throw py::error_already_set();
  return py::reinterpret_steal<py::object>(v);
}

int64_t whole(PyObject* v) {
  if (!PyIndex_Check(v)) {                   // (a whole number in another type)
    PyObject* n = PyNumber_Long(v);
    if (n == nullptr) throw py::error_already_set();
    return whole(py::reinterpret_steal<py::object>(n).ptr());
  }
  const int64_t x = PyLong_AsLongLong(v);
  if (x == -1 && PyErr_Occurred()) throw py::error_already_set();
  return x;
}

int32_t word(int64_t x) {
  if (x < INT32_MIN || x > INT32_MAX) throw std::out_of_range("a decode step's input exceeds 32 bits");
  return (int32_t)x;
}

double real(PyObject* v) {
  const double x = PyFloat_AsDouble(v);
  if (x == -1.0 && PyErr_Occurred()) throw py::error_already_set();
  return x;
}

template <typename T>
T* rows_of(py::array& a, py::ssize_t size, const char* what) {
  if (!py::isinstance<py::array_t<T>>(a) || !(a.flags() & py::array::c_style) || !a.writeable() || a.size() < size)
    throw std::invalid_argument(what);
  return static_cast<T*>(a.mutable_data());
}

// small: int32 fields of mb words each (ids | positions | cache slots | lengths | top_k | steps | state slots); table [mb,
// columns]; f32: temperatures | top_p; seeds.  Rows seqs .. nb - 1 are padding: no cache write, no attention, greedy.
// Returns the widest block table, 1 at least.
int64_t fill_decode(py::list seqs, int64_t block_size, int64_t mb, int64_t nb, bool stateful, py::array small, py::array table,
                    py::array f32, py::array seeds) {
  static const Names* nm = new Names();     // (kept for the process: interned strings)
  const int64_t n = (int64_t)seqs.size();
  if (n > nb || nb > mb || block_size < 1 || table.ndim() != 2 || table.shape(0) < nb)
    throw std::invalid_argument("fill_decode: sizes");
  const int64_t cols = table.shape(1);
  int32_t* hs = rows_of<int32_t>(small, 8 * mb, "fill_decode: small");
  int32_t* bt = rows_of<int32_t>(table, nb * cols, "fill_decode: table");
  float* hf = rows_of<float>(f32, 2 * mb, "fill_decode: f32");
  int64_t* hseed = rows_of<int64_t>(seeds, nb, "fill_decode: seeds");
  int64_t most = 1;
  for (int64_t i = 0; i < n; ++i) {
    PyObject* s = PyList_GET_ITEM(seqs.ptr(), i);
    const int64_t tokens = whole(attr(s, nm->n_tokens).ptr()), inflight = whole(attr(s, nm->inflight).ptr());
    const int64_t p = tokens - 1 + inflight;     // steps queued ahead of this one
    py::object ids = attr(s, nm->tok), blocks = attr(s, nm->block_ids);
    if (!py::isinstance<py::array_t<int32_t>>(ids) || !PyList_Check(blocks.ptr()))
      throw std::invalid_argument("fill_decode: a sequence's tokens and blocks");
    py::array tok = py::reinterpret_borrow<py::array>(ids);
    const int64_t nblk = PyList_GET_SIZE(blocks.ptr());
    if (tokens < 1 || tokens > tok.size() || tok.ndim() != 1 || p < 0 || p / block_size >= nblk || nblk > cols)
      throw std::out_of_range("fill_decode: a sequence's tokens or blocks");
    int32_t* row = bt + i * cols;
    for (int64_t b = 0; b < nblk; ++b) row[b] = word(whole(PyList_GET_ITEM(blocks.ptr(), b)));
    hs[i] = *static_cast<const int32_t*>(tok.data(tokens - 1));     // (replaced on the device when queued ahead)
    hs[mb + i] = word(p);
    hs[2 * mb + i] = word(row[p / block_size] * block_size + p % block_size);
    hs[3 * mb + i] = word(p + 1);
    py::object par = attr(s, nm->params);
    hs[4 * mb + i] = word(whole(attr(par.ptr(), nm->top_k).ptr()));
    hs[5 * mb + i] = word(tokens - whole(attr(s, nm->prompt_len).ptr()) + inflight +
                          131 * whole(attr(s, nm->preemptions).ptr()));
    if (stateful) hs[6 * mb + i] = word(whole(attr(s, nm->state_slot).ptr()));
    hf[i] = (float)real(attr(par.ptr(), nm->temperature).ptr());
    hf[mb + i] = (float)real(attr(par.ptr(), nm->top_p).ptr());
    hseed[i] = whole(attr(par.ptr(), nm->seed).ptr());
    most = nblk > most ? nblk : most;
  }
  for (int64_t i = n; i < nb; ++i) {
    hs[i] = hs[mb + i] = hs[3 * mb + i] = hs[4 * mb + i] = hs[5 * mb + i] = 0;
    hs[2 * mb + i] = -1;
    if (stateful) hs[6 * mb + i] = -1;       // padding rows touch no state
    if (cols > 0) bt[i * cols] = 0;
    hf[i] = 0.f;
    hf[mb + i] = 1.f;
  }
  return most;
}

}  // namespace

void register_step_inputs(py::module_& m) {
  m.def("fill_decode", &fill_decode, py::arg("seqs"), py::arg("block_size"), py::arg("mb"), py::arg("nb"),
        py::arg("stateful"), py::arg("small"), py::arg("table"), py::arg("f32"), py::arg("seeds"));
}
