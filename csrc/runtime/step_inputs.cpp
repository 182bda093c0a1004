// A step's inputs: a decode step's, written from the sequences into the pinned image that one copy takes to the device
// (engine/runner.py: _Staging), and those of a step with prompts (mixed_rows), packed into such an image (pack_words).  Bound by the walk over the sequences' block lists: 50 sequences of 210 blocks took 180 us
// as a Python loop with a numpy assignment per field, of a step of 1240.
#include <pybind11/pybind11.h>
#include <pybind11/numpy.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

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

// Rows of an eager step, as numpy arrays by name: the decode rows' ids, positions and cache slots, then those of the prompts' next
// `ntoks` tokens from `starts` (None: the sequence's computed rows) on; block tables and lengths of both; with `segments` what a
// row segment per sequence needs.  A step of 777 rows took 36 us as numpy calls and 75 with 256 blocks, before anything was
// launched and with the card idle.
py::dict mixed_rows(py::list dseqs, py::list pseqs, py::list ntoks, py::list starts, int64_t bs, bool segments) {
  static const Names* nm = new Names();     // (kept for the process: interned strings)
  static PyObject* const computed = PyUnicode_InternFromString("num_computed");
  const int64_t nd = (int64_t)dseqs.size(), np = (int64_t)pseqs.size(), ns = nd + np;
  if (bs < 1 || (int64_t)ntoks.size() != np || (int64_t)starts.size() != np || ns < 1)
    throw std::invalid_argument("mixed_rows: sizes");
  struct Row {
    PyObject* seq;
    py::object tok, blocks;
    const int32_t* ids;
    int64_t first, count, nblk;               // rows' first position and number
  };
  std::vector<Row> r((size_t)ns);
  int64_t rows = 0, d_most = 0, p_most = 0, max_rows = 0, max_kv = 0;
  for (int64_t i = 0; i < ns; ++i) {
    Row& x = r[(size_t)i];
    x.seq = PyList_GET_ITEM((i < nd ? dseqs : pseqs).ptr(), i < nd ? i : i - nd);
    x.tok = attr(x.seq, nm->tok), x.blocks = attr(x.seq, nm->block_ids);
    const int64_t tokens = whole(attr(x.seq, nm->n_tokens).ptr());
    if (!py::isinstance<py::array_t<int32_t>>(x.tok) || !PyList_Check(x.blocks.ptr()))
      throw std::invalid_argument("mixed_rows: a sequence's tokens and blocks");
    py::array tok = py::reinterpret_borrow<py::array>(x.tok);
    x.nblk = PyList_GET_SIZE(x.blocks.ptr());
    int64_t from;                             // of the row's tokens in the sequence
    if (i < nd) {
      x.first = tokens - 1 + whole(attr(x.seq, nm->inflight).ptr());      // (queued ahead: the id comes from the device)
      x.count = 1, from = tokens - 1;
      d_most = std::max(d_most, x.nblk);
    } else {
      PyObject* a = PyList_GET_ITEM(starts.ptr(), i - nd);
      x.first = from = a == Py_None ? whole(attr(x.seq, computed).ptr()) : whole(a);
      x.count = whole(PyList_GET_ITEM(ntoks.ptr(), i - nd));
      p_most = std::max(p_most, x.nblk);
    }
    if (from < 0 || x.count < 1 || from + x.count > tokens || tokens > tok.size() || tok.ndim() != 1 || tok.strides(0) != 4 ||
        x.first < 0 || (x.first + x.count - 1) / bs >= x.nblk)
      throw std::out_of_range("mixed_rows: a sequence's tokens or blocks");
    x.ids = static_cast<const int32_t*>(tok.data(from));
    word(x.first + x.count);
    rows += x.count;
    max_rows = std::max(max_rows, x.count);
    max_kv = std::max(max_kv, x.first + x.count);
  }
  word(rows);
  auto words = [](int64_t n, int32_t*& p) {
    py::array_t<int32_t> a(n);
    p = a.mutable_data();
    return a;
  };
  auto tables = [](int64_t n, int64_t m, int32_t*& p) {
    py::array_t<int32_t> a({n, m});
    p = a.mutable_data();
    std::fill_n(p, n * m, 0);
    return a;
  };
  py::dict out;
  int32_t *ids, *pos, *slots, *seq_lens, *qsl, *bt, *d_bt = nullptr, *d_sl = nullptr;
  int32_t *start = nullptr, *pos0 = nullptr, *slot = nullptr, *len = nullptr, *sg_bt = nullptr;
  const int64_t most = std::max(d_most, p_most), p_cols = np ? p_most : 1;
  out["ids"] = words(rows, ids), out["pos"] = words(rows, pos), out["slots"] = words(rows, slots);
  out["seq_lens"] = words(np, seq_lens), out["qsl"] = words(np + 1, qsl);
  out["bt"] = tables(std::max<int64_t>(1, np), p_cols, bt);
  if (nd) out["d_bt"] = tables(nd, d_most, d_bt), out["d_sl"] = words(nd, d_sl);
  if (segments) {
    out["sg_start"] = words(ns + 1, start), out["sg_pos0"] = words(ns, pos0), out["sg_slot"] = words(ns, slot);
    out["sg_len"] = words(ns, len), out["sg_bt"] = tables(ns, most, sg_bt);
    out["num_segs"] = ns, out["max_rows"] = max_rows, out["max_kv"] = max_kv;
  }
  int64_t at = 0;
  qsl[0] = 0;
  for (int64_t i = 0; i < ns; ++i) {
    const Row& x = r[(size_t)i];
    int32_t* table = i < nd ? d_bt + i * d_most : bt + (i - nd) * p_cols;
    for (int64_t b = 0; b < x.nblk; ++b) table[b] = word(whole(PyList_GET_ITEM(x.blocks.ptr(), b)));
    if (segments) {
      start[i] = (int32_t)at, pos0[i] = (int32_t)x.first, len[i] = (int32_t)(x.first + x.count);
      slot[i] = word(whole(attr(x.seq, nm->state_slot).ptr()));
      std::copy_n(table, x.nblk, sg_bt + i * most);
    }
    std::copy_n(x.ids, x.count, ids + at);
    for (int64_t k = 0; k < x.count; ++k) {
      const int64_t p = x.first + k;
      pos[at + k] = (int32_t)p;
      slots[at + k] = word(table[p / bs] * bs + p % bs);
    }
    at += x.count;
    if (i < nd) d_sl[i] = (int32_t)(x.first + 1);
    else seq_lens[i - nd] = (int32_t)(x.first + x.count), qsl[i - nd + 1] = (int32_t)(at - nd);
  }
  if (segments) start[ns] = (int32_t)at;
  return out;
}

// Arrays of 4- or 8-byte entries one after the other into an int32 image, each from a whole `align` words on: (words in all, each
// array's first word).  An image that is too small is left as it is.
py::tuple pack_words(py::list arrays, py::array image, int64_t align) {
  int32_t* to = rows_of<int32_t>(image, 0, "pack_words: image");
  if (align < 1) throw std::invalid_argument("pack_words: align");
  py::list offs;
  std::vector<std::pair<py::array, int64_t>> from;
  int64_t n = 0;
  for (py::handle h : arrays) {
    py::array a = py::array::ensure(h, py::array::c_style);
    if (!a) throw py::error_already_set();
    if (a.itemsize() != 4 && a.itemsize() != 8) throw py::type_error("upload: unsupported dtype " + py::str(a.dtype()).cast<std::string>());
    offs.append(n);
    from.emplace_back(a, n);
    n += (a.nbytes() / 4 + align - 1) / align * align;
  }
  n = std::max(n, align);
  if (n <= image.size())
    for (auto& f : from) std::memcpy(to + f.second, f.first.data(), (size_t)f.first.nbytes());
  return py::make_tuple(n, offs);
}

// ids[i] = the i-th of a list of whole numbers: a prompt of 4096 takes 40 us less than through numpy's conversion
void fill_ids(py::array ids, py::list tokens) {
  const int64_t n = (int64_t)tokens.size();
  int32_t* to = rows_of<int32_t>(ids, n, "fill_ids: ids");
  for (int64_t i = 0; i < n; ++i) {
    const int64_t x = whole(PyList_GET_ITEM(tokens.ptr(), i));
    if (x < INT32_MIN || x > INT32_MAX) {        // (as numpy says it)
      PyErr_SetString(PyExc_OverflowError, "a token id exceeds 32 bits");
      throw py::error_already_set();
    }
    to[i] = (int32_t)x;
  }
}

}  // namespace

void register_step_inputs(py::module_& m) {
  m.def("fill_decode", &fill_decode, py::arg("seqs"), py::arg("block_size"), py::arg("mb"), py::arg("nb"),
        py::arg("stateful"), py::arg("small"), py::arg("table"), py::arg("f32"), py::arg("seeds"));
  m.def("mixed_rows", &mixed_rows, py::arg("dseqs"), py::arg("pseqs"), py::arg("ntoks"), py::arg("starts"),
        py::arg("block_size"), py::arg("segments"));
  m.def("pack_words", &pack_words, py::arg("arrays"), py::arg("image"), py::arg("align"));
  m.def("fill_ids", &fill_ids, py::arg("ids"), py::arg("tokens"));
}
