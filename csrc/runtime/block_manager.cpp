// pybind11 module `_runtime`: Python bindings of the native paged-KV block manager (core in block_manager.h) and of the sentence
// encoder's word tokenizer (word_tokenizer.h).
#include <pybind11/numpy.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include "block_manager.h"
#include "word_tokenizer.h"

namespace py = pybind11;
using dllm::BlockManager;

// A batch of texts as one int32 array: the token ids one text behind the other, each token's place in its text, each text's first
// token, its number of tokens.  Texts that are not ASCII are tokenised by `other(text)`.  Returns (array, tokens, longest text).
static py::tuple pack_words(const py::list& texts, int64_t max_len, int64_t vocab, const py::function& other) {
  if (max_len < 2 || vocab <= 1000) throw py::value_error("pack_words: max_len of at least 2, vocab past 1000");
  dllm::WordHasher hash(vocab);
  std::vector<int32_t> ids, starts;
  for (const py::handle t : texts) {
    if (!PyUnicode_Check(t.ptr())) throw py::type_error("pack_words: texts are str");
    starts.push_back((int32_t)ids.size());
    Py_ssize_t n = 0;
    const char* s = PyUnicode_IS_ASCII(t.ptr()) ? PyUnicode_AsUTF8AndSize(t.ptr(), &n) : nullptr;
    if (!s || !hash.append(s, (size_t)n, max_len, ids)) {
      PyErr_Clear();
      for (const py::handle v : other(t)) ids.push_back(v.cast<int32_t>());
    }
  }
  hash.flush(ids);
  const size_t T = ids.size(), B = starts.size();
  py::array_t<int32_t> out((py::ssize_t)(2 * T + 2 * B));
  int32_t* o = out.mutable_data();
  int32_t longest = 0;
  std::copy(ids.begin(), ids.end(), o);
  for (size_t b = 0; b < B; ++b) {
    const int32_t n = (int32_t)(b + 1 < B ? starts[b + 1] : T) - starts[b];
    for (int32_t i = 0; i < n; ++i) o[T + starts[b] + i] = i;
    o[2 * T + b] = starts[b];
    o[2 * T + B + b] = n;
    longest = std::max(longest, n);
  }
  return py::make_tuple(out, (int64_t)T, longest);
}

// A list of plain ints that fit int32, read without a converter's calls an entry (9000 tokens 230 -> 60 us); anything else is left to the
// overload with std::vector.
struct PlainInts { std::vector<int32_t> v; };
namespace pybind11 { namespace detail {
template <> struct type_caster<PlainInts> {
  PYBIND11_TYPE_CASTER(PlainInts, const_name("list[int]"));
  bool load(handle src, bool) {
    if (!PyList_CheckExact(src.ptr())) return false;
    const Py_ssize_t n = PyList_GET_SIZE(src.ptr());
    value.v.resize((size_t)n);
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* o = PyList_GET_ITEM(src.ptr(), i);
      int over = 0;
      const long x = PyLong_CheckExact(o) ? PyLong_AsLongAndOverflow(o, &over) : (over = 1, 0L);
      if (over || x < INT32_MIN || x > INT32_MAX) return false;
      value.v[(size_t)i] = (int32_t)x;
    }
    return true;
  }
};
}}  // namespace pybind11::detail

// A packed chunk's tokens, positions and slots: positions [begin, end) of each sequence, one behind the other.
static py::tuple chunk_inputs(BlockManager& bm, const std::vector<int64_t>& ids, const std::vector<int>& begin, const std::vector<int>& end) {
  if (begin.size() != ids.size() || end.size() != ids.size()) throw std::invalid_argument("ids / begin / end size mismatch");
  int64_t T = 0;
  for (size_t i = 0; i < ids.size(); ++i) T += std::max(0, end[i] - begin[i]);
  py::array_t<int32_t> tok(T), pos(T), slot(T);
  int64_t at = 0;
  for (size_t i = 0; i < ids.size(); ++i) {
    bm.inputs(ids[i], begin[i], end[i], tok.mutable_data() + at, pos.mutable_data() + at, slot.mutable_data() + at);
    at += end[i] - begin[i];
  }
  return py::make_tuple(tok, pos, slot);
}

PYBIND11_MODULE(_runtime, m) {
  m.doc() = "distributed_llm_amd native serving runtime (paged-KV block manager, word tokenizer)";
  m.def("pack_words", &pack_words, py::arg("texts"), py::arg("max_len"), py::arg("vocab"), py::arg("other"));
  py::class_<BlockManager>(m, "BlockManager")
      .def(py::init<int, int, bool, int>(), py::arg("num_blocks"), py::arg("block_size") = 16,
           py::arg("prefix_cache") = true, py::arg("placement") = 2)
      .def_property_readonly("block_size", &BlockManager::block_size)
      .def_property_readonly("num_blocks", &BlockManager::num_blocks)
      .def("num_free_blocks", &BlockManager::num_free_blocks)
      .def("num_cached_blocks", &BlockManager::num_cached_blocks)
      .def("has_seq", &BlockManager::has_seq)
      .def("can_allocate", &BlockManager::can_allocate)
      .def("allocate", [](BlockManager& b, int64_t id, const PlainInts& t) { return b.allocate(id, t.v); })
      .def("allocate", &BlockManager::allocate)
      .def("append_token", &BlockManager::append_token)
      .def("slots", &BlockManager::slots)
      .def("chunk_inputs", &chunk_inputs)
      .def("commit_append", &BlockManager::commit_append)
      .def("set_last_tokens", &BlockManager::set_last_tokens)
      .def("commit", &BlockManager::commit)
      .def("block_table", &BlockManager::block_table)
      .def("seq_len", &BlockManager::seq_len)
      .def("committed", &BlockManager::committed)
      .def("free", &BlockManager::free)
      .def("reset", &BlockManager::reset)
      .def("stats", [](const BlockManager& b) {
        py::dict d;
        for (const auto& kv : b.stats()) d[kv.first.c_str()] = kv.second;
        return d;
      })
      .def("check_invariants", &BlockManager::check_invariants);
}
