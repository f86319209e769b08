// Byte-level BPE of texts (host).  models/tokenizer.py defines the semantics and
// is the reference; a batch of texts is one call here: the words of a text are
// found in its UTF-8 bytes, a word is merged once and then looked up.
// 64 texts of 68 words: 0.95 ms word by word in Python, 0.12 here, while the GPU
// waits for the tokens.  Runs without a break, as of base64, are words like others:
// 4000 letters 23 ms with every pair looked at after each merge, 0.36 here and 0.11
// from then on; 32,000 2400 ms, 3.1 and 0.8.
#include <torch/extension.h>
#include <pybind11/numpy.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <functional>
#include <queue>
#include <string>
#include <string_view>
#include <vector>

namespace py = pybind11;

namespace {

bool letter(unsigned char c) { return (unsigned)(c | 32) - 'a' < 26u; }
bool digit(unsigned char c) { return (unsigned)c - '0' < 10u; }

// Length in bytes of the white space at s[i], 0 if there is none.  The set is
// that of \s in a Python str pattern.
size_t space(std::string_view s, size_t i) {
  const unsigned char c = s[i];
  if (c < 0x80) return (c >= 9 && c <= 13) || (c >= 0x1c && c <= 0x20) ? 1 : 0;
  const unsigned char d = i + 1 < s.size() ? s[i + 1] : 0;
  if (c == 0xc2) return d == 0x85 || d == 0xa0 ? 2 : 0;       // U+0085, U+00A0
  if (c < 0xe1 || c > 0xe3 || i + 2 >= s.size()) return 0;
  const unsigned p = (c & 15u) << 12 | (d & 63u) << 6 | (s[i + 2] & 63u);
  return p == 0x1680 || (p >= 0x2000 && p <= 0x200a) || p == 0x2028 ||
                 p == 0x2029 || p == 0x202f || p == 0x205f || p == 0x3000
             ? 3 : 0;
}

// End of the word that starts at s[i]:
//   's 't 're 've 'm 'll 'd | ?letters | ?digits | ?others |
//   white space up to the last of it, or alone
size_t word_end(std::string_view s, size_t i) {
  const size_t n = s.size();
  if (s[i] == '\'' && i + 1 < n) {
    const char c = s[i + 1], d = i + 2 < n ? s[i + 2] : 0;
    if (c == 's' || c == 't') return i + 2;
    if ((c == 'r' || c == 'v') && d == 'e') return i + 3;
    if (c == 'm') return i + 2;
    if (c == 'l' && d == 'l') return i + 3;
    if (c == 'd') return i + 2;
  }
  size_t j = i + (s[i] == ' ' && i + 1 < n ? 1 : 0);
  if (letter(s[j])) {
    while (j < n && letter(s[j])) ++j;
    return j;
  }
  if (digit(s[j])) {
    while (j < n && digit(s[j])) ++j;
    return j;
  }
  if (!space(s, j)) {
    while (j < n && !letter(s[j]) && !digit(s[j]) && !space(s, j)) ++j;
    return j;
  }
  size_t last = i;                     // start of the run's last character
  for (j = i; j < n;) {
    const size_t w = space(s, j);
    if (!w) break;
    last = j;
    j += w;
  }
  return j == n || last == i ? j : last;
}

class Bpe {
 public:
  // merges: pairs of symbols, 0..255 bytes and 256 + i what merge i makes;
  // specials: texts that are a token of their own, in order of preference;
  // base: token of byte 0
  Bpe(const py::list& merges,
      std::vector<std::pair<std::string, int>> specials, int base)
      : specials_(std::move(specials)), base_(base) {
    for (const auto& sp : specials_) starts_[(unsigned char)sp.first[0]] = true;
    clear();
    size_t places = 16;
    while (places < 2 * merges.size()) places *= 2;
    merged_.assign(places, {0, 0});
    for (size_t i = 0; i < merges.size(); ++i) {
      PyObject* pair = PyList_GET_ITEM(merges.ptr(), (Py_ssize_t)i);
      if (!PyTuple_Check(pair) || PyTuple_GET_SIZE(pair) != 2)
        throw py::type_error("a merge is a pair of symbols");
      const unsigned long a = PyLong_AsUnsignedLong(PyTuple_GET_ITEM(pair, 0));
      const unsigned long b = PyLong_AsUnsignedLong(PyTuple_GET_ITEM(pair, 1));
      if (PyErr_Occurred()) throw py::error_already_set();
      *find(key((uint32_t)a, (uint32_t)b)) = {
          key((uint32_t)a, (uint32_t)b), 256 + (uint32_t)i};
    }
  }

  py::list encode(const py::str& text, int first) {
    std::vector<int32_t> ids;
    run(text, first, SIZE_MAX, ids);
    py::list out(ids.size());
    for (size_t i = 0; i < ids.size(); ++i) out[i] = py::int_(ids[i]);
    return out;
  }

  // The tokens of all texts one after another and their numbers; at most
  // `longest` of each.
  py::tuple encode_batch(const py::list& texts, int first, size_t longest) {
    std::vector<int32_t> all, ids;
    py::array_t<int64_t> lens((py::ssize_t)texts.size());
    int64_t* len = lens.mutable_data();
    for (const auto& t : texts) {
      ids.clear();
      run(py::cast<py::str>(t), first, longest, ids);
      const size_t n = std::min(ids.size(), longest);
      all.insert(all.end(), ids.begin(), ids.begin() + n);
      *len++ = (int64_t)n;
    }
    py::array_t<int32_t> flat((py::ssize_t)all.size());
    std::memcpy(flat.mutable_data(), all.data(), all.size() * sizeof(int32_t));
    return py::make_tuple(flat, lens);
  }

 private:
  static constexpr size_t kKeep = 65536, kStart = 2048;      // words
  static constexpr size_t kBytes = 16 << 20;                  // of them
  static constexpr size_t kShort = 48;   // up to here every pair is looked at
  struct Merge {
    uint64_t key;                                 // 0: a free place
    uint32_t symbol;
  };
  static uint64_t key(uint32_t a, uint32_t b) {
    return ((uint64_t)a << 32 | b) + 1;
  }

  Merge* find(uint64_t k) {            // its place, or the free one for it
    size_t at = (k * 0x9e3779b97f4a7c15ull >> 32) & (merged_.size() - 1);
    while (merged_[at].key && merged_[at].key != k)
      at = (at + 1) & (merged_.size() - 1);
    return &merged_[at];
  }

  // at least the first `most` tokens of a text, if it has as many
  void run(const py::str& text, int first, size_t most,
           std::vector<int32_t>& ids) {
    Py_ssize_t n = 0;
    const char* p = PyUnicode_AsUTF8AndSize(text.ptr(), &n);
    if (!p) throw py::error_already_set();         // lone surrogates
    const std::string_view s(p, (size_t)n);
    if (first >= 0) ids.push_back(first);
    size_t from = 0;
    for (size_t i = 0; i < s.size();) {
      const std::pair<std::string, int>* hit = nullptr;
      if (starts_[(unsigned char)s[i]])
        for (const auto& sp : specials_)
          if (s.compare(i, sp.first.size(), sp.first) == 0) {
            hit = &sp;
            break;
          }
      if (!hit) {
        ++i;
        continue;
      }
      words(s.substr(from, i - from), most, ids);
      if (ids.size() >= most) return;
      ids.push_back(hit->second);
      from = i += hit->first.size();
    }
    words(s.substr(from), most, ids);
  }

  void words(std::string_view s, size_t most, std::vector<int32_t>& ids) {
    for (size_t i = 0; i < s.size() && ids.size() < most;) {
      const size_t j = word_end(s, i);
      word(s.substr(i, j - i), ids);
      i = j;
    }
  }

  // A word's tokens, once found, stay in an open table of at least twice as many
  // places, which grows up to kKeep words of kBytes.
  void word(std::string_view w, std::vector<int32_t>& ids) {
    const uint64_t h = hash(w);
    size_t at = h & (table_.size() - 1);
    for (; table_[at]; at = (at + 1) & (table_.size() - 1)) {
      const Known& k = known_[table_[at] - 1];
      if (k.hash == h && k.size == w.size() &&
          std::memcmp(bytes_.data() + k.word, w.data(), w.size()) == 0) {
        ids.insert(ids.end(), tokens_.begin() + k.first,
                   tokens_.begin() + k.first + k.count);
        return;
      }
    }
    merge(w);
    ids.insert(ids.end(), syms_.begin(), syms_.end());
    if (w.size() > kBytes) return;
    if (known_.size() >= kKeep || bytes_.size() + w.size() > kBytes) {
      clear();
      at = h & (table_.size() - 1);
    } else if (2 * known_.size() >= table_.size()) {
      grow();
      for (at = h & (table_.size() - 1); table_[at];)
        at = (at + 1) & (table_.size() - 1);
    }
    known_.push_back({h, (uint32_t)bytes_.size(), (uint32_t)w.size(),
                      (uint32_t)tokens_.size(), (uint32_t)syms_.size()});
    table_[at] = (uint32_t)known_.size();
    bytes_.append(w);
    tokens_.insert(tokens_.end(), syms_.begin(), syms_.end());
  }

  static uint64_t hash(std::string_view w) {
    uint64_t h = w.size() * 0x9e3779b97f4a7c15ull;
    for (size_t i = 0; i < w.size(); i += 8) {
      uint64_t x = 0;
      std::memcpy(&x, w.data() + i, std::min<size_t>(8, w.size() - i));
      h = (h ^ x) * 0xff51afd7ed558ccdull;
      h ^= h >> 32;
    }
    return h;
  }

  void grow() {
    table_.assign(2 * table_.size(), 0);
    for (size_t i = 0; i < known_.size(); ++i) {
      size_t at = known_[i].hash & (table_.size() - 1);
      while (table_[at]) at = (at + 1) & (table_.size() - 1);
      table_[at] = 1 + (uint32_t)i;
    }
  }

  void clear() {
    table_.assign(kStart, 0);
    known_.clear();
    bytes_.clear();
    tokens_.clear();
  }

  // leaves the word's tokens in syms_: the pair of lowest rank, the first of
  // equals, until none is left
  __attribute__((noinline)) void merge(std::string_view w) {
    syms_.assign(w.size(), 0);
    for (size_t i = 0; i < w.size(); ++i) syms_[i] = (unsigned char)w[i];
    if (w.size() > kShort) merge_long();
    else merge_short();
    for (auto& x : syms_) x += base_;
  }

  void merge_short() {
    while (syms_.size() > 1) {
      uint32_t best = UINT32_MAX;
      size_t at = 0;
      for (size_t i = 0; i + 1 < syms_.size(); ++i) {
        const Merge* m = find(key(syms_[i], syms_[i + 1]));
        if (m->key && m->symbol < best) {
          best = m->symbol;
          at = i;
        }
      }
      if (best == UINT32_MAX) break;
      syms_[at] = (int32_t)best;
      syms_.erase(syms_.begin() + (std::ptrdiff_t)at + 1);
    }
  }

  // The same order from a heap of the pairs, symbols in a list: n log n, where
  // looking at every pair after each merge is n^2.  A pair whose symbols have
  // changed since is passed over.
  void merge_long() {
    using Pair = std::pair<uint32_t, uint32_t>;           // symbol, place
    const uint32_t n = (uint32_t)syms_.size();
    std::vector<uint32_t> next(n), prev(n);
    std::priority_queue<Pair, std::vector<Pair>, std::greater<Pair>> heap;
    auto made = [&](uint32_t i) {                         // of i and its next
      const Merge* m = find(key(syms_[i], syms_[next[i]]));
      return m->key ? m->symbol : UINT32_MAX;
    };
    auto push = [&](uint32_t i) {
      if (next[i] == n) return;
      const uint32_t s = made(i);
      if (s != UINT32_MAX) heap.push({s, i});
    };
    for (uint32_t i = 0; i < n; ++i) {
      next[i] = i + 1;
      prev[i] = i - 1;
    }
    for (uint32_t i = 0; i < n; ++i) push(i);
    while (!heap.empty()) {
      const auto [s, i] = heap.top();
      heap.pop();
      if (syms_[i] < 0 || next[i] == n || made(i) != s) continue;
      const uint32_t gone = next[i];
      syms_[i] = (int32_t)s;
      syms_[gone] = -1;
      next[i] = next[gone];
      if (next[i] != n) prev[next[i]] = i;
      push(i);
      if (i) push(prev[i]);
    }
    syms_.erase(std::remove(syms_.begin(), syms_.end(), -1), syms_.end());
  }

  std::vector<Merge> merged_;                     // open, half full at most
  struct Known {
    uint64_t hash;
    uint32_t word, size, first, count;            // in bytes_ and tokens_
  };
  std::vector<uint32_t> table_;                   // 1 + place in known_, or 0
  std::vector<Known> known_;
  std::string bytes_;
  std::vector<int32_t> tokens_;
  bool starts_[256] = {};                         // bytes that begin a special
  std::vector<std::pair<std::string, int>> specials_;
  std::vector<int32_t> syms_;
  int base_;
};

}  // namespace

void register_bpe(py::module_& m) {
  py::class_<Bpe>(m, "Bpe")
      .def(py::init<const py::list&,
                    std::vector<std::pair<std::string, int>>, int>())
      .def("encode", &Bpe::encode)
      .def("encode_batch", &Bpe::encode_batch);
}
