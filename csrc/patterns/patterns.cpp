// Host-side pattern data plane (operator_amd._patterns), CPU only.
//
//  * compile_dfa: literal factors -> Aho-Corasick trie ->
//    complete DFA over case-folded byte equivalence classes, states numbered
//    breadth-first (shallow = hot = first rows, staged in LDS by ac_scan),
//    uint16 table with an "has outputs" flag bit, CSR output lists.
//  * pack_docs: lays a batch of pod logs out for ac_scan (NUL-padded to a
//    multiple of the segment size) and memcpys them into a (pinned) staging
//    buffer with a thread pool, so H2D is one contiguous copy.
//  * score_events: turns verified factor hits
//    into scored events per doc (proximity search of secondary matchers), the
//    same algorithm as operator_amd/patterns/oracle.py.
//
// Replaces the reference's external log-parser (J/service/LogParserClient.java:36-55);
// the pattern schema and scoring are our design.
#include <pybind11/pybind11.h>
#include <pybind11/numpy.h>
#include <pybind11/stl.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <deque>
#include <map>
#include <stdexcept>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>
#if defined(__SSE2__)
#include <emmintrin.h>
#endif

#include "scorer.h"

namespace py = pybind11;

namespace {

constexpr int kMaxFactorLen = 64;
constexpr uint32_t kMaxStates = 32768;

inline uint8_t fold(uint8_t b) { return (b >= 'A' && b <= 'Z') ? uint8_t(b + 32) : b; }

py::dict compile_dfa(const std::vector<std::string>& factors) {
  // ---- byte classes: class 0 = every byte that occurs in no factor ----
  std::array<int, 256> cls{};
  cls.fill(0);
  int nclass = 1;
  for (const auto& f : factors) {
    if (f.empty()) throw std::invalid_argument("empty factor");
    if (f.size() > kMaxFactorLen) throw std::invalid_argument("factor longer than 64 bytes");
    for (unsigned char c : f) {
      if (c == 0 || c == '\n') throw std::invalid_argument("factor contains NUL or newline");
      const uint8_t b = fold(c);
      if (cls[b] == 0) cls[b] = nclass++;
    }
  }
  for (int b = 'A'; b <= 'Z'; ++b) cls[b] = cls[b + 32];
  int log2c = 3;
  while ((1 << log2c) < nclass) ++log2c;
  const int C = 1 << log2c;

  // ---- trie (goto function) ----
  std::vector<std::vector<int32_t>> go;  // [state][class] -> child or -1
  std::vector<std::vector<uint32_t>> own_out;
  std::vector<int> depth;
  go.emplace_back(C, -1);
  own_out.emplace_back();
  depth.push_back(0);
  size_t max_len = 0;
  for (size_t fi = 0; fi < factors.size(); ++fi) {
    int s = 0;
    for (unsigned char c : factors[fi]) {
      const int k = cls[fold(c)];
      if (go[s][k] < 0) {
        go[s][k] = static_cast<int32_t>(go.size());
        go.emplace_back(C, -1);
        own_out.emplace_back();
        depth.push_back(depth[s] + 1);
        if (go.size() > kMaxStates) throw std::length_error("pattern set exceeds 32768 DFA states");
      }
      s = go[s][k];
    }
    own_out[s].push_back(static_cast<uint32_t>(fi));
    max_len = std::max(max_len, factors[fi].size());
  }
  const size_t S = go.size();

  // ---- BFS: failure links, complete transitions, BFS renumbering ----
  std::vector<int32_t> fail(S, 0), order;
  order.reserve(S);
  std::vector<std::vector<int32_t>> delta(S, std::vector<int32_t>(C, 0));
  std::vector<std::vector<uint32_t>> out(S);
  std::deque<int32_t> q;
  order.push_back(0);
  for (int k = 0; k < C; ++k) {
    const int32_t c = go[0][k];
    if (c > 0) { fail[c] = 0; delta[0][k] = c; q.push_back(c); }
    else delta[0][k] = 0;
  }
  out[0] = own_out[0];
  while (!q.empty()) {
    const int32_t s = q.front();
    q.pop_front();
    order.push_back(s);
    out[s] = own_out[s];
    for (uint32_t o : out[fail[s]]) out[s].push_back(o);
    for (int k = 0; k < C; ++k) {
      const int32_t c = go[s][k];
      if (c > 0) {
        fail[c] = delta[fail[s]][k];
        delta[s][k] = c;
        q.push_back(c);
      } else {
        delta[s][k] = delta[fail[s]][k];
      }
    }
  }
  std::vector<uint32_t> rank(S);
  for (size_t i = 0; i < S; ++i) rank[order[i]] = static_cast<uint32_t>(i);

  std::string table(S * C * 2, '\0');
  auto* tab = reinterpret_cast<uint16_t*>(&table[0]);
  std::vector<uint32_t> out_off(S + 1, 0), out_ids;
  std::vector<int> depth_bfs(S);
  for (size_t i = 0; i < S; ++i) {
    const int32_t s = order[i];
    depth_bfs[i] = depth[s];
    for (int k = 0; k < C; ++k) {
      const int32_t n = delta[s][k];
      uint16_t e = static_cast<uint16_t>(rank[n]);
      if (!out[n].empty()) e |= 0x8000;
      tab[i * C + k] = e;
    }
    out_off[i] = static_cast<uint32_t>(out_ids.size());
    std::vector<uint32_t> o = out[s];
    std::sort(o.begin(), o.end());
    o.erase(std::unique(o.begin(), o.end()), o.end());
    out_ids.insert(out_ids.end(), o.begin(), o.end());
  }
  out_off[S] = static_cast<uint32_t>(out_ids.size());

  std::string cls_bytes(256, '\0');
  for (int b = 0; b < 256; ++b) cls_bytes[b] = static_cast<char>(cls[b]);
  py::dict d;
  d["cls_map"] = py::bytes(cls_bytes);
  d["log2_classes"] = log2c;
  d["num_classes_used"] = nclass;
  d["num_states"] = S;
  d["table"] = py::bytes(table);
  d["out_off"] = py::bytes(reinterpret_cast<const char*>(out_off.data()), out_off.size() * 4);
  d["out_ids"] = py::bytes(reinterpret_cast<const char*>(out_ids.data()), std::max<size_t>(out_ids.size(), 1) * 4);
  d["num_out"] = out_ids.size();
  d["max_len"] = max_len;
  d["depth"] = depth_bfs;
  return d;
}

// Profile-guided state numbering for ac_scan's LDS hot set. Breadth-first order
// is only a proxy for "often visited": on log text, 0.4 % of transitions leave
// the first 1024 BFS states, but with 128 chains per wave that puts 42 % of the
// wave's byte steps behind an L2 / Infinity-Cache round trip (measured on the
// 1000-pattern synthetic library). Here the DFA is walked over a sample of the
// text actually being scanned, states are ranked by visit count (root stays 0,
// unvisited states keep BFS order after the visited ones), and the table and
// output lists are permuted. Matches are invariant under renumbering; only the
// hot prefix the kernel stages in LDS changes. Returns the permuted arrays and
// the fraction of sampled transitions that land in the first `hot` states
// before and after.
py::dict reorder_dfa(const std::string& table_b, const std::string& out_off_b, const std::string& out_ids_b,
                     int log2c, int64_t num_states, const std::string& cls_b, const std::string& sample, int hot) {
  const int C = 1 << log2c;
  const int64_t S = num_states;
  if (static_cast<int64_t>(table_b.size()) != S * C * 2) throw std::invalid_argument("table size mismatch");
  if (static_cast<int64_t>(out_off_b.size()) != (S + 1) * 4) throw std::invalid_argument("out_off size mismatch");
  if (cls_b.size() != 256) throw std::invalid_argument("cls_map must have 256 entries");
  const auto* tab = reinterpret_cast<const uint16_t*>(table_b.data());
  const auto* off = reinterpret_cast<const uint32_t*>(out_off_b.data());
  const auto* ids = reinterpret_cast<const uint32_t*>(out_ids_b.data());
  const auto* cls = reinterpret_cast<const uint8_t*>(cls_b.data());
  std::vector<uint64_t> visits(S, 0);
  {
    py::gil_scoped_release nogil;
    uint32_t s = 0;
    for (unsigned char b : sample) {
      s = tab[(static_cast<size_t>(s) << log2c) | cls[b]] & 0x7fffu;
      ++visits[s];
    }
  }
  std::vector<uint32_t> order(S);
  for (int64_t i = 0; i < S; ++i) order[i] = static_cast<uint32_t>(i);
  // root first, then by visits (desc), ties in BFS order (stable)
  std::stable_sort(order.begin() + 1, order.end(), [&](uint32_t a, uint32_t b) { return visits[a] > visits[b]; });
  // The cold states (past the hot prefix) in CHAIN order: a cold excursion is a log
  // line matching a pattern literal, i.e. a walk down one trie path, one dependent
  // global-table read per byte in the kernel's exact re-walk. Numbered so that each
  // state's most-visited trie child (the goto edge: depth + 1) is the next state, the
  // walk follows `dfa_chain` bytes (16 states per 16-byte read) instead of the table.
  // Chains start at the shallowest unplaced state (depth = BFS distance from the root).
  const int64_t H = std::min<int64_t>(std::max(hot, 0), S);
  if (H < S) {
    std::vector<int32_t> depth(S, -1);
    std::vector<uint32_t> bfs;
    bfs.reserve(S);
    depth[0] = 0;
    bfs.push_back(0);
    for (size_t h = 0; h < bfs.size(); ++h) {
      const uint32_t s = bfs[h];
      for (int k = 0; k < C; ++k) {
        const uint32_t t = tab[static_cast<size_t>(s) * C + k] & 0x7fffu;
        if (depth[t] < 0) {
          depth[t] = depth[s] + 1;
          bfs.push_back(t);
        }
      }
    }
    std::vector<char> placed(S, 0);
    for (int64_t i = 0; i < H; ++i) placed[order[i]] = 1;
    std::vector<uint32_t> heads(order.begin() + H, order.end());
    std::stable_sort(heads.begin(), heads.end(), [&](uint32_t a, uint32_t b) { return depth[a] < depth[b]; });
    std::vector<uint32_t> chained(order.begin(), order.begin() + H);
    for (uint32_t h : heads) {
      for (uint32_t s = h; !placed[s];) {
        placed[s] = 1;
        chained.push_back(s);
        int64_t best = -1;
        for (int k = 0; k < C; ++k) {
          const uint32_t t = tab[static_cast<size_t>(s) * C + k] & 0x7fffu;
          if (!placed[t] && depth[t] == depth[s] + 1 && (best < 0 || visits[t] > visits[best])) best = t;
        }
        if (best < 0) break;
        s = static_cast<uint32_t>(best);
      }
    }
    order.swap(chained);
  }
  std::vector<uint32_t> rank(S);
  for (int64_t i = 0; i < S; ++i) rank[order[i]] = static_cast<uint32_t>(i);
  std::string nt(S * C * 2, '\0');
  auto* ntab = reinterpret_cast<uint16_t*>(&nt[0]);
  std::vector<uint32_t> noff(S + 1, 0), nids;
  nids.reserve(off[S]);
  for (int64_t i = 0; i < S; ++i) {
    const uint32_t o = order[i];
    for (int k = 0; k < C; ++k) {
      const uint16_t e = tab[static_cast<size_t>(o) * C + k];
      ntab[i * C + k] = static_cast<uint16_t>(rank[e & 0x7fffu] | (e & 0x8000u));
    }
    noff[i] = static_cast<uint32_t>(nids.size());
    for (uint32_t k = off[o]; k < off[o + 1]; ++k) nids.push_back(ids[k]);
  }
  noff[S] = static_cast<uint32_t>(nids.size());
  uint64_t total = 0, hot_before = 0, hot_after = 0;
  for (int64_t i = 0; i < S; ++i) {
    total += visits[i];
    if (i < hot) hot_before += visits[i];
    if (rank[i] < static_cast<uint32_t>(hot)) hot_after += visits[i];
  }
  py::dict d;
  d["table"] = py::bytes(nt);
  d["out_off"] = py::bytes(reinterpret_cast<const char*>(noff.data()), noff.size() * 4);
  d["out_ids"] = py::bytes(reinterpret_cast<const char*>(nids.data()), std::max<size_t>(nids.size(), 1) * 4);
  d["hot_before"] = total ? double(hot_before) / double(total) : 1.0;
  d["hot_after"] = total ? double(hot_after) / double(total) : 1.0;
  d["sampled"] = total;
  return d;
}

// Per-state chain byte for ac_scan's exact re-walk (csrc/kernels/scan.hip slow_sub):
// chain[s] = 0x40 | k | (0x80 if s + 1 has outputs) when class k takes s to s + 1, else 0.
// Only for <= 64 classes (all zero otherwise: the kernel then reads the table). Padded to
// a multiple of 16 bytes plus 16, so the kernel's aligned 16-byte window reads stay inside.
py::bytes dfa_chain(const std::string& table_b, int log2c, int64_t num_states) {
  const int C = 1 << log2c;
  const int64_t S = num_states;
  if (static_cast<int64_t>(table_b.size()) != S * C * 2) throw std::invalid_argument("table size mismatch");
  const auto* tab = reinterpret_cast<const uint16_t*>(table_b.data());
  std::string ch(static_cast<size_t>((S + 15) / 16 * 16 + 16), '\0');
  if (C <= 64) {
    for (int64_t s = 0; s + 1 < S; ++s)
      for (int k = 0; k < C; ++k) {
        const uint16_t e = tab[static_cast<size_t>(s) * C + k];
        if ((e & 0x7fffu) == static_cast<uint32_t>(s + 1)) {
          ch[s] = static_cast<char>(0x40 | k | ((e & 0x8000u) ? 0x80 : 0));
          break;
        }
      }
  }
  return py::bytes(ch);
}

// Layout: doc i occupies [first_seg[i]*seg, first_seg[i+1]*seg), content then NUL padding (>= 1 byte).
py::tuple plan_docs(const std::vector<size_t>& lens, int64_t seg) {
  if (seg < 64 || (seg & (seg - 1))) throw std::invalid_argument("seg_bytes must be a power of two >= 64");
  std::vector<int64_t> first(lens.size() + 1, 0);
  for (size_t i = 0; i < lens.size(); ++i) {
    const int64_t padded = (static_cast<int64_t>(lens[i]) + 1 + seg - 1) / seg;  // >= 1 NUL byte
    first[i + 1] = first[i] + padded;
  }
  return py::make_tuple(first.back() * seg, first);
}

// n bytes past the caches (dst 16-B aligned): a buffer that only the GPU reads next, without the read that an ordinary
// store makes of the line it replaces.
inline void copy_past_cache(char* d, const char* s, size_t n) {
#if defined(__SSE2__)
  for (; n >= 64; n -= 64, d += 64, s += 64)
    for (int i = 0; i < 64; i += 16)
      _mm_stream_si128(reinterpret_cast<__m128i*>(d + i), _mm_loadu_si128(reinterpret_cast<const __m128i*>(s + i)));
  _mm_sfence();   // before the piece counts as done
#endif
  std::memcpy(d, s, n);
}

// Copies docs into dst (uintptr, >= total bytes) per the plan, zero-filling padding, on `threads` threads, the waiting one
// among them: wait(n) returns once the first n docs are in place, so a caller uploads them while the rest is copied.
// Pieces of at most kPackPiece bytes are taken in order, so a batch of one long log is split too. dst stays valid
// until close() (or the destructor), which ends the copying.
class PackJob {
 public:
  PackJob(std::vector<py::bytes> docs, const std::vector<int64_t>& first, int64_t seg, uintptr_t dst, int threads)
      : docs_(std::move(docs)) {
    if (first.size() != docs_.size() + 1) throw std::invalid_argument("plan/doc count mismatch");
    char* out = reinterpret_cast<char*>(dst);
    size_t total = 0;
    ends_.reserve(docs_.size() + 1);
    ends_.push_back(0);
    for (size_t i = 0; i < docs_.size(); ++i) {
      char* p = nullptr;
      Py_ssize_t n = 0;
      if (PyBytes_AsStringAndSize(docs_[i].ptr(), &p, &n) != 0) throw py::error_already_set();
      const int64_t cap = (first[i + 1] - first[i]) * seg;
      if (static_cast<int64_t>(n) + 1 > cap) throw std::invalid_argument("plan too small");
      char* d = out + first[i] * seg;
      for (int64_t o = 0; o < cap; o += kPackPiece) {
        const int64_t len = std::min(kPackPiece, cap - o), text = std::max<int64_t>(0, std::min<int64_t>(len, n - o));
        pieces_.push_back({d + o, p + (text ? o : 0), static_cast<size_t>(text), static_cast<size_t>(len - text)});
      }
      ends_.push_back(pieces_.size());
      total += static_cast<size_t>(cap);
    }
    past_cache_ = total >= kPastCache && dst % 16 == 0 && seg % 16 == 0;
    done_ = std::vector<std::atomic<uint8_t>>(pieces_.size());
    const int more = std::min<int>(threads, static_cast<int>(pieces_.size())) - 1;
    if (more > 0) pool_.resize(more);
    start(0);
    start(1);
  }
  ~PackJob() { close(); }

  void wait(int64_t n) {
    if (n < 0 || n >= static_cast<int64_t>(ends_.size())) throw std::out_of_range("PackJob.wait: docs");
    py::gil_scoped_release nogil;
    for (const size_t end = ends_[n]; ready_ < end;) {
      if (done_[ready_].load(std::memory_order_acquire)) ++ready_;
      else if (closed_) throw std::runtime_error("PackJob.wait: closed");
      else if (!step()) std::this_thread::yield();   // every piece is taken: some are still being copied
    }
  }

  void close() {
    closed_ = true;
    next_.store(pieces_.size());
    if (pool_.empty()) return;
    py::gil_scoped_release nogil;
    for (auto& th : pool_)   // a thread's own two come behind it
      if (th.joinable()) th.join();
    pool_.clear();
  }

 private:
  struct Piece {
    char* dst;
    const char* src;
    size_t text, zeros;
  };
  static constexpr int64_t kPackPiece = 256 << 10;
  // 84 MB in place on the GPU: 1.9 ms past the caches, 2.1 to 2.3 through them; 4.6 MB the same either way
  static constexpr size_t kPastCache = 8 << 20;

  // Thread t, which starts 2 t + 2 and 2 t + 3 before it copies: one takes 14 us to start, so fifteen of them one behind the other kept the
  // first piece waiting for 220 us.
  void start(size_t t) {
    if (t >= pool_.size()) return;
    try {
      pool_[t] = std::thread([this, t] {
        start(2 * t + 2);
        start(2 * t + 3);
        while (step()) {}
      });
    } catch (const std::exception&) {   // no more threads to be had: those there are, and the waiting one
    }
  }

  bool step() {
    size_t i = next_.load(std::memory_order_relaxed);
    do {
      if (i >= pieces_.size()) return false;
    } while (!next_.compare_exchange_weak(i, i + 1));
    const Piece& p = pieces_[i];
    if (past_cache_) copy_past_cache(p.dst, p.src, p.text);
    else std::memcpy(p.dst, p.src, p.text);
    std::memset(p.dst + p.text, 0, p.zeros);
    done_[i].store(1, std::memory_order_release);
    return true;
  }

  std::vector<py::bytes> docs_;
  std::vector<Piece> pieces_;
  std::vector<size_t> ends_;   // pieces in front of doc i
  std::vector<std::atomic<uint8_t>> done_;
  std::atomic<size_t> next_{0};
  size_t ready_ = 0;           // pieces known to be in place
  bool past_cache_ = false, closed_ = false;
  std::vector<std::thread> pool_;
};

void pack_docs(std::vector<py::bytes> docs, const std::vector<int64_t>& first, int64_t seg, uintptr_t dst, int threads) {
  const int64_t n = static_cast<int64_t>(docs.size());
  PackJob(std::move(docs), first, seg, dst, threads).wait(n);
}

py::list score_events(const std::vector<int64_t>& hit_doc, const std::vector<int64_t>& hit_matcher,
                      const std::vector<int64_t>& hit_line, int64_t num_docs, const std::vector<int64_t>& pat_primary,
                      const std::vector<double>& pat_conf, const std::vector<int64_t>& pat_sev,
                      const std::vector<std::vector<int64_t>>& pat_sec, const std::vector<std::vector<double>>& pat_w,
                      const std::vector<std::vector<int64_t>>& pat_win, int64_t num_matchers) {
  const size_t n = hit_doc.size();
  if (hit_matcher.size() != n || hit_line.size() != n) throw std::invalid_argument("hit arrays differ in length");
  py::array_t<int64_t> hits({(py::ssize_t)n, (py::ssize_t)3});
  int64_t* h = hits.mutable_data();
  for (size_t i = 0; i < n; ++i) {
    h[3 * i] = hit_doc[i];
    h[3 * i + 1] = hit_matcher[i];
    h[3 * i + 2] = hit_line[i];
  }
  return Scorer(pat_primary, pat_conf, pat_sev, pat_sec, pat_w, pat_win, num_matchers).score(hits, num_docs);
}

}  // namespace

void register_verify(py::module_& m);   // verify.cpp (N3 / N4)
void register_results(py::module_& m);  // results.cpp

PYBIND11_MODULE(_patterns, m) {
  m.doc() = "operator_amd host pattern compiler / packer / scorer";
  m.def("compile_dfa", &compile_dfa, py::arg("factors"));
  m.def("dfa_chain", &dfa_chain, py::arg("table"), py::arg("log2_classes"), py::arg("num_states"));
  m.def("reorder_dfa", &reorder_dfa, py::arg("table"), py::arg("out_off"), py::arg("out_ids"), py::arg("log2_classes"),
        py::arg("num_states"), py::arg("cls_map"), py::arg("sample"), py::arg("hot"));
  m.def("plan_docs", &plan_docs, py::arg("lens"), py::arg("seg_bytes"));
  m.def("pack_docs", &pack_docs, py::arg("docs"), py::arg("first_seg"), py::arg("seg_bytes"), py::arg("dst"),
        py::arg("threads") = 8);
  py::class_<PackJob>(m, "PackJob")
      .def(py::init<std::vector<py::bytes>, const std::vector<int64_t>&, int64_t, uintptr_t, int>(), py::arg("docs"),
           py::arg("first_seg"), py::arg("seg_bytes"), py::arg("dst"), py::arg("threads") = 8)
      .def("wait", &PackJob::wait, py::arg("docs"))
      .def("close", &PackJob::close);
  m.def("score_events", &score_events);
  py::class_<Scorer>(m, "Scorer")
      .def(py::init<const std::vector<int64_t>&, std::vector<double>, std::vector<int64_t>, std::vector<std::vector<int64_t>>,
                    std::vector<std::vector<double>>, std::vector<std::vector<int64_t>>, int64_t>(),
           py::arg("primary"), py::arg("conf"), py::arg("severity"), py::arg("secondary"), py::arg("weights"), py::arg("windows"),
           py::arg("num_matchers"))
      .def("score", &Scorer::score, py::arg("hits"), py::arg("num_docs"));
  m.attr("MAX_FACTOR_LEN") = kMaxFactorLen;
  m.attr("MAX_STATES") = kMaxStates;
  register_verify(m);
  register_results(m);
}
