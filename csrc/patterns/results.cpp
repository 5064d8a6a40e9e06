// Verified hits of a batch -> its AnalysisResult objects: scoring, the queries for context windows, decoding, and the pydantic
// models, without a Python object in between. What bounds it: the interpreter's allocations, a dozen per result and eleven per event (a
// batch of 64 logs with 192 events took 790 us in Python, from the hits on).
#include <pybind11/numpy.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include <chrono>
#include <ctime>
#include <memory>

#include "lines.h"
#include "scorer.h"

namespace py = pybind11;

namespace {

py::object steal(PyObject* o) {
  if (!o) throw py::error_already_set();
  return py::reinterpret_steal<py::object>(o);
}

py::str name(const char* s) { return py::reinterpret_steal<py::str>(PyUnicode_InternFromString(s)); }

void put(const py::object& dict, const py::object& key, const py::object& value) {
  if (PyDict_SetItem(dict.ptr(), key.ptr(), value.ptr()) != 0) throw py::error_already_set();
}

// Lets go of the interpreter's lock every 8 ms: 51200 events of 1024 logs take 130 ms and more here, which kept every other thread waiting
// to the end. A thread that waits asks for the lock after 5 ms (the interpreter's default), and a lock that was asked for is not taken back before
// the other had it; let go more often it would be, before that thread is awake, and its 5 ms would start again. The clock is read every 64 times,
// about 0.3 ms: read for every event it was 4 % of a batch of 64 logs.
class Turns {
 public:
  void operator()() {
    if (++count_ % 64) return;
    const auto now = std::chrono::steady_clock::now();
    if (count_ == 64) last_ = now;
    if (now - last_ < std::chrono::milliseconds(8)) return;
    { py::gil_scoped_release others; }
    last_ = std::chrono::steady_clock::now();
  }

 private:
  uint32_t count_ = 0;
  std::chrono::steady_clock::time_point last_;
};

py::object number(int64_t v) { return steal(PyLong_FromLongLong(v)); }

// A pydantic model from a complete dict of its fields, as match.py _mk makes it: all fields set, no extras.
class Model {
 public:
  Model(py::type cls, py::object fields)
      : cls_(std::move(cls)), fields_(std::move(fields)), none_(py::tuple(0)), dict_(name("__dict__")), set_(name("__pydantic_fields_set__")),
        extra_(name("__pydantic_extra__")), private_(name("__pydantic_private__")) {}

  py::object make(const py::object& values) const {
    auto* t = reinterpret_cast<PyTypeObject*>(cls_.ptr());
    py::object m = steal(t->tp_new(t, none_.ptr(), nullptr));
    slot(m, dict_, values);
    slot(m, set_, steal(PySet_New(fields_.ptr())));
    slot(m, extra_, steal(PyDict_New()));
    slot(m, private_, py::none());
    return m;
  }

 private:
  static void slot(const py::object& m, const py::str& key, const py::object& v) {
    if (PyObject_GenericSetAttr(m.ptr(), key.ptr(), v.ptr()) != 0) throw py::error_already_set();
  }

  py::type cls_;
  py::object fields_, none_;
  py::str dict_, set_, extra_, private_;
};

struct Pattern {
  int64_t context_lines;
  int rank;
  py::object matched, remediation;
};

// What an engine's results share.
struct ResultTables {
  ResultTables(py::object scorer_, const std::vector<int64_t>& context_lines, const std::vector<int64_t>& ranks, const py::list& matched,
               const py::list& remediation, const std::vector<py::str>& severities_, py::type event, py::object event_fields, py::type summary,
               py::object summary_fields, py::type result, py::object result_fields, py::str engine_)
      : keep(std::move(scorer_)), scorer(keep.cast<const Scorer&>()), severities(severities_), event(std::move(event), std::move(event_fields)),
        summary(std::move(summary), std::move(summary_fields)), result(std::move(result), std::move(result_fields)), engine(std::move(engine_)),
        round_(py::type::of(py::float_(0.0)).attr("__round__")) {
    const size_t n = context_lines.size();
    if (n < scorer.patterns() || ranks.size() != n || matched.size() != n || remediation.size() != n)
      throw std::invalid_argument("ResultTables: a row per pattern");
    for (size_t i = 0; i < n; ++i) {
      if (ranks[i] < 0 || ranks[i] >= (int64_t)severities.size()) throw std::out_of_range("ResultTables: severity rank");
      patterns.push_back({context_lines[i], (int)ranks[i], matched[i], remediation[i]});
    }
  }

  py::object rounded(double v, const py::object& digits) const {
    PyObject* args[2] = {nullptr, digits.ptr()};
    const py::float_ f(v);
    args[0] = f.ptr();
    return steal(PyObject_Vectorcall(round_.ptr(), args, 2, nullptr));
  }

  py::object keep;
  const Scorer& scorer;
  std::vector<Pattern> patterns;
  std::vector<py::str> severities;
  Model event, summary, result;
  py::str engine;
  py::object round_;
  py::object three = py::int_(3), six = py::int_(6);
  py::str line_number = name("line_number"), matched_pattern = name("matched_pattern"), score = name("score"), context = name("context"),
          matched_line = name("matched_line"), remediation = name("remediation"), highest = name("highest_severity"),
          significant = name("significant_events"), total = name("total_events"), distribution = name("severity_distribution"),
          analysis_id = name("analysis_id"), pod_name = name("pod_name"), pod_namespace = name("pod_namespace"), events = name("events"),
          summary_key = name("summary"), metadata = name("metadata"), engine_key = name("engine"), checked = name("patternsChecked"),
          lines = name("totalLines"), bytes = name("bytes"), took = name("processingTimeMs");
};

int64_t newlines_of(std::string_view d) {
  int64_t n = 0;
  for (size_t a = line_end(d, 0); a < d.size(); a = line_end(d, a + 1)) ++n;
  return n;
}

// version 4 UUID of 16 random bytes
py::object uuid4(const uint8_t* r) {
  static const char hex[] = "0123456789abcdef";
  char s[36];
  int at = 0;
  for (int i = 0; i < 16; ++i) {
    const uint8_t b = i == 6 ? (r[i] & 0x0f) | 0x40 : i == 8 ? (r[i] & 0x3f) | 0x80 : r[i];
    if (i == 4 || i == 6 || i == 8 || i == 10) s[at++] = '-';
    s[at++] = hex[b >> 4];
    s[at++] = hex[b & 15];
  }
  return steal(PyUnicode_FromStringAndSize(s, 36));
}

// One batch: scored when it is made; its context windows are set once, then each result is built on its own.
class ResultBatch {
 public:
  // hits [n, 4] = (doc, matcher, line, byte offset); random: 16 bytes per doc
  ResultBatch(py::object tables, const py::list& docs, py::array_t<int64_t, py::array::c_style | py::array::forcecast> hits, int64_t max_events,
              double significance, py::bytes random)
      : keep_(std::move(tables)), t_(keep_.cast<const ResultTables&>()), docs_(steal(PyList_GetSlice(docs.ptr(), 0, (Py_ssize_t)docs.size()))),
        random_(std::move(random)) {
    if (hits.ndim() != 2 || hits.shape(1) != 4) throw std::invalid_argument("ResultBatch: hits [n, 4]");
    for (py::handle d : docs_)
      if (!PyBytes_Check(d.ptr())) throw py::type_error("ResultBatch: docs are bytes");
    if (view(random_).size() < 16 * docs_.size()) throw std::invalid_argument("ResultBatch: 16 random bytes per doc");
    const int64_t *h = hits.data(), num_hits = hits.shape(0), num_docs = (int64_t)docs_.size();
    py::gil_scoped_release others;
    const auto all = t_.scorer.events(h, num_hits, 4, num_docs);
    logs_.resize(all.size());
    for (size_t d = 0; d < all.size(); ++d) {
      Log& g = logs_[d];
      g.counts.assign(t_.severities.size(), 0);
      g.total = all[d].size();
      for (const auto& e : all[d]) {
        ++g.counts[t_.patterns[e.pat].rank];
        g.significant += e.score >= significance;
      }
      g.first = events_.size();
      // as a slice [:max_events] takes them
      const int64_t n = (int64_t)g.total, keep = max_events < 0 ? std::max<int64_t>(0, n + max_events) : std::min(n, max_events);
      for (int64_t i = 0; i < keep; ++i)
        events_.push_back({all[d][i], d, std::max<int64_t>(0, h[4 * all[d][i].at + 3])});
    }
  }

  // [n, 3] = (doc, byte offset, context lines) of every reported event
  py::array_t<int64_t> queries() const {
    py::array_t<int64_t> q({(py::ssize_t)events_.size(), (py::ssize_t)3});
    int64_t* p = q.mutable_data();
    for (const auto& e : events_) {
      *p++ = (int64_t)e.doc;
      *p++ = e.offset;
      *p++ = t_.patterns[e.ev.pat].context_lines;
    }
    return q;
  }

  // The context windows, located here or given: spans [n, 4] = (window start, end, line start, end) within their docs.
  void windows(const py::object& given) {
    py::array_t<int64_t, py::array::c_style | py::array::forcecast> spans;
    if (!given.is_none()) {
      spans = given;
      if (spans.ndim() != 2 || spans.shape(1) != 4 || (size_t)spans.shape(0) < events_.size()) throw std::invalid_argument("windows: spans [n, 4]");
    }
    auto where = [&](size_t i) -> Window {
      const auto d = view(docs_[events_[i].doc]);
      if (given.is_none()) return window(d, (size_t)events_[i].offset, t_.patterns[events_[i].ev.pat].context_lines);
      const int64_t* r = spans.data() + 4 * i;
      if (r[0] < 0 || r[0] > r[2] || r[2] > r[3] || r[3] > r[1] || r[1] > (int64_t)d.size())
        throw std::out_of_range("windows: span outside its document");
      return {(size_t)r[0], (size_t)r[1], (size_t)r[2], (size_t)r[3]};
    };
    std::vector<std::pair<py::list, py::object>> text;
    text.reserve(events_.size());
    Turns turns;
    for (size_t i = 0; i < events_.size(); ++i) {
      text.push_back(window_lines(view(docs_[events_[i].doc]), where(i)));
      turns();
    }
    text_ = std::move(text);
  }

  // Result i: newlines of its log (< 0: counted here), processing time in ms.
  py::object build(size_t i, const py::object& pod_name, const py::object& pod_namespace, int64_t newlines, double ms) const {
    Turns turns;
    return build(i, pod_name, pod_namespace, newlines, ms, turns);
  }

  py::object build(size_t i, const py::object& pod_name, const py::object& pod_namespace, int64_t newlines, double ms, Turns& turns) const {
    if (i >= logs_.size()) throw py::index_error("ResultBatch: doc");
    if (text_.size() != events_.size()) throw std::runtime_error("ResultBatch: the context windows come first");
    const Log& g = logs_[i];
    const auto doc = view(docs_[i]);
    const size_t n = (i + 1 < logs_.size() ? logs_[i + 1].first : events_.size()) - g.first;
    py::list events;
    for (size_t j = 0; j < n; ++j) {
      const Event& e = events_[g.first + j];
      const Pattern& p = t_.patterns[e.ev.pat];
      py::dict d;
      put(d, t_.line_number, number(e.ev.line + 1));
      put(d, t_.matched_pattern, p.matched);
      put(d, t_.score, t_.rounded(e.ev.score, t_.six));
      put(d, t_.context, text_[g.first + j].first);
      put(d, t_.matched_line, text_[g.first + j].second);
      put(d, t_.remediation, p.remediation);
      events.append(t_.event.make(d));
      turns();
    }
    py::dict share, s, meta, r;
    py::object highest = py::none();
    for (size_t k = 0; k < g.counts.size(); ++k) {
      if (!g.counts[k]) continue;
      put(share, t_.severities[k], number(g.counts[k]));
      highest = t_.severities[k];
    }
    put(s, t_.highest, highest);
    put(s, t_.significant, number(g.significant));
    put(s, t_.total, number((int64_t)g.total));
    put(s, t_.distribution, share);
    put(meta, t_.engine_key, t_.engine);
    put(meta, t_.checked, number((int64_t)t_.patterns.size()));
    put(meta, t_.lines, number((newlines < 0 ? newlines_of(doc) : newlines) + 1));
    put(meta, t_.bytes, number((int64_t)doc.size()));
    put(meta, t_.took, t_.rounded(ms, t_.three));
    put(r, t_.analysis_id, uuid4(reinterpret_cast<const uint8_t*>(view(random_).data()) + 16 * i));
    put(r, t_.pod_name, pod_name);
    put(r, t_.pod_namespace, pod_namespace);
    put(r, t_.events, events);
    put(r, t_.summary_key, t_.summary.make(s));
    put(r, t_.metadata, meta);
    return t_.result.make(r);
  }

  // Every result; pods: (name, namespace) per doc or None, newlines: per doc or None, t0: time.perf_counter() at the start.
  py::list build_all(const py::object& pods, const py::object& newlines, double t0) const {
    py::list out;
    Turns turns;
    for (size_t i = 0; i < logs_.size(); ++i) {
      py::object pod_name = py::none(), pod_namespace = py::none();
      if (!pods.is_none()) {
        const py::object pod = pods[py::int_(i)];
        pod_name = pod[py::int_(0)];
        pod_namespace = pod[py::int_(1)];
      }
      timespec now;
      clock_gettime(CLOCK_MONOTONIC, &now);
      const double s = (double)now.tv_sec + 1e-9 * (double)now.tv_nsec;
      out.append(build(i, pod_name, pod_namespace, newlines.is_none() ? -1 : newlines[py::int_(i)].cast<int64_t>(), (s - t0) * 1e3, turns));
      turns();
    }
    return out;
  }

  size_t num_events() const { return events_.size(); }

 private:
  struct Log {
    std::vector<int64_t> counts;
    size_t total = 0, first = 0;
    int64_t significant = 0;
  };
  struct Event {
    Scorer::Ev ev;
    size_t doc;
    int64_t offset;
  };

  py::object keep_;
  const ResultTables& t_;
  py::list docs_;
  py::bytes random_;
  std::vector<Log> logs_;
  std::vector<Event> events_;
  std::vector<std::pair<py::list, py::object>> text_;
};

}  // namespace

void register_results(py::module_& m) {
  py::class_<ResultTables>(m, "ResultTables")
      .def(py::init<py::object, const std::vector<int64_t>&, const std::vector<int64_t>&, const py::list&, const py::list&,
                    const std::vector<py::str>&, py::type, py::object, py::type, py::object, py::type, py::object, py::str>(),
           py::arg("scorer"), py::arg("context_lines"), py::arg("ranks"), py::arg("matched"), py::arg("remediation"), py::arg("severities"),
           py::arg("event"), py::arg("event_fields"), py::arg("summary"), py::arg("summary_fields"), py::arg("result"), py::arg("result_fields"),
           py::arg("engine"));
  py::class_<ResultBatch>(m, "ResultBatch")
      .def(py::init<py::object, const py::list&, py::array_t<int64_t, py::array::c_style | py::array::forcecast>, int64_t, double, py::bytes>(),
           py::arg("tables"), py::arg("docs"), py::arg("hits"), py::arg("max_events"), py::arg("significance"), py::arg("random"))
      .def("queries", &ResultBatch::queries)
      .def("windows", &ResultBatch::windows, py::arg("spans") = py::none())
      .def("build", py::overload_cast<size_t, const py::object&, const py::object&, int64_t, double>(&ResultBatch::build, py::const_), py::arg("doc"), py::arg("pod_name"), py::arg("pod_namespace"), py::arg("newlines"), py::arg("ms"))
      .def("build_all", &ResultBatch::build_all, py::arg("pods"), py::arg("newlines"), py::arg("t0"))
      .def("__len__", &ResultBatch::num_events);
}
