// Lines of a log (verify.cpp, results.cpp).
#pragma once

#include <pybind11/pybind11.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string_view>
#include <utility>
#include <vector>

namespace py = pybind11;

inline std::string_view view(py::handle bytes) { return {PyBytes_AS_STRING(bytes.ptr()), (size_t)PyBytes_GET_SIZE(bytes.ptr())}; }

// first byte of the line that ends before `end` (d[end] is its newline, or the end of the log)
inline size_t line_start(std::string_view d, size_t end) {
  const void* p = end > 0 ? memrchr(d.data(), '\n', end) : nullptr;
  return p ? (size_t)(static_cast<const char*>(p) - d.data()) + 1 : 0;
}

inline size_t line_end(std::string_view d, size_t from) {
  const void* p = from < d.size() ? std::memchr(d.data() + from, '\n', d.size() - from) : nullptr;
  return p ? (size_t)(static_cast<const char*>(p) - d.data()) : d.size();
}

inline std::pair<size_t, size_t> line_bounds(std::string_view d, size_t off) {
  off = std::min(off, d.size());
  return {line_start(d, off), line_end(d, off)};
}

// (window start, window end, line start, line end): the line of byte `off` and up to k lines on either side
struct Window {
  size_t from, to, line, line_to;
};

inline Window window(std::string_view d, size_t off, int64_t k) {
  const auto [s, e] = line_bounds(d, off);
  Window w{s, e, s, e};
  for (int64_t j = 0; j < k && w.from > 0; ++j) w.from = line_start(d, w.from - 1);
  for (int64_t j = 0; j < k && w.to + 1 < d.size(); ++j) w.to = line_end(d, w.to + 1);
  return w;
}

inline py::str decode(std::string_view v) {
  PyObject* o = PyUnicode_DecodeUTF8(v.data(), (Py_ssize_t)v.size(), "replace");
  if (!o) throw py::error_already_set();
  return py::reinterpret_steal<py::str>(o);
}

// the window's lines, and its own line among them
inline std::pair<py::list, py::object> window_lines(std::string_view d, const Window& w) {
  size_t n = 1 + std::count(d.data() + w.from, d.data() + w.to, '\n'), a = w.from;
  py::list ctx(n);
  py::object line;
  for (size_t i = 0; i < n; ++i) {
    const size_t b = std::min(line_end(d, a), w.to);
    py::str t = decode(d.substr(a, b - a));
    if (a == w.line && b == w.line_to) line = t;
    ctx[i] = std::move(t);
    a = b + 1;
  }
  if (!line) line = decode(d.substr(w.line, w.line_to - w.line));
  return {std::move(ctx), std::move(line)};
}
