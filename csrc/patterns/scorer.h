// Event scoring on the host (patterns.cpp, results.cpp).
#pragma once

#include <pybind11/numpy.h>
#include <pybind11/pybind11.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <vector>

namespace py = pybind11;

// ---------------------------------------------------------------------------
// Event scoring. Inputs are per-hit arrays (doc, matcher, line) of VERIFIED,
// de-duplicated hits, plus per-pattern matcher tables. Algorithm (our design,
// mirrored exactly by operator_amd/patterns/oracle.py::score_doc):
//   for each primary hit (doc d, line L) of pattern p:
//     bonus = sum_j w_j * (1 - |dL_j| / (W_j + 1))  over secondaries j whose
//             nearest hit in doc d lies within |dL_j| <= W_j
//     score = confidence_p * (1 + bonus) / (1 + sum_j w_j)
// Events are sorted by (score desc, severity desc, doc line asc, pattern asc).
// ---------------------------------------------------------------------------
// A pattern set's scoring tables, kept between batches; score() is the host form of the scorer.
class Scorer {
 public:
  Scorer(const std::vector<int64_t>& primary, std::vector<double> conf, std::vector<int64_t> sev,
         std::vector<std::vector<int64_t>> sec, std::vector<std::vector<double>> w, std::vector<std::vector<int64_t>> win,
         int64_t num_matchers)
      : conf_(std::move(conf)), sev_(std::move(sev)), sec_(std::move(sec)), w_(std::move(w)), win_(std::move(win)), primary_of_(num_matchers) {
    const size_t P = primary.size();
    if (conf_.size() < P || sev_.size() < P || sec_.size() < P || w_.size() < P || win_.size() < P)
      throw std::invalid_argument("pattern tables shorter than the patterns");
    for (size_t p = 0; p < P; ++p) {
      if (primary[p] < 0 || primary[p] >= num_matchers) throw std::out_of_range("pattern primary");
      if (w_[p].size() < sec_[p].size() || win_[p].size() < sec_[p].size()) throw std::invalid_argument("secondary tables too short");
      primary_of_[primary[p]].push_back(static_cast<int>(p));
    }
  }

  struct Ev {
    double score;
    int sev;
    int64_t line;
    int pat;
    int64_t at;   // the hit it comes from
  };

  // hits [n][stride] = (doc, matcher, line, ...) -> per doc its events, best first
  std::vector<std::vector<Ev>> events(const int64_t* h, int64_t n, int stride, int64_t num_docs) const {
    std::vector<std::vector<Hit>> by_doc(num_docs);
    for (int64_t i = 0; i < n; ++i, h += stride) {
      if (h[0] < 0 || h[0] >= num_docs) throw std::out_of_range("hit doc");
      by_doc[h[0]].push_back({h[1], h[2], i});
    }
    std::vector<std::vector<Ev>> all(num_docs);
    for (int64_t d = 0; d < num_docs; ++d) {
      auto& v = by_doc[d];
      auto& evs = all[d];
      std::sort(v.begin(), v.end());
      v.erase(std::unique(v.begin(), v.end(), [](const Hit& a, const Hit& b) { return a.matcher == b.matcher && a.line == b.line; }), v.end());
      for (const auto& hit : v) {
        if (hit.matcher < 0 || hit.matcher >= (int64_t)primary_of_.size()) continue;
        for (int p : primary_of_[hit.matcher]) {
          double bonus = 0.0, wsum = 0.0;
          for (size_t j = 0; j < sec_[p].size(); ++j) {
            const double w = w_[p][j];
            wsum += w;
            const int64_t dist = nearest(v, sec_[p][j], hit.line);
            if (dist >= 0 && dist <= win_[p][j]) bonus += w * (1.0 - double(dist) / double(win_[p][j] + 1));
          }
          evs.push_back({conf_[p] * (1.0 + bonus) / (1.0 + wsum), static_cast<int>(sev_[p]), hit.line, p, hit.at});
        }
      }
      std::sort(evs.begin(), evs.end(), [](const Ev& a, const Ev& b) {
        if (a.score != b.score) return a.score > b.score;
        if (a.sev != b.sev) return a.sev > b.sev;
        if (a.line != b.line) return a.line < b.line;
        return a.pat < b.pat;
      });
    }
    return all;
  }

  size_t patterns() const { return conf_.size(); }

  // hits [n, 3] = (doc, matcher, line) -> per doc its events (pattern, line, score), best first
  py::list score(py::array_t<int64_t, py::array::c_style | py::array::forcecast> hits, int64_t num_docs) const {
    if (hits.ndim() != 2 || hits.shape(1) != 3) throw std::invalid_argument("hits [n, 3]");
    const int64_t *h = hits.data(), n = hits.shape(0);
    std::vector<std::vector<Ev>> all;
    {
      py::gil_scoped_release others;
      all = events(h, n, 3, num_docs);
    }
    py::list result;
    for (const auto& evs : all) {
      py::list dl(evs.size());
      for (size_t i = 0; i < evs.size(); ++i) dl[i] = py::make_tuple(evs[i].pat, evs[i].line, evs[i].score);
      result.append(std::move(dl));
    }
    return result;
  }

 private:
  struct Hit {
    int64_t matcher, line, at;
    bool operator<(const Hit& o) const { return matcher != o.matcher ? matcher < o.matcher : line != o.line ? line < o.line : at < o.at; }
  };

  // distance of the nearest line of matcher m among a doc's sorted hits, or -1
  static int64_t nearest(const std::vector<Hit>& v, int64_t m, int64_t line) {
    auto lo = std::lower_bound(v.begin(), v.end(), Hit{m, line, -1});
    int64_t best = -1;
    if (lo != v.end() && lo->matcher == m) best = lo->line - line;
    if (lo != v.begin()) {
      auto pr = std::prev(lo);
      if (pr->matcher == m) {
        const int64_t dd = line - pr->line;
        if (best < 0 || dd < best) best = dd;
      }
    }
    return best;
  }

  std::vector<double> conf_;
  std::vector<int64_t> sev_;
  std::vector<std::vector<int64_t>> sec_;
  std::vector<std::vector<double>> w_;
  std::vector<std::vector<int64_t>> win_;
  std::vector<std::vector<int>> primary_of_;
};

