// Host side of k_groups_fwd / k_groups_bwd: a sparse matrix [row][output] as groups of rows and at most kOut outputs with dense
// coefficients.  Rows and outputs that terms join, directly or through others, stay together; parts are joined in the order of
// their smallest row while their outputs fit one group, and a part of more outputs than that is cut by outputs.
#pragma once

#include <algorithm>
#include <cstddef>
#include <numeric>
#include <vector>

namespace grhip {

struct LincombGroups {
  static constexpr int kOut = 6, kJobRows = 32;
  struct Group {
    int t0, t1, t2;          // rows t0 .. t1 with coefficients, t1 .. t2 without any
    int nout, out[kOut];     // outputs, padded with the first
  };
  int nrow = 0, nout = 0;
  std::vector<int> job;      // groups job[k] .. job[k + 1] belong to one wave
  std::vector<Group> group;
  std::vector<int> idx;      // row number; sign bit: an earlier group of the job holds the row too
  std::vector<double> w;     // [row of idx][kOut]
};

// terms: row r, output f, coefficient v; a row's terms in ascending order of outputs.  The rows of a group keep the order in
// which the terms name them first.
inline LincombGroups lincomb_groups(int nrow, int nout, const std::vector<int> &r, const std::vector<int> &f, const std::vector<double> &v)
{
  constexpr int K = LincombGroups::kOut;
  // parts: union-find over rows and outputs
  std::vector<int> up((size_t) nrow + nout);
  std::iota(up.begin(), up.end(), 0);
  auto root = [&](int a) {
    while (up[a] != a) a = up[a] = up[up[a]];
    return a;
  };
  for (size_t t = 0; t < r.size(); t++) up[root(r[t])] = root(nrow + f[t]);
  std::vector<int> number((size_t) nrow + nout, -1);
  struct Part { std::vector<int> rows, outs; };
  std::vector<Part> parts;
  auto part = [&](int a) -> Part & {
    int &q = number[root(a)];
    if (q < 0) { q = (int) parts.size(); parts.emplace_back(); }
    return parts[q];
  };
  std::vector<std::vector<size_t>> terms((size_t) nrow);
  std::vector<int> bare;    // rows without terms
  for (size_t t = 0; t < r.size(); t++) {
    if (terms[r[t]].empty()) part(r[t]).rows.push_back(r[t]);
    terms[r[t]].push_back(t);
  }
  for (int a = 0; a < nrow; a++)
    if (terms[a].empty()) bare.push_back(a);
  for (int b = 0; b < nout; b++) part(nrow + b).outs.push_back(b);

  LincombGroups G;
  G.nrow = nrow;
  G.nout = nout;
  G.job.push_back(0);
  std::vector<char> seen((size_t) nrow, 0);
  size_t next_bare = 0, rows_in_job = 0;
  auto close_job = [&] {
    if ((int) G.group.size() > G.job.back()) G.job.push_back((int) G.group.size());
    rows_in_job = 0;
  };
  // one group: `outs` (at most K) and those of `rows` that have a term there
  auto add = [&](const std::vector<int> &rows, const int *outs, int no, size_t bare_rows) {
    LincombGroups::Group g{};
    g.t0 = (int) G.idx.size();
    g.nout = no;
    for (int k = 0; k < K; k++) g.out[k] = outs[k < no ? k : 0];
    for (int a : rows) {
      double c[K] = {};
      bool any = false;
      for (size_t t : terms[a])
        for (int k = 0; k < no; k++)
          if (f[t] == outs[k]) { c[k] += v[t]; any = true; }
      if (!any) continue;
      G.idx.push_back(seen[a] ? (int) ((unsigned) a | 0x80000000u) : a);
      seen[a] = 1;
      G.w.insert(G.w.end(), c, c + K);
    }
    g.t1 = (int) G.idx.size();
    for (size_t q = 0; q < bare_rows && next_bare < bare.size(); q++) {
      G.idx.push_back(bare[next_bare++]);
      G.w.insert(G.w.end(), K, 0.0);
    }
    g.t2 = (int) G.idx.size();
    rows_in_job += (size_t) (g.t2 - g.t0);
    G.group.push_back(g);
  };
  std::vector<int> rows, outs;
  const size_t bare_each = nout > 0 ? (bare.size() * K + nout - 1) / nout : 0;    // dealt out by the outputs of a group
  auto flush = [&] {
    if (outs.empty()) return;
    add(rows, outs.data(), (int) outs.size(), bare_each);
    rows.clear();
    outs.clear();
    if (rows_in_job >= (size_t) LincombGroups::kJobRows) close_job();
  };
  for (const Part &p : parts) {
    if ((int) (outs.size() + p.outs.size()) > K) flush();
    if ((int) p.outs.size() > K) {
      for (size_t o = 0; o < p.outs.size(); o += K) add(p.rows, p.outs.data() + o, (int) std::min<size_t>(K, p.outs.size() - o), 0);
      close_job();
      continue;
    }
    rows.insert(rows.end(), p.rows.begin(), p.rows.end());
    outs.insert(outs.end(), p.outs.begin(), p.outs.end());
  }
  flush();
  if (next_bare < bare.size() && !G.group.empty()) {    // only after parts that were cut
    LincombGroups::Group g = G.group.back();
    close_job();
    g.t0 = g.t1 = (int) G.idx.size();
    for (; next_bare < bare.size(); next_bare++) {
      G.idx.push_back(bare[next_bare]);
      G.w.insert(G.w.end(), K, 0.0);
    }
    g.t2 = (int) G.idx.size();
    g.nout = 0;
    G.group.push_back(g);
  }
  close_job();
  return G;
}

}    // namespace grhip
