// Prints the groups of a sparse matrix read from stdin: "nrow nout nterms", then "row output value" per term.
#include "../grace_runtime_amd/csrc/lincomb_groups.hpp"

#include <cstdio>

int main()
{
  int nrow, nout, nt;
  if (std::scanf("%d %d %d", &nrow, &nout, &nt) != 3) return 1;
  std::vector<int> r(nt), f(nt);
  std::vector<double> v(nt);
  for (int t = 0; t < nt; t++)
    if (std::scanf("%d %d %lf", &r[t], &f[t], &v[t]) != 3) return 1;
  const grhip::LincombGroups g = grhip::lincomb_groups(nrow, nout, r, f, v);
  for (size_t k = 0; k + 1 < g.job.size(); k++)
    for (int q = g.job[k]; q < g.job[k + 1]; q++) {
      const auto &a = g.group[q];
      std::printf("group %zu %d %d %d %d", k, a.t0, a.t1, a.t2, a.nout);
      for (int o : a.out) std::printf(" %d", o);
      std::printf("\n");
    }
  for (size_t t = 0; t < g.idx.size(); t++) {
    std::printf("row %d %d", g.idx[t] & 0x7fffffff, g.idx[t] < 0 ? 1 : 0);
    for (int o = 0; o < g.kOut; o++) std::printf(" %.17g", g.w[t * g.kOut + o]);
    std::printf("\n");
  }
}
