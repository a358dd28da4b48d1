// Runs the kernels of the message layers' pair sums by themselves on small random problems and compares every value with the
// same sums in fp64 on the host:
//
//   pair_kernels fwd|bwd 64|32 <lmax + 1>
//   pair_kernels compare <value> <wanted value> <bound>     the comparison itself, on the host
//
// Sizes: channels that fill a wave, half a wave, or part of one; slots that leave the last wave partly empty; atoms with no bond,
// fewer and more bonds than a chunk; a radial row per bond and per pair of atoms; launches that count as few and as many waves;
// adjoints for every slot (GRACE-3L) and for all but the last (GRACE-2L), with values behind them that have to stay.
// Bound of a value: (longest chain of additions) eps (sum of the absolute terms).  Prints the worst ratio of difference to bound,
// 1e300 where a difference is no number or a value without a bound differs.
#include "kernel_program.hpp"

#include <cstring>

template<class T> struct Problem {
  int natoms, nslot, C, nl, nlm, noutp, ystr;
  std::vector<long long> eoff;
  std::vector<int> ej, erow;
  std::vector<T> Y, R, dR, M, gP;
  Problem(int natoms_, int nslot_, int C_, int nl_, bool pairs)
      : natoms(natoms_), nslot(nslot_), C(C_), nl(nl_), nlm(nl_ * nl_), noutp(nl_ * C_), ystr(pair_row_stride(nl_ * nl_, sizeof(T)))
  {
    const int bonds[] = {17, 0, 16, 1, 33, 2, 15, 5, 3};
    eoff.push_back(0);
    for (int i = 0; i < natoms; i++) {
      for (int b = 0; b < bonds[i % 9]; b++) ej.push_back((i + 1 + b) % natoms);
      eoff.push_back((long long) ej.size());
    }
    const size_t E = ej.size();
    if (pairs)
      for (size_t e = 0; e < E; e++) erow.push_back((int) ((e * 7 + 3) % E));
    Y = randoms<T>((E + 1) * ystr);
    for (size_t e = 0; e < E; e++) {
      Y[e * ystr] = (T) 0.28209479177387814;    // l = 0: a constant without gradient
      Y[e * ystr + nlm] = Y[e * ystr + 2 * nlm] = (T) 0;
      for (int q = 3 * nlm; q < ystr; q++) Y[e * ystr + q] = (T) 0;
    }
    R = randoms<T>((E + 1) * noutp);
    dR = randoms<T>((E + 1) * noutp);
    M = randoms<T>((size_t) natoms * nslot * C);
    gP = randoms<T>((size_t) natoms * nslot * nlm * C);
  }
  size_t row(size_t e) const { return erow.empty() ? e : (size_t) erow[e]; }
};

static double worst = 0.0;
static void compare(double got, double want, double bound)
{
  const double d = std::fabs(got - want), ratio = bound > 0 ? d / bound : d == 0 ? 0.0 : 1e300;
  if (!(ratio <= worst)) worst = ratio <= 1e300 ? ratio : 1e300;    // not a number: neither comparison holds
}

template<class T> static void run_fwd(const Problem<T> &p, int simds)
{
  const double eps = sizeof(T) == 4 ? 1.1920929e-7 : 2.220446049250313e-16;
  long long *eoff = upload(p.eoff);
  int *ej = upload(p.ej), *erow = p.erow.empty() ? nullptr : upload(p.erow);
  T *Y = upload(p.Y), *R = upload(p.R), *M = upload(p.M);
  const size_t nP = (size_t) p.natoms * p.nslot * p.nlm * p.C;
  T *P = upload(std::vector<T>(nP, (T) 77));
  PairFwdArgs<T> a{};
  a.eoff = eoff; a.ej = ej; a.erow = erow; a.Y = Y; a.R1 = R; a.M = M; a.P = P;
  a.nslot = p.nslot; a.C = p.C; a.noutp = p.noutp; a.ystride = p.ystr; a.natoms = p.natoms;
  launch_pair_fwd<T>(a, p.nl, simds, 0);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipDeviceSynchronize());
  const std::vector<T> got = download(P, nP);
  for (int i = 0; i < p.natoms; i++)
    for (int s = 0; s < p.nslot; s++)
      for (int l = 0, f = 0; l < p.nl; l++)
        for (int m = 0; m < 2 * l + 1; m++, f++)
          for (int n = 0; n < p.C; n++) {
            double sum = 0.0, mag = 0.0;
            for (long long e = p.eoff[i]; e < p.eoff[i + 1]; e++) {
              const double t = (double) p.Y[e * p.ystr + f] * (double) p.R[p.row(e) * p.noutp + l * p.C + n] *
                               (double) p.M[((size_t) p.ej[e] * p.nslot + s) * p.C + n];
              sum += t;
              mag += std::fabs(t);
            }
            compare((double) got[(((size_t) i * p.nslot + s) * p.nlm + f) * p.C + n], sum, eps * (double) (p.eoff[i + 1] - p.eoff[i] + 2) * mag);
          }
  for (void *q : {(void *) eoff, (void *) ej, (void *) erow, (void *) Y, (void *) R, (void *) M, (void *) P})
    if (q) HIP_CHECK(hipFree(q));
}

// nI: slots that have an adjoint
template<class T> static void run_bwd(const Problem<T> &p, const int *drow, int nI)
{
  const double eps = sizeof(T) == 4 ? 1.1920929e-7 : 2.220446049250313e-16;
  const PairMfmaPlan plan = pair_mfma_plan(p.nslot, p.C, p.nl, sizeof(T), pair_mfma_waves(0));
  if (!plan.ok || plan.ystr != p.ystr) throw Error("no plan");
  const size_t E = p.ej.size(), nM = (size_t) p.natoms * nI * p.C;
  long long *eoff = upload(p.eoff);
  int *ej = upload(p.ej), *erow = p.erow.empty() ? nullptr : upload(p.erow);
  T *Y = upload(p.Y), *R = upload(p.R), *dR = upload(p.dR), *M = upload(p.M), *gP = upload(p.gP), *gM = nullptr;
  {
    std::vector<T> zeros(nM, (T) 0);
    zeros.resize(nM + p.C, (T) 3);    // what a slot without an adjoint would add to behind the last atom
    gM = upload(zeros);
  }
  double *bsum = upload(std::vector<double>(3 * E, 0.0));
  PairMfmaArgs<T> a{};
  a.eoff = eoff; a.ej = ej; a.erow = erow; a.YG = Y; a.R1 = R; a.dR1 = dR; a.M = M; a.gP = gP; a.gM = gM; a.bsum = bsum;
  a.nslot = p.nslot; a.nI = nI; a.C = p.C; a.noutp = p.noutp; a.natoms = p.natoms;
  for (int q = 0; q < 16; q++) a.drow[q] = drow[q];
  launch_pair_bwd_mfma<T, true>(plan, a, p.nl, 0);
  HIP_CHECK(hipGetLastError());
  HIP_CHECK(hipDeviceSynchronize());
  const std::vector<T> gotM = download(gM, nM + p.C);
  const std::vector<double> gotB = download(bsum, 3 * E);
  std::vector<double> wantM(nM, 0.0), magM(nM, 0.0), wantB(3 * E, 0.0), magB(3 * E, 0.0);
  for (int i = 0; i < p.natoms; i++)
    for (long long e = p.eoff[i]; e < p.eoff[i + 1]; e++)
      for (int s = 0; s < p.nslot; s++)
        for (int l = 0, f = 0; l < p.nl; l++)
          for (int m = 0; m < 2 * l + 1; m++, f++)
            for (int n = 0; n < p.C; n++) {
              const double g = p.gP[(((size_t) i * p.nslot + s) * p.nlm + f) * p.C + n], r = p.R[p.row(e) * p.noutp + l * p.C + n],
                           d = p.dR[p.row(e) * p.noutp + l * p.C + n];
              const size_t jm = ((size_t) p.ej[e] * nI + s) * p.C + n;
              const double mv = p.M[((size_t) p.ej[e] * p.nslot + s) * p.C + n];
              const double y = p.Y[e * p.ystr + f], y1 = p.Y[e * p.ystr + p.nlm + f], y2 = p.Y[e * p.ystr + 2 * p.nlm + f];
              const double t[4] = {g * r * y, g * d * y * mv, g * r * y1 * mv, g * r * y2 * mv};
              if (s < nI) {
                wantM[jm] += t[0];
                magM[jm] += std::fabs(t[0]);
              }
              for (int k = 0; k < 3; k++) {
                wantB[3 * e + k] += t[k + 1];
                magB[3 * e + k] += std::fabs(t[k + 1]);
              }
            }
  // additions a value goes through: the functions of an l, the l, the slots of a wave; then the bonds of a target, or lanes and waves
  const double chain = p.nlm + p.nl + 4.0;
  std::vector<int> into(p.natoms, 0);
  for (int j : p.ej) into[j]++;
  for (size_t q = 0; q < nM; q++) compare((double) gotM[q], wantM[q], eps * (chain + into[q / ((size_t) nI * p.C)]) * magM[q]);
  for (int n = 0; n < p.C; n++) compare((double) gotM[nM + n], 3.0, 0.0);
  for (size_t q = 0; q < 3 * E; q++) compare(gotB[q], wantB[q], eps * (chain + p.nslot + p.C) * magB[q]);
  for (void *q : {(void *) eoff, (void *) ej, (void *) erow, (void *) Y, (void *) R, (void *) dR, (void *) M, (void *) gP, (void *) gM, (void *) bsum})
    if (q) HIP_CHECK(hipFree(q));
}

template<class T> static void run(bool fwd, int nl)
{
  int drow[16];
  probe<T>(drow);
  for (int C : {16, 32, 48, 64, 80})
    for (int nslot : {1, 2, 5, 7})
      for (int natoms : {1, 10})
        for (int pairs = 0; pairs < 2; pairs++) {
          if (C == 80 && natoms > 1 && nslot > 2) continue;    // the host's sums
          const Problem<T> p(natoms, nslot, C, nl, pairs != 0);
          if (fwd) for (int simds : {1, 1 << 20}) run_fwd<T>(p, simds);
          else for (int nI = std::max(1, nslot - 1); nI <= nslot; nI++) run_bwd<T>(p, drow, nI);
        }
}

int main(int argc, char **argv)
{
  if (argc == 5 && std::strcmp(argv[1], "compare") == 0) {
    compare(std::atof(argv[2]), std::atof(argv[3]), std::atof(argv[4]));
    std::printf("%.6g\n", worst);
    return 0;
  }
  if (argc != 4) {
    std::fprintf(stderr, "usage: pair_kernels fwd|bwd 64|32 <lmax + 1>\n       pair_kernels compare <value> <wanted value> <bound>\n");
    return 2;
  }
  try {
    const bool fwd = std::strcmp(argv[1], "fwd") == 0;
    const int nl = std::atoi(argv[3]);
    if (nl < 1 || nl > 7) throw Error("lmax + 1 out of range");
    if (std::atoi(argv[2]) == 64) run<double>(fwd, nl);
    else run<float>(fwd, nl);
  } catch (const std::exception &e) {
    std::fprintf(stderr, "%s\n", e.what());
    return 1;
  }
  std::printf("%.6g\n", worst);
  return 0;
}
