// The species form of the radial network (GRACE-3L), k_radial_few against k_radial: the same sums in the same order, so every bit of
// every row agrees, whatever number of bonds a launch has and wherever its range begins, and no row outside of the range is written.
//
//   radial_kernels 64|32 64|128        precision, hidden width
//
// Prints how many values differ.
#include "kernel_program.hpp"

#include <cstring>

template<class T, int HB> static long long run(int nl, int C)
{
  int drow[16];
  probe<T>(drow);
  const int nrb = 10, ks0 = (nrb + 3) / 4, nel = 3, noutp = nl * C, nob = noutp / 16, H = HB * 16;
  const long long line = (HB == 4 ? 3 : 2) * 256, rows = 16 * line + 40;    // tiles where the engines change over with 256 CUs
  auto weights = [&](size_t n, int inputs) {
    std::vector<T> w = randoms<T>(n);
    for (T &x : w) x *= (T) std::sqrt(3.0 / inputs);
    return w;
  };
  const size_t n0 = (size_t) HB * ks0 * 64, n1 = (size_t) HB * HB * 4 * 64, n2 = ((size_t) nob * HB * 4 + kRadialPrefetch) * 64;
  std::vector<double> x(rows);
  for (double &v : x) v = 0.51 + 0.49 * uniform();
  std::vector<int> mu(rows), mi(rows);
  for (int &v : mu) v = std::min(nel - 1, (int) ((uniform() + 1) * 0.5 * nel));
  for (int &v : mi) v = std::min(nel - 1, (int) ((uniform() + 1) * 0.5 * nel));
  RadialArgs<T> a{};
  T *w0 = upload(weights(n0, nrb)), *w1 = upload(weights(n1, H)), *w2 = upload(weights(n2, H)), *z = upload(randoms<T>((size_t) nel * C)),
    *bi = upload(randoms<T>((size_t) nel * H)), *bj = upload(randoms<T>((size_t) nel * H)), *b1 = upload(randoms<T>(H)), *out[2][2];
  double *dx = upload(x);
  int *dmu = upload(mu), *dmi = upload(mi);
  long long *edges = upload(std::vector<long long>(1, 0));
  a.n_edges = edges;
  a.x = dx; a.emu = dmu; a.emi = dmi; a.w0 = w0; a.w1 = w1; a.w2 = w2; a.z = z; a.bias_i = bi; a.bias_j = bj; a.bias1 = b1;
  a.nrb = nrb; a.p = 6; a.ks0 = ks0; a.nob = nob; a.noutp = noutp; a.C = C; a.nel = nel; a.act = 0;
  for (int q = 0; q < 16; q++) a.drow[q] = drow[q];
  const std::vector<T> untouched((size_t) rows * noutp, (T) 77);
  for (auto &o : out)
    for (T *&p : o) p = upload(untouched);
  const size_t few_lds = (size_t) radial_few_lds(HB) * sizeof(T), base = (n0 + n1) * sizeof(T);
  const bool w2l = base + n2 * sizeof(T) <= 150 * 1024;
  const size_t lds = base + (w2l ? n2 * sizeof(T) : 0);
  a.w2_in_lds = w2l;
  auto whole = w2l ? k_radial<T, HB, 0, 1, true, false> : k_radial<T, HB, 0, 1, false, false>;
  auto few = k_radial_few<T, HB, 0, 1>;
  HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(whole), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(few), hipFuncAttributeMaxDynamicSharedMemorySize, (int) few_lds));
  long long differ = 0;
  for (long long count : {1ll, 15ll, 16ll, 17ll, 255ll, 16 * 256ll + 1, 16 * line - 3, 16 * line})
    for (int listed = 0; listed < 2; listed++) {    // the count as an argument, and on the device with blocks to spare or too few
      a.e_begin = listed ? 0 : 37;
      a.e_count = listed ? -1 : std::min(count, rows - a.e_begin);
      HIP_CHECK(hipMemcpy(edges, &count, sizeof count, hipMemcpyHostToDevice));
      for (auto &o : out)
        for (T *p : o) HIP_CHECK(hipMemcpy(p, untouched.data(), untouched.size() * sizeof(T), hipMemcpyHostToDevice));
      const unsigned blocks = listed ? (count > 300 ? (unsigned) (count / 50) : (unsigned) line) : (unsigned) ((a.e_count + 15) / 16);
      a.Rz = out[0][0]; a.dRz = out[0][1];
      hipLaunchKernelGGL(whole, dim3(256), dim3(radial_threads(HB, 1, w2l)), lds, 0, a);
      HIP_CHECK(hipGetLastError());
      a.Rz = out[1][0]; a.dRz = out[1][1];
      hipLaunchKernelGGL(few, dim3(blocks), dim3(64 * HB), few_lds, 0, a);
      HIP_CHECK(hipGetLastError());
      HIP_CHECK(hipDeviceSynchronize());
      for (int k = 0; k < 2; k++) {
        const std::vector<T> want = download(out[0][k], untouched.size()), got = download(out[1][k], untouched.size());
        for (size_t q = 0; q < want.size(); q++) {
          const long long e = (long long) (q / noutp) - a.e_begin, n = a.e_count < 0 ? count : a.e_count;
          const bool inside = e >= 0 && e < n;
          differ += std::memcmp(&want[q], &got[q], sizeof(T)) != 0 || !std::isfinite(got[q]) || (got[q] == (T) 77) == inside;
        }
      }
    }
  for (void *p : {(void *) w0, (void *) w1, (void *) w2, (void *) z, (void *) bi, (void *) bj, (void *) b1, (void *) dx, (void *) dmu, (void *) dmi,
                  (void *) edges, (void *) out[0][0], (void *) out[0][1], (void *) out[1][0], (void *) out[1][1]})
    HIP_CHECK(hipFree(p));
  return differ;
}

template<class T> static long long widths(int hidden)
{
  // few outputs, whose weights sit in LDS, and those of the GRACE-3L benchmark model (64 channels, lmax 5), which do not
  return hidden == 64 ? run<T, 4>(3, 16) + run<T, 4>(5, 32) : run<T, 8>(5, 16) + run<T, 8>(6, 64);
}

int main(int argc, char **argv)
{
  const int hidden = argc == 3 ? std::atoi(argv[2]) : 0;
  if (hidden != 64 && hidden != 128) {
    std::fprintf(stderr, "usage: radial_kernels 64|32 64|128\n");
    return 2;
  }
  try {
    std::printf("%lld\n", std::atoi(argv[1]) == 64 ? widths<double>(hidden) : widths<float>(hidden));
  } catch (const std::exception &e) {
    std::fprintf(stderr, "%s\n", e.what());
    return 1;
  }
  return 0;
}
