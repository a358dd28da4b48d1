// What the programs that run kernels by themselves share: errors, buffers, random numbers, the layout of the matrix instructions.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <stdexcept>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

struct Error : std::runtime_error {
  using std::runtime_error::runtime_error;
};
#define HIP_CHECK(expr)                                                                         \
  do {                                                                                          \
    const hipError_t err_ = (expr);                                                             \
    if (err_ != hipSuccess) throw Error(std::string(#expr) + ": " + hipGetErrorString(err_));   \
  } while (0)
#include "../grace_runtime_amd/csrc/kernels_2l.hpp"

using namespace grhip;

template<class U> static U *upload(const std::vector<U> &v)
{
  U *p = nullptr;
  HIP_CHECK(hipMalloc(&p, std::max<size_t>(v.size(), 1) * sizeof(U)));
  if (!v.empty()) HIP_CHECK(hipMemcpy(p, v.data(), v.size() * sizeof(U), hipMemcpyHostToDevice));
  return p;
}
template<class U> static std::vector<U> download(const U *p, size_t n)
{
  std::vector<U> v(n);
  if (n) HIP_CHECK(hipMemcpy(v.data(), p, n * sizeof(U), hipMemcpyDeviceToHost));
  return v;
}

static unsigned long long state = 1;
static double uniform()    // in [-1, 1)
{
  state = state * 6364136223846793005ull + 1442695040888963407ull;
  return (double) (state >> 11) / 4503599627370496.0 - 1.0;
}
template<class T> static std::vector<T> randoms(size_t n)
{
  std::vector<T> v(n);
  for (T &x : v) x = (T) uniform();
  return v;
}

// accumulator row of (lane / 16, register) of a 16x16x4 MFMA, from the product of rows 0 .. 15 with ones
template<class T> static void probe(int *drow)
{
  std::vector<T> A(64, (T) 0), B(64, (T) 0);
  for (int q = 0; q < 16; q++) {
    A[4 * q] = (T) q;    // k = 0 alone
    B[q] = (T) 1;
  }
  T *dA = upload(A), *dB = upload(B), *dD = upload(std::vector<T>(256, (T) -1));
  hipLaunchKernelGGL(k_mfma_probe<T>, dim3(1), dim3(64), 0, 0, dA, dB, dD);
  HIP_CHECK(hipDeviceSynchronize());
  const std::vector<T> D = download(dD, 256);
  for (int g = 0; g < 4; g++)
    for (int v = 0; v < 4; v++) drow[4 * g + v] = (int) D[(16 * g) * 4 + v];
  for (void *p : {(void *) dA, (void *) dB, (void *) dD}) HIP_CHECK(hipFree(p));
}
