// HIP kernels of the GRACE-1L energy/forces/virial pass for gfx950 (wave64, MFMA).  Included by engine_1l.hip only.
//
// Stage map (reference stages in libgrace/src/fused_1l.cpp:260-372 and the staged pipeline of
// libgrace/include/grace/kk/grace_1l_kk.h:449-454):
//   k_edge_count / k_edge_fill   bond filter r^2 < rc^2, unit vectors, x = r / rc        (bonds.h:120-162)
//   k_radial                     Chebyshev x envelope basis + radial MLP value/tangent on MFMA, times z[mu_j]
//                                (radial_x.h:11-60; spline tables of the CPU path replaced by the exact MLP)
//   k_scatter_a                  A[lm][n] = sum_b Y_lm R_nl z                            (fused_cpu.h:947-982)
//   k_gemm_jobs                  FC forward / reverse as tile GEMMs on MFMA               (fused_cpu.h:349-364)
//   k_prod_fwd / k_prod_bwd      channel-wise CG products                                 (fused_cpu.h:409-475)
//   k_reduce_fwd / k_reduce_bwd  rho reduce with per-element weights                      (fused_cpu.h:637-649)
//   k_energy_hidden, k_energy    fp64 readout MLP and its reverse                         (fused_1l.cpp:378-427)
//   k_bond_bwd                   per-bond force, pair scatter, virial                     (fused_cpu.h:836-860,1027-1050)
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace grhip {

constexpr int kKernMaxL = 6;                                // largest lmax of the kernels
constexpr int kMaxNlm = (kKernMaxL + 1) * (kKernMaxL + 1);
constexpr int kMaxPlm = (kKernMaxL + 1) * (kKernMaxL + 2) / 2;
constexpr int kBondChunk = 32;                          // bonds staged per pass of the per-atom kernels
constexpr int kMaxRadBasis = 16;
constexpr int kRadialPrefetch = 16;                     // weight fragments the radial kernel reads ahead: padding of the layer-2 weights                        // radial basis functions (padded to a multiple of 4)

// spherical-harmonics recursion coefficients (fused_cpu.h:686-704), by index l (l + 1) / 2 + m
struct ShCoef {
  double a[kMaxPlm], b[kMaxPlm], c[kKernMaxL + 1], d[kKernMaxL + 1];
  int lmax;
};

// Real spherical harmonics Y[lm] (stride ys) of the unit vector (rx, ry, rz) and, with GRAD, the gradient
// G[lm][3] of their polynomial extension.  Same recursion as fused_cpu.h:712-798, one bond per thread, fp64.
// LMAX: compile-time bound of co.lmax (the register arrays of the recursion are sized by it).
// With e1, e2 and D2 given, the gradient is stored as its two components along e1 and e2 instead: G[lm] = grad . e1,
// D2[lm] = grad . e2.
template<bool GRAD, class TY, int LMAX = kKernMaxL>
__device__ inline void sh_eval(const ShCoef &co, double rx, double ry, double rz, TY *Y, TY *G, const double *e1 = nullptr,
                               const double *e2 = nullptr, TY *D2 = nullptr)
{
  auto put = [&](int lm, double gx, double gy, double gz) {
    if (e1) {
      G[lm] = (TY) (gx * e1[0] + gy * e1[1] + gz * e1[2]);
      D2[lm] = (TY) (gx * e2[0] + gy * e2[1] + gz * e2[2]);
    } else {
      G[3 * lm] = (TY) gx; G[3 * lm + 1] = (TY) gy; G[3 * lm + 2] = (TY) gz;
    }
  };
  double plm[(LMAX + 1) * (LMAX + 2) / 2], dplm[(LMAX + 1) * (LMAX + 2) / 2];
  const int lmax = co.lmax < LMAX ? co.lmax : LMAX;
  plm[0] = 1.0;
  dplm[0] = 0.0;
  if (LMAX > 0 && lmax > 0) {
    const double s3 = 1.7320508075688772, s15 = -1.224744871391589;
    plm[LMAX > 0 ? 1 : 0] = s3 * rz; dplm[LMAX > 0 ? 1 : 0] = s3;
    plm[LMAX > 0 ? 2 : 0] = s15;     dplm[LMAX > 0 ? 2 : 0] = 0.0;
#pragma unroll
    for (int l = 2; l <= LMAX; l++) {
      if (l <= lmax) {
#pragma unroll
        for (int mm = 0; mm < l - 1; mm++) {
          const int id = l * (l + 1) / 2 + mm, i1 = (l - 1) * l / 2 + mm, i2 = (l - 2) * (l - 1) / 2 + mm;
          const double ca = co.a[id], cb = co.b[id];
          plm[id] = ca * (rz * plm[i1] + cb * plm[i2]);
          if (GRAD) dplm[id] = ca * (plm[i1] + rz * dplm[i1] + cb * dplm[i2]);
        }
        const int prev = (l - 1) * l / 2 + l - 1, i0 = l * (l + 1) / 2 + l - 1, i1 = l * (l + 1) / 2 + l;
        const double sd = co.d[l], sc = co.c[l];
        plm[i0] = sd * plm[prev] * rz;
        plm[i1] = sc * plm[prev];
        if (GRAD) {
          dplm[i0] = sd * (dplm[prev] * rz + plm[prev]);
          dplm[i1] = sc * dplm[prev];
        }
      }
    }
  }
  const double sq2 = 1.4142135623730951;
#pragma unroll
  for (int l = 0; l <= LMAX; l++) {
    if (l <= lmax) {
      const int c = l * (l + 1), p0 = l * (l + 1) / 2;
      Y[c] = (TY) plm[p0];
      if (GRAD) put(c, 0.0, 0.0, dplm[p0]);
      double pr = rx, pi = ry, prx = 1.0, pry = 0.0, pix = 0.0, piy = 1.0;
#pragma unroll
      for (int mm = 1; mm <= l; mm++) {
        const double sg = (mm % 2 == 0) ? sq2 : -sq2;
        const double pv = plm[p0 + mm];
        Y[c + mm] = (TY) (sg * pr * pv);
        Y[c - mm] = (TY) (sg * pi * pv);
        if (GRAD) {
          const double dpv = dplm[p0 + mm];
          put(c + mm, sg * prx * pv, sg * pry * pv, sg * pr * dpv);
          put(c - mm, sg * pix * pv, sg * piy * pv, sg * pi * dpv);
          const double nrx = prx * rx + pr - pix * ry, nry = pry * rx - piy * ry - pi;
          const double nix = prx * ry + pix * rx + pi, niy = pry * ry + pr + piy * rx;
          prx = nrx; pry = nry; pix = nix; piy = niy;
        }
        const double nr = pr * rx - pi * ry, ni = pr * ry + pi * rx;
        pr = nr; pi = ni;
      }
    }
  }
}

// Message rows to and from an exchange buffer (the pack / unpack kernels of the reference's GPU engines,
// libgrace/include/grace/kk/grace_2l_kk.h:141-157): rows[atom][function][CP], of which nf functions x C channels travel
// as doubles; the atoms are list[0 .. n) or first .. first + n.  ADD: the buffer is added to the rows (reverse exchange).
// Else the rows are set whole: the channels C .. CP - 1 of a ghost's row, which no other kernel writes, become zero.  Readers
// multiply them by zero weights, which is not enough where the memory held NaN.
template<class T>
__global__ void k_comm_pack(const T *rows, long long stride, int nf, int C, int CP, const int *list, int first, int n, double *buf)
{
  const long long e = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (e >= (long long) n * nf * C) return;
  const int c = (int) (e % C), fn = (int) ((e / C) % nf), k = (int) (e / ((long long) C * nf));
  const int atom = list ? list[k] : first + k;
  buf[e] = (double) rows[atom * stride + (long long) fn * CP + c];
}
template<class T, bool ADD>
__global__ void k_comm_unpack(T *rows, long long stride, int nf, int C, int CP, const int *list, int first, int n, const double *buf)
{
  const long long e = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  const int W = ADD ? C : CP;
  if (e >= (long long) n * nf * W) return;
  const int c = (int) (e % W), fn = (int) ((e / W) % nf), k = (int) (e / ((long long) W * nf));
  const int atom = list ? list[k] : first + k;
  T *dst = rows + atom * stride + (long long) fn * CP + c;
  const double v = c < C ? buf[((long long) k * nf + fn) * C + c] : 0.0;
  // several entries of a send list may name one atom (an atom with several images): atomic add
  if (ADD) atomicAdd(dst, (T) v);
  else *dst = (T) v;
}

// plain copy of n doubles: the calibration kernel for the HBM counters (FETCH_SIZE / WRITE_SIZE per byte moved)
static __global__ void k_copy_calibration(const double *src, double *dst, long long n)
{
  for (long long i = blockIdx.x * (long long) blockDim.x + threadIdx.x; i < n; i += (long long) gridDim.x * blockDim.x) dst[i] = src[i];
}

// read-only stream over n doubles (16 bytes per lane and step, one partial sum written per block): what a kernel that
// only reads can draw from HBM, next to the copy kernel's rate for one that reads and writes as much
static __global__ void k_read_calibration(const double *src, double *partial, long long n)
{
  const double2 *s2 = reinterpret_cast<const double2 *>(src);
  double acc = 0.0;
  for (long long i = blockIdx.x * (long long) blockDim.x + threadIdx.x; i < n / 2; i += (long long) gridDim.x * blockDim.x) {
    const double2 v = s2[i];
    acc += v.x + v.y;
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) atomicAdd(&partial[blockIdx.x], acc);
}

// ---------------------------------------------------------------------------------------------------------------
// bond filter
// ---------------------------------------------------------------------------------------------------------------
struct BondSrc {
  const int *mu;              // [n] model element of each atom
  const long long *offset;    // [n + 1]
  const int *j;               // [nb]
  const double *rij;          // [nb][3] or null
  const double *x;            // [n][3]      (with rij null)
  const int *image;           // [nb]
  const double *shifts;       // [nimg][3]
  const double *cut;          // [nel][nel] pair cutoffs
  int nel;
};

__device__ inline void bond_vec(const BondSrc &s, int i, long long q, double &dx, double &dy, double &dz)
{
  if (s.rij) {
    dx = s.rij[3 * q]; dy = s.rij[3 * q + 1]; dz = s.rij[3 * q + 2];
  } else {    // x_j - x_i + shift, in this order (system.h:36-42)
    const int jj = s.j[q];
    const double *xi = s.x + 3 * (long long) i, *xj = s.x + 3 * (long long) jj, *sh = s.shifts + 3 * (long long) s.image[q];
    dx = xj[0] - xi[0] + sh[0];
    dy = xj[1] - xi[1] + sh[1];
    dz = xj[2] - xi[2] + sh[2];
  }
}

// What a pass clears before it adds to it: the records and forces (one buffer) and the per-atom virials, and the flag of a bond of
// length zero.  k_edge_count does it, the first kernel of a pass: as fills of their own they were three launches, which with a few
// hundred atoms the GPU waits for (the host issues a launch in about 5 us).
struct PassClear {
  double *out, *vatom;
  long long nout, nvatom;
  int *zero_bond;             // (i, j) of a bond of length zero, or (-1, -1)
};

// one wave per atom: number of bonds with 0 < r^2 < rc^2
static __global__ void k_edge_count(BondSrc s, int n, int *count, PassClear z)
{
  const long long t0 = blockIdx.x * (long long) blockDim.x + threadIdx.x, step = (long long) gridDim.x * blockDim.x;
  for (long long q = t0; q < z.nout; q += step) z.out[q] = 0.0;
  for (long long q = t0; q < z.nvatom; q += step) z.vatom[q] = 0.0;
  if (t0 < 2) z.zero_bond[t0] = -1;
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (i >= n) return;
  const int mi = s.mu[i];
  int c = 0;
  for (long long q = s.offset[i] + lane; q < s.offset[i + 1]; q += 64) {
    double dx, dy, dz;
    bond_vec(s, i, q, dx, dy, dz);
    const double rsq = dx * dx + dy * dy + dz * dz;
    const double rc = s.cut[mi * s.nel + s.mu[s.j[q]]];
    if (rsq < rc * rc && rsq != 0.0) c++;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_down(c, o, 64);
  if (lane == 0) count[i] = c;
}

// Exclusive scan of count[n] into eoff[n + 1], a block of 1024 threads per kScanBlock counts (count: 16-byte aligned).  A block adds
// up the counts in front of its own itself, so the blocks need neither a second launch nor each other: it reads 4 n / 2 bytes on
// average from the L2.  One block that walked the list took 1.9 us per 1024 counts (65 536 atoms 122 us, 32 000 62, 4001 10);
// now 8.9, 7.6 and 5.4 us.
constexpr int kScanBlock = 8192;
static __global__ __launch_bounds__(1024) void k_scan(const int *__restrict__ count, int n, long long *__restrict__ eoff)
{
  __shared__ long long wsum[16], wpre[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const long long b0 = (long long) blockIdx.x * kScanBlock, base = b0 + 8 * t;
  long long pre = 0;
#pragma unroll 4
  for (long long i = 4 * t; i < b0; i += 4096) {    // b0 is a multiple of 4096
    const int4 v = *reinterpret_cast<const int4 *>(count + i);
    pre += (long long) v.x + v.y + v.z + v.w;
  }
  __align__(16) int v[8];
  long long own = 0;
  if (base + 8 <= n) {
    *reinterpret_cast<int4 *>(v) = *reinterpret_cast<const int4 *>(count + base);
    *reinterpret_cast<int4 *>(v + 4) = *reinterpret_cast<const int4 *>(count + base + 4);
  } else {
    for (int k = 0; k < 8; k++) v[k] = base + k < n ? count[base + k] : 0;
  }
  for (int k = 0; k < 8; k++) own += v[k];
  long long inc = own;
  for (int o = 1; o < 64; o <<= 1) {
    const long long up = __shfl_up(inc, o, 64);
    if (lane >= o) inc += up;
  }
  for (int o = 32; o > 0; o >>= 1) pre += __shfl_xor(pre, o, 64);
  if (lane == 63) wsum[wave] = inc;
  if (lane == 0) wpre[wave] = pre;
  __syncthreads();
  long long at = inc - own;
  for (int w = 0; w < 16; w++) at += wpre[w] + (w < wave ? wsum[w] : 0);
  for (int k = 0; k < 8; k++) {
    if (base + k < n) eoff[base + k] = at;
    at += v[k];
  }
  if (blockIdx.x == gridDim.x - 1 && t == 1023) eoff[n] = at;
}
inline void launch_scan(hipStream_t stream, const int *count, int n, long long *eoff)
{
  hipLaunchKernelGGL(k_scan, dim3(n > 0 ? (unsigned) ((n - 1) / kScanBlock + 1) : 1u), dim3(1024), 0, stream, count, n, eoff);
}

// Energy and virial are added per atom with atomics to records of 8 doubles (energy, virial[6], unused).  Additions to one
// record follow each other at about 12 ns (k_energy_2l: 0.40 ms for 32 000 atoms of one structure, 0.11 ms for 42 000 atoms of
// 512 structures), so one structure alone has kRecordCopies records that its atoms use in turn and whoever reads them adds
// up; a list of several structures (sid) has one record each.  64 copies: one 64-byte line for each of the blocks that end
// at about the same time, and 4 kB for the host to add.
constexpr int kRecordCopies = 64;
__device__ inline long long record_of(const int *sid, int i) { return 8ll * (sid ? sid[i] : i & (kRecordCopies - 1)); }

// records of the structures, `copies` for each -> energy [nstruct], virial [nstruct][6] (null: skipped)
static __global__ void k_unpack_records(const double *rec, int nstruct, int copies, double *energy, double *virial)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nstruct) return;
  double v[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int q = 0; q < copies; q++)
    for (int k = 0; k < 7; k++) v[k] += rec[8 * ((long long) s * copies + q) + k];
  if (energy) energy[s] = v[0];
  if (virial)
    for (int k = 0; k < 6; k++) virial[6 * (long long) s + k] = v[1 + k];
}

// f[atom[q]] += fe[q], eatom[atom[q]] += ee[q] for the n rows of the engine (null pointers are skipped)
// adds the pass's forces (rows 0 .. nf) and atom energies (rows 0 .. ne) to the caller's arrays; atom: caller's index of row q,
// null when the rows are in the caller's order
static __global__ void k_add_results(const int *atom, int nf, int ne, const double *fe, double *f, const double *ee, double *eatom)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nf && q >= ne) return;
  const long long i = atom ? atom[q] : q;
  if (f && q < nf) {
    f[3 * i] += fe[3 * (long long) q];
    f[3 * i + 1] += fe[3 * (long long) q + 1];
    f[3 * i + 2] += fe[3 * (long long) q + 2];
  }
  if (eatom && q < ne) eatom[i] += ee[q];
}

// dst[atom[q]][k] += src[q][k], k < ncomp, for rows of sstride values in src and ncomp values in dst (atom null: row q)
static __global__ void k_add_rows(const int *atom, int n, const double *src, int sstride, int ncomp, double *dst)
{
  const long long t = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (t >= (long long) ncomp * n) return;
  const long long q = t / ncomp;
  const int k = (int) (t % ncomp);
  dst[ncomp * (atom ? (long long) atom[q] : q) + k] += src[sstride * q + k];
}

struct Edges {
  int *ei, *ej, *emu;         // central atom, neighbour, neighbour element
  double *rh;                 // [E][3] unit vectors
  double *r, *x, *rc;         // length, r / rc, rc
  int *erow;                  // its own number (k_edge_pairs), or null
};

// One wave per atom, four per block: in-cutoff bonds in list order -> compact edge arrays at eoff[i].  The first bond of length 0
// that is seen is recorded in zero_bond (cleared by k_edge_count) and reported in `flag`, (i, j) in the host's pinned memory.
// SCAN: the block also adds up the counts of the atoms in front of its own and writes its part of eoff, which saves the launch of
// k_scan (4.6 us and the gap behind it) where a pass has few atoms.  A block reads 2 n bytes of counts on average, n^2 / 2 bytes in
// all: 8 MB from the L2 with 4096 atoms, about what the launch costs.
constexpr int kFillScanAtoms = 4096;
template<bool SCAN>
static __global__ __launch_bounds__(256) void k_edge_fill(BondSrc s, int n, const int *__restrict__ count, long long *eoff, Edges e, int *zero_bond, int *flag)
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = blockIdx.x * 4 + wave;
  long long w = 0;
  if (SCAN) {
    __shared__ int part[4];
    int c = 0;
    for (int q = threadIdx.x; q < (int) blockIdx.x * 4; q += 256) c += count[q];
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if (lane == 0) part[wave] = c;
    __syncthreads();
    if (i >= n) return;
    w = (long long) part[0] + part[1] + part[2] + part[3];
    for (int k = 0; k < wave; k++) w += count[blockIdx.x * 4 + k];
    if (lane == 0) {
      eoff[i] = w;
      if (i == n - 1) eoff[n] = w + count[i];
    }
  } else {
    if (i >= n) return;
    w = eoff[i];
  }
  const int mi = s.mu[i];
  const long long q0 = s.offset[i], q1 = s.offset[i + 1];
  for (long long base = q0; base < q1; base += 64) {
    const long long q = base + lane;
    bool keep = false;
    double dx = 0, dy = 0, dz = 0, rsq = 0, rc = 0;
    int jj = 0;
    if (q < q1) {
      bond_vec(s, i, q, dx, dy, dz);
      rsq = dx * dx + dy * dy + dz * dz;
      jj = s.j[q];
      rc = s.cut[mi * s.nel + s.mu[jj]];
      keep = (rsq < rc * rc) && rsq != 0.0;
      if (rsq == 0.0 && 0.0 < rc * rc && atomicCAS(zero_bond, -1, i) == -1) {
        __hip_atomic_store(flag + 1, jj, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(flag, i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
    const unsigned long long m = __ballot(keep);
    if (keep) {
      const long long p = w + __popcll(m & ((1ull << lane) - 1ull));
      const double r = sqrt(rsq), ir = 1.0 / r;
      e.ei[p] = i;
      e.ej[p] = jj;
      e.emu[p] = s.mu[jj];
      e.rh[3 * p] = dx * ir; e.rh[3 * p + 1] = dy * ir; e.rh[3 * p + 2] = dz * ir;
      e.r[p] = r;
      e.rc[p] = rc;
      e.x[p] = r / rc;
      if (e.erow) e.erow[p] = (int) p;
    }
    w += __popcll(m);
  }
}

// One row of radial functions for the two directions of a bond.  The radial network of GRACE-1L and 2L sees only r / rc, and
// the bonds i -> j and j -> i have the same length, so a pass over many bonds evaluates the network once per pair: erow[e] is
// the bond whose row bond e uses (a row stands at its own bond's place); k_edge_rows lists the bonds that have a row.
// k_edge_fill has set erow[e] = e.  Of two atoms the one that pair_owner() names looks for the counterparts of its bonds --
// the bonds of the other atom with the opposite unit vector and the same argument to 16 ulp (bond vectors that a caller
// computed for each direction round differently) -- and points them at its own bond, which nobody points elsewhere.  A bond
// without a counterpart in the list (a ghost's row, another chunk of atoms, a list that is not symmetric) and a bond of an
// atom with its own image keep their rows.  `same`: largest difference of the two arguments over their sum, kSameArgument, or 0
// with ordered sums: which bonds meet their counterpart follows the chunk size, and the bits of a result must not.
// One wave per atom.  What the search waits for is memory latency (index of the neighbour, start of its row, the row, the
// counterpart's vector), so a lane first fetches the row of its own bond's neighbour for 64 bonds at a time, and then 16 bonds
// are looked up together, 16 lanes each, 80 entries of every row in flight.
constexpr double kSameArgument = 1.8e-15;    // 16 ulp of a value near 1
__device__ inline bool pair_owner(int i, int j) { return ((i + j) & 1) ? i < j : i > j; }    // half of the bonds of every atom
static __global__ __launch_bounds__(256) void k_edge_pairs(const long long *__restrict__ eoff, int a0, int natoms, const int *__restrict__ ej,
                                                           const double *__restrict__ rh, const double *__restrict__ x, int *__restrict__ erow,
                                                           double same)
{
  __shared__ int s_row[4][64], s_len[4][64], s_e[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gq = lane >> 4, lq = lane & 15;
  const int ia = blockIdx.x * 4 + wave, i = a0 + ia;
  if (ia >= natoms) return;
  const int e0 = (int) eoff[i], e1 = (int) eoff[i + 1];
  for (int b0 = e0; b0 < e1; b0 += 64) {
    const int e = b0 + lane;
    const int j = e < e1 ? ej[e] : -1;
    const bool look = j >= a0 && j < a0 + natoms && j != i && pair_owner(i, j);
    const unsigned long long mask = __ballot(look);
    const int nlook = __popcll(mask);
    __builtin_amdgcn_wave_barrier();
    if (look) {
      const int r = __popcll(mask & ((1ull << lane) - 1ull)), start = (int) eoff[j];
      s_row[wave][r] = start;
      s_len[wave][r] = (int) eoff[j + 1] - start;
      s_e[wave][r] = e;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int t = 0; t < nlook; t += 16) {
      int row[4], n[4], eb[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int q = t + 4 * k + gq;
        row[k] = q < nlook ? s_row[wave][q] : 0;
        n[k] = q < nlook ? s_len[wave][q] : 0;
        eb[k] = q < nlook ? s_e[wave][q] : 0;
      }
      int base = 0;
      bool more;
      do {    // one round per 80 entries of the longest of the 16 rows
        int nb[4][5];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
          for (int m = 0; m < 5; m++) {
            const int at = base + 16 * m + lq;
            nb[k][m] = at < n[k] ? ej[row[k] + at] : -1;
          }
        unsigned hit[4], any = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
          hit[k] = 0;
#pragma unroll
          for (int m = 0; m < 5; m++) hit[k] |= nb[k][m] == i ? 1u << m : 0u;
          any |= hit[k];
        }
        while (__ballot(any != 0)) {    // one round unless a row names atom i more than once (images of a small cell)
          any = 0;
#pragma unroll
          for (int k = 0; k < 4; k++)
            if (hit[k]) {
              const long long m = row[k] + base + 16 * (__ffs(hit[k]) - 1) + lq, ek = eb[k];
              const double d = fabs(rh[3 * m] + rh[3 * ek]) + fabs(rh[3 * m + 1] + rh[3 * ek + 1]) + fabs(rh[3 * m + 2] + rh[3 * ek + 2]);
              const double xm = x[m], xe = x[ek];
              if (d < 1e-9 && fabs(xm - xe) <= same * (xm + xe)) erow[m] = (int) ek;
              hit[k] &= hit[k] - 1;
              any |= hit[k];
            }
        }
        base += 80;
        more = base < n[0] || base < n[1] || base < n[2] || base < n[3];
      } while (__ballot(more));
    }
  }
}
// The bonds of [e_begin, e_end) that have a row of their own (erow[e] == e): uid[q], ux[q] = their numbers and arguments,
// *nrows their count (cleared by the caller).  A block lists kRowsPerBlock bonds and takes its place in the list with one
// atomic addition (additions to one address follow each other at 12 ns).
constexpr int kRowsPerBlock = 4096;
static __global__ __launch_bounds__(1024) void k_edge_rows(const long long *__restrict__ eoff, int a0, int natoms, const int *__restrict__ erow,
                                                           const double *__restrict__ x, int *__restrict__ uid, double *__restrict__ ux,
                                                           unsigned long long *nrows)
{
  __shared__ int cnt[16];
  __shared__ unsigned long long first;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const long long e0 = eoff[a0] + (long long) blockIdx.x * kRowsPerBlock, e1 = eoff[a0 + natoms];
  if (e0 >= e1) return;
  unsigned long long mask[kRowsPerBlock / 1024];
  int own = 0;
#pragma unroll
  for (int k = 0; k < kRowsPerBlock / 1024; k++) {
    const long long e = e0 + wave * (kRowsPerBlock / 16) + k * 64 + lane;
    mask[k] = __ballot(e < e1 && erow[e] == (int) e);
    own += __popcll(mask[k]);
  }
  if (lane == 0) cnt[wave] = own;
  __syncthreads();
  if (t == 0) {
    int total = 0;
    for (int w = 0; w < 16; w++) total += cnt[w];
    first = atomicAdd(nrows, (unsigned long long) total);
  }
  __syncthreads();
  long long u = (long long) first;
  for (int w = 0; w < wave; w++) u += cnt[w];
#pragma unroll
  for (int k = 0; k < kRowsPerBlock / 1024; k++) {
    const long long e = e0 + wave * (kRowsPerBlock / 16) + k * 64 + lane;
    if (mask[k] >> lane & 1) {
      const long long q = u + __popcll(mask[k] & ((1ull << lane) - 1ull));
      uid[q] = (int) e;
      ux[q] = x[e];
    }
    u += __popcll(mask[k]);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// radial MLP on the matrix cores
// ---------------------------------------------------------------------------------------------------------------
template<class T> struct Mfma;
template<> struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  __device__ static inline v4 mma(double a, double b, v4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
};
template<> struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  __device__ static inline v4 mma(float a, float b, v4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

// D = A B for one wave with A[i][k], B[k][j] held as (i or j = lane % 16, k = lane / 16): every lane writes its four
// accumulator values; the host derives which (row, column) each (lane, register) holds
template<class T> __global__ void k_mfma_probe(const T *A, const T *B, T *D)
{
  const int lane = threadIdx.x;
  typename Mfma<T>::v4 acc = {0, 0, 0, 0};
  acc = Mfma<T>::mma(A[(lane & 15) * 4 + (lane >> 4)], B[(lane >> 4) * 16 + (lane & 15)], acc);
  for (int v = 0; v < 4; v++) D[lane * 4 + v] = acc[v];
}

template<class T> struct RadialArgs {
  const long long *n_edges;   // device scalar: edges of this pass are [e_begin, e_begin + count)
  long long e_begin, e_count; // e_count < 0: take *n_edges - e_begin
  const double *x;            // [E] r / rc
  const int *emu;             // [E] neighbour element
  const int *uid;             // LISTED: [count] row that entry q of the pass writes (k_edge_pairs), without species weights
  const T *w0, *w1, *w2;      // fragment-ordered weights (norms folded in)
  const T *z;                 // [nel][C]
  T *Rz, *dRz;                // [E][noutp]  columns l * C + n
  int nrb, p, ks0;            // basis functions, envelope order, k-steps of layer 0
  int nob, noutp;             // 16-column blocks and padded width of the output
  int C, nel, act;            // radial channels, elements, activation (0 SiLU, 1 tanh)
  int w2_in_lds;
  int drow[16];               // accumulator row of (lane / 16, register)
  // species form (MODE 1 of k_radial): the basis is the bare T_k(2x - 1); layer 0 adds bias_i[element of the central
  // atom] + bias_j[element of the neighbour], layer 1 adds bias1, and the envelope multiplies the output
  const int *emi;             // [E] element of the central atom
  const T *bias_i, *bias_j;   // [nel][HB * 16]
  const T *bias1;             // [HB * 16]
};

// reciprocal: hardware estimate + Newton steps (2 in fp64: full precision; 1 in fp32)
__device__ inline double fast_rcp(double x)
{
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  r = fma(fma(-x, r, 1.0), r, r);
  return r;
}
__device__ inline float fast_rcp(float x)
{
  float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.0f), r, r);
}

template<class T, int ACT> __device__ inline void act_pair(T &s, T &ds)
{
  if (ACT == 1) {
    const T t = tanh(s);
    ds = ds * ((T) 1 - t * t);
    s = t;
  } else {
    const T sg = fast_rcp((T) 1 + exp(-s));
    ds = sg * ((T) 1 + s * ((T) 1 - sg)) * ds;
    s = s * sg;
  }
}

// x^n for a non-negative integer n by squaring
__device__ inline double ipow(double x, int n)
{
  double r = 1.0, b = x;
  while (n > 0) {
    if (n & 1) r *= b;
    b *= b;
    n >>= 1;
  }
  return r;
}

// One wave = 16 edges.  Layers 0 and 1 run as D[feature][edge] = W^T H with the weights as the A operand, so the
// accumulator registers of one layer are exactly the B operand of the next (no data movement between layers: the
// k index of a step is the accumulator row held by that lane, and the weight fragments are stored in that order).
// Layer 2 swaps the operands, D[edge][column], so that 16 lanes write 16 consecutive columns of one edge row.
// Every k-step feeds all row blocks of the value and the tangent stream (2 HB independent accumulator chains).
// ACT: 0 SiLU, 1 tanh (compile-time: the fp64 tanh is large, and both activations inlined 32 times overflow the
// instruction cache).
// Radial functions from tables, as the reference's engines evaluate them (spline_eval, libgrace/include/grace/fused_cpu.h:
// 1052-1074; tables of Grace1LFused::build_splines, libgrace/src/fused_1l.cpp:102-129): N intervals over x = r / rc in
// [0, 1], per interval the cubic through the values and derivatives of the radial MLP at its two ends,
//   R(t) = f0 + t (d0 + t (c2 + t c3)),  c2 = -3 f0 - 2 d0 + 3 f1 - d1,  c3 = 2 f0 + d0 - 2 f1 + d1,  d = f' / N,
//   dR/dx = N (d0 + t (2 c2 + 3 c3 t)),  k = min(int(x N), N - 1),  t = x N - k.
// COEF false (fp64): F, D are [N + 1][noutp] value and d/dx at the knots (what k_radial returns for x = k / N and unit
// species weights) and the cubic's coefficients are formed per use, so the table is half the size of stored coefficients
// and stays in the L2.  COEF true (fp32): F is [N][4][noutp] coefficients formed in fp64 by k_spline_coef (c2 and c3 are
// differences of nearly equal values: formed in fp32 they would cost four digits of dR/dx), D unused.
// One block = noutp threads rounded up to a wave, a thread per column, blocks stride over the edges; rows as k_radial.
// Species form (GRACE-3L: the MLP takes the embeddings of both atoms of the bond; per-pair tables of the reference,
// libgrace/src/fused_3l.cpp:487-520): emi set: one table per ordered pair of species, table number sp[emi[e]] nsp +
// sp[emu[e]] (sp: element -> species of the engine), the tables one after the other in F and D.
// WEIGHTS false: rows without species weights, z is not read.  A form of its own for layers that have none: with weights of one
// read for every value, 175 cells of GRACE-2L in fp64 took 0.366 -> 0.451 ms, 3999 atoms in fp32 0.078 -> 0.090.
template<class T, bool COEF, bool WEIGHTS>
__global__ void k_radial_spline(const long long *__restrict__ n_edges, long long e_begin, long long e_count, const double *__restrict__ x,
                                const int *__restrict__ emu, const T *__restrict__ F, const T *__restrict__ D, int N, const T *__restrict__ z, int C,
                                int noutp, T *__restrict__ Rz, T *__restrict__ dRz, const int *__restrict__ emi = nullptr,
                                const int *__restrict__ sp = nullptr, int nsp = 1)
{
  const long long cnt = e_count >= 0 ? e_count : *n_edges - e_begin;
  const int col = threadIdx.x;
  if (col >= noutp) return;
  const int n = col % C;
  const T h = (T) (1.0 / N);
  constexpr int U = 4;    // edges of one step: their table reads are in flight together
  for (long long el0 = (long long) blockIdx.x * U; el0 < cnt; el0 += (long long) gridDim.x * U) {
    T c0[U], c1[U], c2[U], c3[U], t[U], zc[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const long long e = e_begin + (el0 + u < cnt ? el0 + u : cnt - 1);
      const double sx = x[e] * N;
      int k = (int) sx;
      k = k > N - 1 ? N - 1 : (k < 0 ? 0 : k);
      t[u] = (T) (sx - k);
      zc[u] = WEIGHTS ? z[emu[e] * C + n] : (T) 1;
      const long long pair = emi ? (long long) sp[emi[e]] * nsp + sp[emu[e]] : 0;
      if (COEF) {
        const T *c = F + (pair * N + k) * 4 * noutp + col;
        c0[u] = c[0]; c1[u] = c[noutp]; c2[u] = c[2 * noutp]; c3[u] = c[3 * noutp];
      } else {
        const T *f = F + (pair * (N + 1) + k) * noutp + col, *d = D + (pair * (N + 1) + k) * noutp + col;
        c0[u] = f[0]; c1[u] = d[0]; c2[u] = f[noutp]; c3[u] = d[noutp];    // f0, f0', f1, f1'
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (el0 + u >= cnt) break;
      const long long e = e_begin + el0 + u;
      T a0 = c0[u], a1 = c1[u], a2 = c2[u], a3 = c3[u];
      if (!COEF) {
        const T f1 = a2, d1 = a3 * h;
        a1 *= h;
        a2 = (T) -3 * a0 - (T) 2 * a1 + (T) 3 * f1 - d1;
        a3 = (T) 2 * a0 + a1 - (T) 2 * f1 + d1;
      }
      const T tt = t[u];
      __builtin_nontemporal_store((a0 + tt * (a1 + tt * (a2 + tt * a3))) * zc[u], &Rz[e * noutp + col]);
      __builtin_nontemporal_store((a1 + tt * ((T) 2 * a2 + tt * (T) 3 * a3)) * (T) N * zc[u], &dRz[e * noutp + col]);
    }
  }
}
// coefficients [N][4][noutp] of the cubics in fp32 from the knot values and derivatives in fp64
static __global__ void k_spline_coef(const double *__restrict__ F, const double *__restrict__ D, int N, int noutp, float *__restrict__ coef)
{
  const long long q = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (q >= (long long) N * noutp) return;
  const long long k = q / noutp;
  const int col = (int) (q % noutp);
  const double f0 = F[k * noutp + col], f1 = F[(k + 1) * noutp + col], d0 = D[k * noutp + col] / N, d1 = D[(k + 1) * noutp + col] / N;
  float *c = coef + k * 4 * noutp + col;
  c[0] = (float) f0;
  c[noutp] = (float) d0;
  c[2 * noutp] = (float) (-3.0 * f0 - 2.0 * d0 + 3.0 * f1 - d1);
  c[3 * noutp] = (float) (2.0 * f0 + d0 - 2.0 * f1 + d1);
}

// Threads of a block: hidden width 64 with every weight in LDS runs three waves per SIMD (168 registers; two waves at 180
// were 2 % slower in fp64, 6 % in fp32), the other forms would spill at that size; width 128 runs one wave per SIMD.
constexpr int radial_threads(int hb, int mode, bool w2l) { return hb <= 4 ? (w2l && mode == 0 ? 768 : 512) : 256; }

// LISTED: the rows of a list (RadialArgs::uid) instead of consecutive ones.  A form of its own: with the test inside the loads
// and stores the three networks of GRACE-3L, whose rows are never listed, took 2.49 ms each instead of 2.36 (10 000 atoms fp32),
// and the listed rows 1.48 instead of 1.37 (GRACE-2L, 32 000 atoms fp64; fp32 0.81, 0.74).
template<class T, int HB, int ACT, int MODE, bool W2L, bool LISTED> __global__ __launch_bounds__((radial_threads(HB, MODE, W2L))) void k_radial(RadialArgs<T> a)
{
  typedef typename Mfma<T>::v4 v4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *w0s = reinterpret_cast<T *>(smem_raw);
  T *w1s = w0s + HB * a.ks0 * 64;
  T *w2s = w1s + HB * HB * 4 * 64;
  {
    const int n0 = HB * a.ks0 * 64, n1 = HB * HB * 4 * 64, n2 = W2L ? (a.nob * HB * 4 + kRadialPrefetch) * 64 : 0;
    for (int q = threadIdx.x; q < n0; q += blockDim.x) w0s[q] = a.w0[q];
    for (int q = threadIdx.x; q < n1; q += blockDim.x) w1s[q] = a.w1[q];
    for (int q = threadIdx.x; q < n2; q += blockDim.x) w2s[q] = a.w2[q];
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const long long cnt = a.e_count >= 0 ? a.e_count : *a.n_edges - a.e_begin;
  const long long ntiles = (cnt + 15) / 16;
  const int p = a.p;
  const double cf0 = 0.5 * (p + 1) * (p + 2), cf1 = (double) p * (p + 2), cf2 = 0.5 * p * (p + 1), cfd = 0.5 * p * (p + 1) * (p + 2);
  // The memory counter of a wave retires loads and stores in order: a load issued behind a store waits for that store
  // to complete.  The per-edge inputs of the NEXT tile (x of this lane's column, element and x of this lane's four
  // output rows) are therefore requested before the first store of the current tile.
  const int KZ = a.C >> 4;                        // distinct columns n = (16 cb + c) mod C of a lane: c + 16 k, k < KZ <= 4
  // Tiles go to the blocks in turn: a pass of few tiles then runs on as many CUs as there are tiles instead of filling the
  // waves of the first blocks (464 tiles: 39 blocks of 12 waves before).
  const long long tstep = (long long) gridDim.x * nw;
  long long tile = (long long) wave * gridDim.x + blockIdx.x;
  double x_n = 0.5, xv_n[4] = {0.5, 0.5, 0.5, 0.5};
  int emu_n[4] = {0, 0, 0, 0};    // element of the neighbour; LISTED: the row
  const int *const emu_src = LISTED ? a.uid : a.emu + a.e_begin;
  auto fetch_edge_inputs = [&](long long tl) {
    const long long el = tl * 16 + c;
    x_n = (tl < ntiles && el < cnt) ? a.x[a.e_begin + el] : 0.5;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const long long er = tl * 16 + a.drow[g * 4 + v];
      const bool ok = tl < ntiles && er < cnt;
      emu_n[v] = ok ? emu_src[er] : 0;
      if (MODE == 1) xv_n[v] = ok ? a.x[a.e_begin + er] : 0.5;
    }
  };
  fetch_edge_inputs(tile);
  for (; tile < ntiles; tile += tstep) {
    const long long eloc = tile * 16 + c;
    const long long e = a.e_begin + eloc;
    const double x = x_n;
    double xv[4];
#pragma unroll
    for (int v = 0; v < 4; v++) xv[v] = xv_n[v];
    // basis g_k = T_k(2x - 1) fcut_p(x), k = 1..nrb, and d/dx (radial_x.h:11-26); this lane supplies k = 4 s + g
    T h0[kMaxRadBasis / 4], dh0[kMaxRadBasis / 4];
    {
      const double xpm = ipow(x, p - 1), xp = xpm * x, xp1 = xp * x, xp2 = xp1 * x;
      const double fc = 1.0 - cf0 * xp + cf1 * xp1 - cf2 * xp2;
      const double dfc = cfd * (-xpm + 2.0 * xp - xp1);
      const double t = 2.0 * x - 1.0;
      double Tp = 1.0, Tc = t, dTp = 0.0, dTc = 2.0;
#pragma unroll
      for (int s = 0; s < kMaxRadBasis / 4; s++) { h0[s] = (T) 0; dh0[s] = (T) 0; }
      for (int k = 0; k < a.nrb; k++) {
        const double gk = MODE == 1 ? Tc : Tc * fc, dgk = MODE == 1 ? dTc : dTc * fc + Tc * dfc;
        if ((k & 3) == g) {
#pragma unroll
          for (int s = 0; s < kMaxRadBasis / 4; s++)
            if (s == (k >> 2)) { h0[s] = (T) gk; dh0[s] = (T) dgk; }
        }
        const double Tn = 2.0 * t * Tc - Tp, dTn = 2.0 * (2.0 * Tc + t * dTc) - dTp;
        Tp = Tc; dTp = dTc; Tc = Tn; dTc = dTn;
      }
    }
    // ---- layer 0
    v4 h1[HB], dh1[HB];
#pragma unroll
    for (int rb = 0; rb < HB; rb++) { h1[rb] = v4{0, 0, 0, 0}; dh1[rb] = v4{0, 0, 0, 0}; }
#pragma unroll
    for (int s = 0; s < kMaxRadBasis / 4; s++)
      if (s < a.ks0) {
#pragma unroll
        for (int rb = 0; rb < HB; rb++) {
          const T w = w0s[(rb * a.ks0 + s) * 64 + lane];
          h1[rb] = Mfma<T>::mma(w, h0[s], h1[rb]);
          dh1[rb] = Mfma<T>::mma(w, dh0[s], dh1[rb]);
        }
      }
    if (MODE == 1) {
      const long long ee = eloc < cnt ? e : a.e_begin;
      const T *bi = a.bias_i + (long long) a.emi[ee] * (HB * 16), *bj = a.bias_j + (long long) a.emu[ee] * (HB * 16);
#pragma unroll
      for (int rb = 0; rb < HB; rb++)
#pragma unroll
        for (int v = 0; v < 4; v++) h1[rb][v] += bi[rb * 16 + a.drow[g * 4 + v]] + bj[rb * 16 + a.drow[g * 4 + v]];
    }
#pragma unroll
    for (int rb = 0; rb < HB; rb++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        T s_ = h1[rb][v], d_ = dh1[rb][v];
        act_pair<T, ACT>(s_, d_);
        h1[rb][v] = s_; dh1[rb][v] = d_;
      }
    // ---- layer 1
    // An fp64 MFMA holds its wave for the 64 cycles it runs, and nothing else of the wave issues meanwhile: what hides
    // the latency of a weight fragment is to request it a few steps (2 MFMAs each) before its use.  The scheduling
    // barriers keep the compiler from moving the request back next to the use.
    v4 h2[HB], dh2[HB];
#pragma unroll
    for (int rb = 0; rb < HB; rb++) { h2[rb] = v4{0, 0, 0, 0}; dh2[rb] = v4{0, 0, 0, 0}; }
    {
      constexpr int NS = HB * 4 * HB;
      // step q = (kb, s, rb): fragment ((rb HB + kb) 4 + s) of w1
      auto frag = [&](int q) { return w1s[(((q % HB) * HB + q / (4 * HB)) * 4 + (q / HB) % 4) * 64 + lane]; };
      T wa_ = frag(0), wb_ = frag(1);
#pragma unroll
      for (int q = 0; q < NS; q++) {
        const int kb = q / (4 * HB), s_ = (q / HB) % 4, rb = q % HB;
        const T w = wa_;
        wa_ = wb_;
        if (q + 2 < NS) wb_ = frag(q + 2);
        __builtin_amdgcn_sched_barrier(0);
        h2[rb] = Mfma<T>::mma(w, h1[kb][s_], h2[rb]);
        dh2[rb] = Mfma<T>::mma(w, dh1[kb][s_], dh2[rb]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (MODE == 1) {
#pragma unroll
      for (int rb = 0; rb < HB; rb++)
#pragma unroll
        for (int v = 0; v < 4; v++) h2[rb][v] += a.bias1[rb * 16 + a.drow[g * 4 + v]];
    }
#pragma unroll
    for (int rb = 0; rb < HB; rb++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        T s_ = h2[rb][v], d_ = dh2[rb][v];
        act_pair<T, ACT>(s_, d_);
        h2[rb][v] = s_; dh2[rb][v] = d_;
      }
    // ---- layer 2 (linear), operands swapped: rows = edges, columns = outputs; one block of 16 columns at a time (a
    // single dependent accumulator chain keeps the matrix pipe full, and one block's weights are all that is in flight)
    // The z values of a column block are requested one block ahead and the inputs of the next tile before the first
    // store of this one: no load is issued behind a store whose completion it would then wait for.
    // rows of the tile as 32-bit offsets from its first row (the tile is wave-uniform), or their numbers in the list, -1: no
    // such edge
    const long long first = LISTED ? 0 : (a.e_begin + tile * 16) * a.noutp;
    T *const Rt = a.Rz + first, *const dRt = a.dRz + first;
    int zrow[4], row_v[4];
    T env_v[4], denv_v[4], zc[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int rl = a.drow[g * 4 + v];
      row_v[v] = tile * 16 + rl < cnt ? (LISTED ? emu_n[v] : rl * a.noutp) : -1;
      zrow[v] = emu_n[v] * a.C + c;
      zc[v] = LISTED ? (T) 1 : a.z[zrow[v]];
      if (MODE == 1) {
        const double xpm = ipow(xv[v], p - 1), xp = xpm * xv[v], xp1 = xp * xv[v], xp2 = xp1 * xv[v];
        env_v[v] = (T) (1.0 - cf0 * xp + cf1 * xp1 - cf2 * xp2);
        denv_v[v] = (T) (cfd * (-xpm + 2.0 * xp - xp1));
      }
    }
    fetch_edge_inputs(tile + tstep);
    // weight fragments of layer 2 run PF steps ahead of their use, across the column blocks (the fragments of
    // consecutive steps are consecutive in memory): LDS when they fit, else global memory, hence the depth
    constexpr int PF = W2L ? 2 : 16, NQ = HB * 4;
    static_assert(PF <= kRadialPrefetch, "padding of the layer-2 weights");
    // two separate pointers: one pointer that may be either would make every read a flat load, which waits for the
    // stores of the block before it
    const T *wl = (W2L ? (const T *) w2s : a.w2) + lane;
    T wq[PF];
#pragma unroll
    for (int i = 0; i < PF; i++) wq[i] = wl[i * 64];
    for (int cb = 0; cb < a.nob; cb++) {
      T zn[4];
      const int kn = ((cb + 1) & (KZ - 1)) * 16;       // column n = c + 16 k of z in the next block
#pragma unroll
      for (int v = 0; v < 4; v++) zn[v] = LISTED ? (T) 1 : a.z[zrow[v] + kn];
      v4 acc = {0, 0, 0, 0}, dacc = {0, 0, 0, 0};
      const T *wc = wl + (long long) cb * NQ * 64;
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        const T w_ = wq[q % PF];
        wq[q % PF] = wc[(q + PF) * 64];               // beyond the last block: the zero padding of the weights
        __builtin_amdgcn_sched_barrier(0);
        acc = Mfma<T>::mma(h2[q / 4][q % 4], w_, acc);
        dacc = Mfma<T>::mma(dh2[q / 4][q % 4], w_, dacc);
        __builtin_amdgcn_sched_barrier(0);
      }
      const int col = cb * 16 + c;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        if (row_v[v] >= 0) {
          const long long o = LISTED ? (long long) row_v[v] * a.noutp + col : row_v[v] + col;
          // streaming stores: the rows are read by other kernels after the whole array has been written
          if (MODE == 1) {
            __builtin_nontemporal_store((T) (acc[v] * env_v[v] * zc[v]), &Rt[o]);
            __builtin_nontemporal_store((T) ((dacc[v] * env_v[v] + acc[v] * denv_v[v]) * zc[v]), &dRt[o]);
          } else {
            __builtin_nontemporal_store((T) (acc[v] * zc[v]), &Rt[o]);
            __builtin_nontemporal_store((T) (dacc[v] * zc[v]), &dRt[o]);
          }
        }
        zc[v] = zn[v];
      }
    }
  }
}

// barrier of a block that exchanges through LDS only: __syncthreads would also wait for the loads and stores in flight
__device__ inline void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// k_radial for few edges: the HB waves of a block share a tile of 16 edges.  Wave w forms row block w of both hidden layers, whose
// values go to LDS in the order in which the next layer takes them (an accumulator register is one k of the next operand), and
// the column blocks w, w + HB .. of the output; the sums are those of k_radial in the same order.  The weights come from L2, those of
// layer 1 and of a wave's first column block ahead of everything else.  In k_radial a wave walks the whole network for its tile
// (29 700 cycles of matrix instructions in fp64 at width 64, 132 000 at width 128) behind the copy of all weights to LDS, however
// many SIMDs have nothing to do.
// Measured, k_radial / k_radial_few, us: width 64, 160 outputs, fp64 8 tiles 27 / 12, 371 tiles 30 / 19, 768 32 / 27, 1024 33 / 34; fp32 371
// tiles 20 / 13, 768 22 / 18, 1024 23 / 21; width 128, 384 outputs, fp64 128 tiles 89 / 35, 371 93 / 67, 512 95 / 73, 768 100 / 106; fp32 371
// tiles 65 / 38, 512 66 / 40, 1024 71 / 74.  What bounds it: one tile per CU takes the latency of its three layers (the activations
// of 16 values per wave run at one wave per SIMD), more tiles take turns.
// dynamic LDS: radial_few_lds(HB) values.
constexpr int radial_few_lds(int hb) { return 2 * 2 * hb * 4 * 64; }
template<class T, int HB, int ACT, int MODE> __global__ __launch_bounds__(64 * HB, HB == 4 ? 3 : 2) void k_radial_few(RadialArgs<T> a)
{
  typedef typename Mfma<T>::v4 v4;
  constexpr int NS = HB * 4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *const hs = reinterpret_cast<T *>(smem_raw);          // [stage][value, tangent][row block, register][lane]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const long long cnt = a.e_count >= 0 ? a.e_count : *a.n_edges - a.e_begin;
  const long long ntiles = (cnt + 15) / 16;
  const int p = a.p;
  const double cf0 = 0.5 * (p + 1) * (p + 2), cf1 = (double) p * (p + 2), cf2 = 0.5 * p * (p + 1), cfd = 0.5 * p * (p + 1) * (p + 2);
  const int KZ = a.C >> 4;
  // weights of the next 16 steps of a layer; behind those of layer 1 come those of the wave's first column block, and so on
  constexpr int PF = 16;
  T wq[PF];
  const T *const wl1 = a.w1 + (w * NS) * 64 + lane, *const wl2 = a.w2 + lane;
  auto column = [&](int cb) { return wl2 + (long long) cb * NS * 64; };
  // value and tangent of stage `stage` times NS steps of weights, of which the first PF wait in wq; next: the weights after them
  auto multiply = [&](int stage, const T *weights, const T *next, bool rows, v4 &h, v4 &dh) {
    const T *hp = hs + stage * 2 * NS * 64 + lane;
#pragma unroll
    for (int q = 0; q < NS; q++) {
      const T wv = wq[q % PF];
      wq[q % PF] = q + PF < NS ? weights[(q + PF) * 64] : next[(q + PF - NS) * 64];
      const T x = hp[q * 64], dx = hp[(NS + q) * 64];
      h = rows ? Mfma<T>::mma(x, wv, h) : Mfma<T>::mma(wv, x, h);
      dh = rows ? Mfma<T>::mma(dx, wv, dh) : Mfma<T>::mma(wv, dx, dh);
      if (q % 8 == 7) __builtin_amdgcn_sched_barrier(0);    // or the operands of all steps are read ahead, and spilled
    }
  };
#pragma unroll
  for (int q = 0; q < PF; q++) wq[q] = wl1[q * 64];
  auto put = [&](int stage, const v4 &h, const v4 &dh) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      hs[((stage * 2 + 0) * NS + w * 4 + v) * 64 + lane] = h[v];
      hs[((stage * 2 + 1) * NS + w * 4 + v) * 64 + lane] = dh[v];
    }
  };
  auto activate = [&](v4 &h, v4 &dh) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      T s_ = h[v], d_ = dh[v];
      act_pair<T, ACT>(s_, d_);
      h[v] = s_; dh[v] = d_;
    }
  };
  for (long long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const long long eloc = tile * 16 + c;
    const double x = eloc < cnt ? a.x[a.e_begin + eloc] : 0.5;
    int row_v[4], zrow[4];
    double xv[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int rl = a.drow[g * 4 + v];
      const bool ok = tile * 16 + rl < cnt;
      row_v[v] = ok ? rl * a.noutp : -1;
      zrow[v] = (ok ? a.emu[a.e_begin + tile * 16 + rl] : 0) * a.C + c;
      xv[v] = MODE == 1 && ok ? a.x[a.e_begin + tile * 16 + rl] : 0.5;
    }
    // basis, as in k_radial
    T h0[kMaxRadBasis / 4], dh0[kMaxRadBasis / 4];
    {
      const double xpm = ipow(x, p - 1), xp = xpm * x, xp1 = xp * x, xp2 = xp1 * x;
      const double fc = 1.0 - cf0 * xp + cf1 * xp1 - cf2 * xp2;
      const double dfc = cfd * (-xpm + 2.0 * xp - xp1);
      const double t = 2.0 * x - 1.0;
      double Tp = 1.0, Tc = t, dTp = 0.0, dTc = 2.0;
#pragma unroll
      for (int s = 0; s < kMaxRadBasis / 4; s++) { h0[s] = (T) 0; dh0[s] = (T) 0; }
      for (int k = 0; k < a.nrb; k++) {
        const double gk = MODE == 1 ? Tc : Tc * fc, dgk = MODE == 1 ? dTc : dTc * fc + Tc * dfc;
        if ((k & 3) == g) {
#pragma unroll
          for (int s = 0; s < kMaxRadBasis / 4; s++)
            if (s == (k >> 2)) { h0[s] = (T) gk; dh0[s] = (T) dgk; }
        }
        const double Tn = 2.0 * t * Tc - Tp, dTn = 2.0 * (2.0 * Tc + t * dTc) - dTp;
        Tp = Tc; dTp = dTc; Tc = Tn; dTc = dTn;
      }
    }
    // ---- layer 0, row block w
    {
      v4 h = {0, 0, 0, 0}, dh = {0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < kMaxRadBasis / 4; s++)
        if (s < a.ks0) {
          const T wv = a.w0[(w * a.ks0 + s) * 64 + lane];
          h = Mfma<T>::mma(wv, h0[s], h);
          dh = Mfma<T>::mma(wv, dh0[s], dh);
        }
      if (MODE == 1) {
        const long long ee = a.e_begin + (eloc < cnt ? eloc : 0);
        const T *bi = a.bias_i + (long long) a.emi[ee] * (HB * 16), *bj = a.bias_j + (long long) a.emu[ee] * (HB * 16);
#pragma unroll
        for (int v = 0; v < 4; v++) h[v] += bi[w * 16 + a.drow[g * 4 + v]] + bj[w * 16 + a.drow[g * 4 + v]];
      }
      activate(h, dh);
      put(0, h, dh);
    }
    lds_barrier();
    // ---- layer 1, row block w
    {
      v4 h = {0, 0, 0, 0}, dh = {0, 0, 0, 0};
      multiply(0, wl1, w < a.nob ? column(w) : wl1, false, h, dh);
      if (MODE == 1) {
#pragma unroll
        for (int v = 0; v < 4; v++) h[v] += a.bias1[w * 16 + a.drow[g * 4 + v]];
      }
      activate(h, dh);
      put(1, h, dh);
    }
    lds_barrier();
    // ---- layer 2, column blocks w, w + HB, ..
    T env_v[4], denv_v[4];
    if (MODE == 1) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const double xpm = ipow(xv[v], p - 1), xp = xpm * xv[v], xp1 = xp * xv[v], xp2 = xp1 * xv[v];
        env_v[v] = (T) (1.0 - cf0 * xp + cf1 * xp1 - cf2 * xp2);
        denv_v[v] = (T) (cfd * (-xpm + 2.0 * xp - xp1));
      }
    }
    const long long first = (a.e_begin + tile * 16) * a.noutp;
    T *const Rt = a.Rz + first, *const dRt = a.dRz + first;
    for (int cb = w; cb < a.nob; cb += HB) {
      T z[4];
      const int kn = (cb & (KZ - 1)) * 16;
#pragma unroll
      for (int v = 0; v < 4; v++) z[v] = a.z[zrow[v] + kn];
      v4 acc = {0, 0, 0, 0}, dacc = {0, 0, 0, 0};
      multiply(1, column(cb), cb + HB < a.nob ? column(cb + HB) : wl1, true, acc, dacc);
      const int col = cb * 16 + c;
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (row_v[v] >= 0) {
          const int o = row_v[v] + col;
          if (MODE == 1) {
            Rt[o] = (T) (acc[v] * env_v[v] * z[v]);
            dRt[o] = (T) ((dacc[v] * env_v[v] + acc[v] * denv_v[v]) * z[v]);
          } else {
            Rt[o] = (T) (acc[v] * z[v]);
            dRt[o] = (T) (dacc[v] * z[v]);
          }
        }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// A basis
// ---------------------------------------------------------------------------------------------------------------
// The radial tables for kernels that evaluate them themselves instead of reading rows another kernel wrote (the bond
// loops of the reference's fused GPU engines read their table in the same place, libgrace/include/grace/kk/
// grace_1l_fused_kk_impl.h:405-440; CPU: spline_eval, libgrace/include/grace/fused_cpu.h:1052-1074).  F == nullptr: no
// tables, the kernel reads rows.  Layouts and formulas are those of k_radial_spline.
template<class T> struct RadialTable {
  const T *F, *D;     // fp64: value and d/dx at the knots, [N + 1][noutp] each; fp32: F = coefficients [N][4][noutp], D unused
  int N;              // intervals over x = r / rc in [0, 1]
  const double *x;    // [E] r / rc
  const int *emu;     // [E] neighbour element
  const T *z;         // [nel][C] species weights (all ones where the rows carry none)
};
// interval and offset of x in a table of N intervals
__device__ inline int table_interval(double x, int N, double &t)
{
  const double sx = x * N;
  int k = (int) sx;
  k = k > N - 1 ? N - 1 : (k < 0 ? 0 : k);
  t = sx - k;
  return k;
}
// What the cubic of an interval takes from the bond, formed once for all its columns: t, and in fp64 the length of an interval, in
// fp32 2 t and 3 t^2.
template<class T> struct TableBond {
  T t, u, w;
};
template<class T> __device__ inline TableBond<T> table_bond(double t, int N)
{
  if constexpr (sizeof(T) == 8) return {t, 1.0 / N, 0.0};
  else return {(T) t, (T) 2 * (T) t, (T) 3 * (T) t * (T) t};
}
// Entry q of the four of interval k, column col: NOUT, the width of the rows, is a constant where these are used, so that the
// entries stand at constant distances from one (fp64: two) addresses of a bond.
template<class T> struct TableRow {
  const T *f, *d;
};
template<class T, int NOUT> __device__ inline TableRow<T> table_row(const RadialTable<T> &tb, int k, int col)
{
  if constexpr (sizeof(T) == 8) return {tb.F + (long long) k * NOUT + col, tb.D + (long long) k * NOUT + col};
  else return {tb.F + (long long) k * 4 * NOUT + col, nullptr};
}
template<int NOUT, class T> __device__ inline const T *table_entry(const TableRow<T> &r, int q)
{
  if constexpr (sizeof(T) == 8) return (q & 1 ? r.d : r.f) + (q >> 1) * NOUT;    // f0, d0, f1, d1
  else return r.f + q * NOUT;
}
// The cubic of the four entries: fp64 from value and derivative at both ends, fp32 as stored.  (The fp64 slope in the Hermite basis,
// (f1 - f0) 6 t (1 - t) + .., is half the operations and as accurate, but its rounding, eps N f, is another: 8e-14 of a virial.)
template<class T> struct TableCubic {
  T a0, a1, a2, a3;
};
template<class T> __device__ inline TableCubic<T> table_cubic(T e0, T e1, T e2, T e3, const TableBond<T> &b)
{
  if constexpr (sizeof(T) == 8) {
    const T a1 = e1 * b.u, d1 = e3 * b.u;
    return {e0, a1, (T) -3 * e0 - (T) 2 * a1 + (T) 3 * e2 - d1, (T) 2 * e0 + a1 - (T) 2 * e2 + d1};
  } else {
    return {e0, e1, e2, e3};
  }
}
template<class T> __device__ inline T table_value(const TableCubic<T> &a, const TableBond<T> &b)
{
  return a.a0 + b.t * (a.a1 + b.t * (a.a2 + b.t * a.a3));
}
// dR/dt, of which dR/dx is N times
template<class T> __device__ inline T table_slope(const TableCubic<T> &a, const TableBond<T> &b)
{
  if constexpr (sizeof(T) == 8) return a.a1 + b.t * ((T) 2 * a.a2 + b.t * (T) 3 * a.a3);
  else return a.a1 + b.u * a.a2 + b.w * a.a3;
}

// Where a kernel takes the radial functions of a bond from: its own row, the radial tables, or the row of its pair of atoms
// (k_edge_pairs).  A template argument: tested inside the loads, with factors of one where rows carry their weights, pairing
// cost the kernels that never pair (GRACE-3L, 10 000 atoms fp32: k_scatter_a 0.55 -> 0.84 ms, k_bond_bwd 0.72 -> 0.75) and the
// ones that do (GRACE-1L of 48 channels, 8192 atoms fp32: k_scatter_a 0.37 ms, 0.16 now; GRACE-2L, 32 000 atoms fp32: k_bond_bwd
// 1.44, 1.32 now).
enum class RowsOf { bonds, tables, pairs };

template<class T> struct ScatterArgs {
  const long long *eoff;      // [n + 1]
  const double *rh;           // [E][3]
  const T *Rz;                // [E][noutp]
  // erow set (RowsOf::pairs): bond e uses row erow[e] (k_edge_pairs), whose values times z[emu[e]][n] are the radial functions
  // of the bond
  const int *erow, *emu;
  const T *z;                 // [nel][C]
  RadialTable<T> tb;          // tb.F set: the radial functions come from the tables, Rz is not read
  T *A;                       // [chunk atoms][nlm][C]
  int a0, natoms;             // first atom of the chunk, atoms in it
  int C, nl, nlm, noutp;
  int drow[16];               // accumulator row of (lane / 16, register)
  ShCoef sh;
};

// One block per atom, thread = (l, n).  The harmonics of up to kScatterBonds bonds are computed by all threads into LDS,
// then the radial rows stream through registers in groups of bonds, the loads of the next group in flight while the current
// one is accumulated.  16 bonds per group, 8 with paired rows, whose weights are in flight beside them (16: 107 registers
// spilled in fp64).
constexpr int kScatterBonds = 64;
constexpr int scatter_bonds_per_group(RowsOf rows) { return rows == RowsOf::pairs ? 8 : 16; }

template<class T, int MAXM, int GROUP> __device__ inline void scatter_group(const T *Ysh, int b0, int nb, int lm0, int nm, const T *r, T *acc)
{
#pragma unroll
  for (int u = 0; u < GROUP; u++)
    if (b0 + u < nb) {
      // no branch per m (the lanes of a wave hold two values of l): entries beyond 2l+1 read a valid address and add 0
      const T *y = Ysh + (b0 + u) * kMaxNlm + lm0;
      T yv[MAXM];
#pragma unroll
      for (int m = 0; m < MAXM; m++) yv[m] = y[m < nm ? m : 0];
#pragma unroll
      for (int m = 0; m < MAXM; m++) acc[m] += (m < nm ? yv[m] : (T) 0) * r[u];
    }
}

template<class T, int MAXM, RowsOf ROWS> __global__ void k_scatter_a(ScatterArgs<T> a)
{
  constexpr int GROUP = scatter_bonds_per_group(ROWS);
  __shared__ T Ysh[kScatterBonds * kMaxNlm];
  const int t = threadIdx.x;
  const int i = a.a0 + blockIdx.x;
  const long long e0 = a.eoff[i], e1 = a.eoff[i + 1];
  const int ncol = a.nl * a.C;
  const int l = t < ncol ? t / a.C : 0, n = t % a.C;
  const int nm = 2 * l + 1, lm0 = l * l;
  T acc[MAXM];
#pragma unroll
  for (int m = 0; m < MAXM; m++) acc[m] = (T) 0;
  for (long long base = e0; base < e1; base += kScatterBonds) {
    const int nb = (int) (e1 - base < kScatterBonds ? e1 - base : kScatterBonds);
    const T *rp = a.Rz + (ROWS == RowsOf::pairs ? 0 : base * a.noutp) + (t < ncol ? t : 0);
    auto value = [&](int b) {
      const int bb = b < nb ? b : 0;
      if constexpr (ROWS == RowsOf::pairs) return rp[(long long) a.erow[base + bb] * a.noutp] * a.z[a.emu[base + bb] * a.C + n];
      else return rp[(long long) bb * a.noutp];
    };
    T r0[GROUP], r1[GROUP];
#pragma unroll
    for (int u = 0; u < GROUP; u++) r0[u] = value(u);
    __syncthreads();
    for (int b = t; b < nb; b += blockDim.x) {
      const double *u = a.rh + 3 * (base + b);
      sh_eval<false, T>(a.sh, u[0], u[1], u[2], Ysh + b * kMaxNlm, nullptr);
    }
    __syncthreads();
    for (int b0 = 0; b0 < nb; b0 += 2 * GROUP) {
      const int b1 = b0 + GROUP, b2 = b1 + GROUP;
#pragma unroll
      for (int u = 0; u < GROUP; u++) r1[u] = value(b1 + u);
      scatter_group<T, MAXM, GROUP>(Ysh, b0, nb, lm0, nm, r0, acc);
#pragma unroll
      for (int u = 0; u < GROUP; u++) r0[u] = value(b2 + u);
      scatter_group<T, MAXM, GROUP>(Ysh, b1, nb, lm0, nm, r1, acc);
    }
  }
  if (t < ncol) {
    T *Ai = a.A + (long long) blockIdx.x * a.nlm * a.C;
#pragma unroll
    for (int m = 0; m < MAXM; m++)
      if (m < nm) Ai[(lm0 + m) * a.C + n] = acc[m];
  }
}

// A[lm][n] = sum_b Y_lm(b) Rz[b][l][n] on the matrix cores.  One wave per atom (4 atoms per block); per tile of 16
// bonds and per l:  D_l[m][n] += Y_l^T[m][b] . Rz_l[b][n]  with K = bonds (4 per MFMA step), rows m padded to 16.
// The B operand (Rz) comes straight from memory, 16 lanes reading 128 consecutive bytes of one bond row; the B operands
// of a tile are requested before the harmonics of the tile are evaluated, and each half of the next tile as soon as the
// MFMAs have consumed that half of the current one.  The A operand (Y) comes from the wave's LDS tile.  The
// accumulators of the wave are the atom's A.
// The grid walks the atoms from the LAST to the first: the radial kernel, which runs right before, writes the edge rows
// in ascending order, so the rows it wrote last are the ones still held by the memory-side cache.
// NL = lmax + 1, KB = channels / 16.   dynamic LDS: 4 * scatter_harmonics(NL) * nlm values.
// A wave evaluates the harmonics of the bonds of four tiles at once, one bond per lane: tile by tile 48 of 64 lanes had nothing to
// do (GRACE-1L in fp64, 128 atoms 19.2 -> 16.9 us, 8192 126 -> 118; GRACE-2L 32 000 659 -> 626; fp32 rows, 20 000 atoms 156 -> 142).
// From lmax 5 on, where those of 64 bonds would leave a CU one block in fp64, of a tile.
constexpr int scatter_harmonics(int nl) { return nl <= 5 ? 64 : 16; }
template<class T, int NL, int KB, RowsOf ROWS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_scatter_a_mfma(ScatterArgs<T> a)
{
  constexpr bool PAIRS = ROWS == RowsOf::pairs;
  typedef typename Mfma<T>::v4 v4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  constexpr int YB = scatter_harmonics(NL);
  T *Yw = reinterpret_cast<T *>(smem_raw) + wave * YB * a.nlm;     // [YB bonds][nlm]
  const int ia = a.natoms - 1 - (blockIdx.x * 4 + wave);
  if (ia < 0) return;
  const int i = a.a0 + ia;
  const long long w0 = a.eoff[i], w1 = a.eoff[i + 1];
  const int C = a.C;
  v4 acc[NL][KB];
#pragma unroll
  for (int l = 0; l < NL; l++)
#pragma unroll
    for (int cb = 0; cb < KB; cb++) acc[l][cb] = v4{0, 0, 0, 0};
  T breg[4][NL][KB], zreg[PAIRS ? 4 : 1][KB];
  // paired rows: row and element of the lane's four bonds, fetched a tile ahead of the rows themselves
  int rown[4], mun[4];
  auto rows_of = [&](long long eb) {
    const int nb = (int) (w1 - eb < 16 ? w1 - eb : 16);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int b = 4 * s + g;
      const long long e = eb + (b < nb ? b : 0);
      rown[s] = a.erow[e];
      mun[s] = a.emu[e];
    }
  };
  auto request = [&](long long eb, int h) {
    const int nb = (int) (w1 - eb < 16 ? w1 - eb : 16);
#pragma unroll
    for (int s = 2 * h; s < 2 * h + 2; s++) {
      if (4 * s >= nb) continue;                      // a step with no bond: neither loaded nor multiplied
      const int b = 4 * s + g;                        // k index of this lane in step s = bond of the tile
      // rows beyond the range: any valid row (Y = 0 there)
      const T *row = a.Rz + (PAIRS ? (long long) rown[s] : eb + (b < nb ? b : 0)) * a.noutp + c;
#pragma unroll
      for (int l = 0; l < NL; l++)
#pragma unroll
        for (int cb = 0; cb < KB; cb++) breg[s][l][cb] = row[l * C + cb * 16];
      if constexpr (PAIRS) {
#pragma unroll
        for (int cb = 0; cb < KB; cb++) zreg[s][cb] = a.z[mun[s] * C + cb * 16 + c];
      }
    }
  };
  if (w0 < w1) {
    if constexpr (PAIRS) rows_of(w0);
    request(w0, 0);
    request(w0, 1);
  }
  for (long long eb = w0; eb < w1; eb += 16) {
    const int nb = (int) (w1 - eb < 16 ? w1 - eb : 16);
    const int at = (int) (eb - w0) & (YB - 1);      // place of the tile in its round of harmonics
    if (at == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane < YB) {
        if (eb + lane < w1) {
          const double *u = a.rh + 3 * (eb + lane);
          sh_eval<false, T, NL - 1>(a.sh, u[0], u[1], u[2], Yw + lane * a.nlm, nullptr);
        } else {
          for (int q = 0; q < a.nlm; q++) Yw[lane * a.nlm + q] = (T) 0;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    const bool more = eb + 16 < w1;
    if constexpr (PAIRS) {
      if (more) rows_of(eb + 16);
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int s = 2 * h; s < 2 * h + 2; s++) {
        if (4 * s >= nb) continue;
        const T *yb = Yw + (at + 4 * s + g) * a.nlm;
#pragma unroll
        for (int l = 0; l < NL; l++) {
          const T y = c < 2 * l + 1 ? yb[l * l + c] : (T) 0;       // A operand: row m = c
#pragma unroll
          for (int cb = 0; cb < KB; cb++) {
            T r = breg[s][l][cb];
            if constexpr (PAIRS) r *= zreg[s][cb];
            acc[l][cb] = Mfma<T>::mma(y, r, acc[l][cb]);
          }
        }
      }
      if (more) request(eb + 16, h);
    }
  }
  T *Ai = a.A + (long long) ia * a.nlm * C;
#pragma unroll
  for (int l = 0; l < NL; l++) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int m = a.drow[4 * g + v];
        if (m < 2 * l + 1) {
#pragma unroll
          for (int cb = 0; cb < KB; cb++) Ai[(l * l + m) * C + cb * 16 + c] = acc[l][cb][v];
        }
      }
  }
}

// k_scatter_a_mfma with the B operand formed from the radial tables: lane (g, c) supplies, in step s, the columns
// l C + cb 16 + c of bond 4 s + g, i.e. per (l, cb) four table entries of the bond's interval (16 lanes read 128
// consecutive bytes of a table row; the 2.6 MB table of a 32-channel lmax-4 model stays in the L2), the cubic in t, times
// the species weight.  The entries of step s + 1 are requested when those of step s have been turned into operands, and
// arrive while the matrix instructions of step s run; x and the element of the lane's four bonds of the NEXT tile are
// requested a tile ahead.  No radial row is read: the rows need not exist.  Three waves per SIMD in fp32, with the harmonics of
// four tiles at once: 65 536 atoms 778 -> 674 us.  No branch in a tile, constant distances between the entries of a bond: 32 768
// atoms fp32 355 -> 331 us, 3999 atoms of 78 bonds 73.5 -> 63.4, 4001 atoms fp64 95.6 -> 95.4 (without the scheduling barrier 97);
// both column blocks of a 32-channel step requested a step ahead in fp32: 32 768 atoms 335 -> 327 us.  In fp64 with 16
// channels a tile ends behind its last step with a bond (58 bonds an atom: 15 steps for 16): lmax 6, 3456 atoms 84.3 -> 77.8 us, 128 atoms
// 32.6 -> 29.1, lmax 4 56.8 -> 52.9 and 19.9 -> 18.9; not with 32, 93.3 -> 92.6 and 26.5 -> 29.4.
template<class T, int NL, int KB> __global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 2) void k_scatter_a_tab(ScatterArgs<T> a)
{
  typedef typename Mfma<T>::v4 v4;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  constexpr int YB = scatter_harmonics(NL);
  T *Yw = reinterpret_cast<T *>(smem_raw) + wave * YB * a.nlm;     // [YB bonds][nlm]
  const int ia = a.natoms - 1 - (blockIdx.x * 4 + wave);
  if (ia < 0) return;
  const int i = a.a0 + ia;
  const long long w0 = a.eoff[i], w1 = a.eoff[i + 1];
  const int C = a.C;
  const RadialTable<T> tb = a.tb;
  v4 acc[NL][KB];
#pragma unroll
  for (int l = 0; l < NL; l++)
#pragma unroll
    for (int cb = 0; cb < KB; cb++) acc[l][cb] = v4{0, 0, 0, 0};
  double xs[4], xn[4] = {0, 0, 0, 0};
  int ms[4], mn[4] = {0, 0, 0, 0};
  auto geometry = [&](long long eb, double (&x)[4], int (&m)[4]) {
    const int nb = (int) (w1 - eb < 16 ? w1 - eb : 16);
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int b = 4 * s + g;
      const long long e = eb + (b < nb ? b : 0);
      x[s] = tb.x[e];
      m[s] = tb.emu[e];
    }
  };
  // one (step, 16-column block) at a time, QB of them requested ahead: QB x NL x 4 entries in flight per lane
  constexpr int QB = sizeof(T) == 4 && KB == 2 ? 2 : 1;
  constexpr bool SHORT = sizeof(T) == 8 && KB == 1;    // a tile ends behind its last step with a bond
  T raw[QB][NL][4], zc[QB];
  double tt[QB];
  auto request = [&](int q) {    // q = s KB + cb
    const int s = q / KB, cb = q % KB;
    const int k = table_interval(xs[s], tb.N, tt[q % QB]);
    zc[q % QB] = tb.z[ms[s] * C + cb * 16 + c];
    const TableRow<T> row = table_row<T, NL * KB * 16>(tb, k, c);
#pragma unroll
    for (int l = 0; l < NL; l++)
#pragma unroll
      for (int e = 0; e < 4; e++) raw[q % QB][l][e] = table_entry<NL * KB * 16>(row, e)[(l * KB + cb) * 16];
  };
  if (w0 < w1) geometry(w0, xs, ms);
  for (long long eb = w0; eb < w1; eb += 16) {
#pragma unroll
    for (int q = 0; q < QB; q++) request(q);
    if (eb + 16 < w1) geometry(eb + 16, xn, mn);
    const int at = (int) (eb - w0) & (YB - 1);      // place of the tile in its round of harmonics
    if (at == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane < YB) {
        if (eb + lane < w1) {
          const double *u = a.rh + 3 * (eb + lane);
          sh_eval<false, T, NL - 1>(a.sh, u[0], u[1], u[2], Yw + lane * a.nlm, nullptr);
        } else {
          for (int q = 0; q < a.nlm; q++) Yw[lane * a.nlm + q] = (T) 0;
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // not SHORT: a step without a bond reads the tile's first again and multiplies with harmonics of zero, no branch in the tile
    const int steps = SHORT ? ((int) (w1 - eb < 16 ? w1 - eb : 16) + 3) / 4 * KB : 4 * KB;
#pragma unroll
    for (int q = 0; q < 4 * KB; q++) {
      if (SHORT && q >= steps) break;
      const int s = q / KB, cb = q % KB;
      T bv[NL];
      const TableBond<T> bond = table_bond<T>(tt[q % QB], tb.N);
      const auto &w = raw[q % QB];
#pragma unroll
      for (int l = 0; l < NL; l++) bv[l] = table_value(table_cubic(w[l][0], w[l][1], w[l][2], w[l][3], bond), bond) * zc[q % QB];
      if (q + QB < 4 * KB && (!SHORT || q + QB < steps)) request(q + QB);
      const T *yb = Yw + (at + 4 * s + g) * a.nlm;
#pragma unroll
      for (int l = 0; l < NL; l++) {
        const T y = c < 2 * l + 1 ? yb[l * l + c] : (T) 0;       // A operand: row m = c
        acc[l][cb] = Mfma<T>::mma(y, bv[l], acc[l][cb]);
      }
      if (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);    // entries of a later step requested early spill in fp64
    }
#pragma unroll
    for (int s = 0; s < 4; s++) { xs[s] = xn[s]; ms[s] = mn[s]; }
  }
  T *Ai = a.A + (long long) ia * a.nlm * C;
#pragma unroll
  for (int l = 0; l < NL; l++) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int m = a.drow[4 * g + v];
        if (m < 2 * l + 1) {
#pragma unroll
          for (int cb = 0; cb < KB; cb++) Ai[(l * l + m) * C + cb * 16 + c] = acc[l][cb][v];
        }
      }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// per-atom dense chain.  Per-atom tensors are [atom][function][channel].
// ---------------------------------------------------------------------------------------------------------------
// Atoms are processed in tiles of 16 (one MFMA tile): tile_atoms[tile * 16 + r] is the atom of row r, or -1.  Tiles
// hold atoms of one element, so that element-dependent weights (rho reduce) are uniform per tile.
//
// Job / segment GEMM of the FC layers on the matrix cores.  Job = one output function; its value for a tile is
//   out[atom][fo][0:N] (+)= scale_job * sum_seg  seg_scale * X_src(seg)[atom][fn(seg)][0:K] . W[wtile(seg)][0:K][0:N]
// FC forward:        job f,  segments (Xl, f, Wl[tile_l f]) and (Xr, from c, Wr[tile c]) for every connection c -> f
// FC reverse, left:  job f,  segment  (g, f, Wl^T[tile_l f]), accumulated into gXl
// FC reverse, right: job r,  segments (g, to c, nof[to c] Wr^T[tile c]) for the connections c from r, accumulated
// Rows of the A operand are the 16 atoms (lane % 16).  The channel that step s takes from lane group g = lane / 16 is
// frag_k<T>: 16 bytes of the row per group in turn, so that one load instruction reads 64 consecutive bytes of each of the 16
// rows (with K / 4 consecutive channels per group it touched four times as many cache lines).  Weights are stored in that
// order ([tile][cb][s][lane]).
template<class T> __host__ __device__ constexpr int frag_k(int g, int s)
{
  constexpr int V = 16 / (int) sizeof(T);    // values of a 16-byte piece
  return (s / V) * 4 * V + g * V + s % V;
}
// KS values of the A operand of lane group g, from the row xp (16-byte aligned: rows hold a multiple of 16 channels)
template<int KS, class T> __device__ inline void frag_load(const T *xp, int g, T (&x)[KS])
{
  constexpr int V = 16 / (int) sizeof(T);
  typedef T piece __attribute__((ext_vector_type(16 / sizeof(T))));
#pragma unroll
  for (int p = 0; p < KS / V; p++) {
    const piece w = *reinterpret_cast<const piece *>(xp + (p * 4 + g) * V);
#pragma unroll
    for (int q = 0; q < V; q++) x[p * V + q] = w[q];
  }
}
template<class T> struct GemmJobs {
  const int *job_out;         // [njobs] output function
  const T *job_scale;         // [njobs]
  const int *seg_off;         // [njobs + 1]
  const int *seg_src;         // [nseg] 0: X0 (K0 channels), 1: X1 (K1 channels)
  const int *seg_fn;          // [nseg] function of the source tensor
  const int *seg_w;           // [nseg] weight tile
  const T *seg_scale;         // [nseg]
  const T *WF0, *WF1;         // fragments of the weights used with X0 / X1
  int njobs;
  int max_seg;                // most segments of one job
  int drow[16];               // accumulator row of (lane / 16, register), probed on the device
  const int4 *seg;            // [nseg] source, function, weight tile as one entry (k_gemm_few, k_gemm_wide)
  const int *job_dst;         // [njobs] output tensor
  const T *job_add;           // [njobs] factor of the row of GemmIO::add that is added, or null (k_gemm_few)
};
// The tensors of a launch whose job list reads up to four sources and writes up to four outputs, all of one width
template<class T> struct GemmIO {
  const T *X[4], *WF[4];
  int nf[4];
  T *out[4];
  int nfo[4];
  const T *add;               // out[0] += job_add x this row (shape of out[0])
  unsigned accumulate;        // bit d: added to out[d], not set
};

constexpr int kGemmMaxSeg = 4;      // most weight tiles staged in LDS at a time (the launch passes the number, mseg)
constexpr int kGemmTilesPerWave = 2;

template<class T, int KB0, int KB1, int NB>
__global__ __launch_bounds__(512) void k_gemm_jobs(GemmJobs<T> J, const T *X0, int nf0, const T *X1, int nf1, T *out, int nfo,
                                                   const int *tile_atoms, int ntiles, int accumulate, int reps, int mseg)
{
  // mseg <= kGemmMaxSeg weight tiles are staged at a time (dynamic LDS: mseg tiles; wide tiles are staged fewer at a
  // time so that several blocks fit a CU).  reps > 1 (only when every job has one segment): the block stages its
  // weight tile once and walks `reps` groups of atom tiles with it
  typedef typename Mfma<T>::v4 v4;
  constexpr int TPW = kGemmTilesPerWave;
  constexpr int KS0 = KB0 * 4, KS1 = KB1 * 4, KSM = KS0 > KS1 ? KS0 : KS1, K0 = KB0 * 16, K1 = KB1 * 16, N = NB * 16;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *wl = reinterpret_cast<T *>(smem_raw);      // [mseg][NB][KSM][64]
  __shared__ int s_src[kGemmMaxSeg], s_fn[kGemmMaxSeg];
  __shared__ T s_scale[kGemmMaxSeg];
  const int job = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int sg0 = J.seg_off[job], sg1 = J.seg_off[job + 1];
  const int fo = J.job_out[job];
  const T js = J.job_scale[job];
  for (int rep = 0; rep < reps; rep++) {
    const int tile0 = ((blockIdx.y * reps + rep) * nwave + wave) * TPW;
    if (rep > 0 && (blockIdx.y * reps + rep) * nwave * TPW >= ntiles) break;    // uniform over the block
    v4 acc[TPW][NB];
    int arow[TPW];            // atom of this lane's A row
#pragma unroll
    for (int i = 0; i < TPW; i++) {
      const int tile = tile0 + i;
      arow[i] = tile < ntiles ? tile_atoms[tile * 16 + c] : -1;
#pragma unroll
      for (int cb = 0; cb < NB; cb++) acc[i][cb] = v4{0, 0, 0, 0};
    }
    for (int sg = sg0; sg < sg1; sg += mseg) {
      const int ns = sg1 - sg < mseg ? sg1 - sg : mseg;
      if (rep == 0) {
        __syncthreads();
        for (int q = 0; q < ns; q++) {
          const int src = J.seg_src[sg + q];
          const int ks = src == 0 ? KS0 : KS1;
          const T *wf = (src == 0 ? J.WF0 : J.WF1) + (long long) J.seg_w[sg + q] * NB * ks * 64;
          for (int e = threadIdx.x; e < NB * ks * 64; e += blockDim.x) {
            const int cb = e / (ks * 64), rem = e % (ks * 64);
            wl[(q * NB + cb) * KSM * 64 + rem] = wf[e];
          }
          if (threadIdx.x == 0) { s_src[q] = src; s_fn[q] = J.seg_fn[sg + q]; s_scale[q] = J.seg_scale[sg + q]; }
        }
        __syncthreads();
      }
#pragma unroll
      for (int i = 0; i < TPW; i++) {
        for (int q = 0; q < ns; q++) {
          const T sc = s_scale[q];
          const T *wq = wl + q * NB * KSM * 64 + lane;
          if (s_src[q] == 0) {
            T x[KS0];
            if (arow[i] >= 0) {
              frag_load<KS0>(X0 + ((long long) arow[i] * nf0 + s_fn[q]) * K0, g, x);
#pragma unroll
              for (int s = 0; s < KS0; s++) x[s] *= sc;
            } else {
#pragma unroll
              for (int s = 0; s < KS0; s++) x[s] = (T) 0;
            }
#pragma unroll
            for (int cb = 0; cb < NB; cb++)
#pragma unroll
              for (int s = 0; s < KS0; s++) acc[i][cb] = Mfma<T>::mma(x[s], wq[(cb * KSM + s) * 64], acc[i][cb]);
          } else {
            T x[KS1];
            if (arow[i] >= 0) {
              frag_load<KS1>(X1 + ((long long) arow[i] * nf1 + s_fn[q]) * K1, g, x);
#pragma unroll
              for (int s = 0; s < KS1; s++) x[s] *= sc;
            } else {
#pragma unroll
              for (int s = 0; s < KS1; s++) x[s] = (T) 0;
            }
#pragma unroll
            for (int cb = 0; cb < NB; cb++)
#pragma unroll
              for (int s = 0; s < KS1; s++) acc[i][cb] = Mfma<T>::mma(x[s], wq[(cb * KSM + s) * 64], acc[i][cb]);
          }
        }
      }
    }
    // accumulator (g, v) holds row drow[4 g + v] of the tile, column cb * 16 + c
#pragma unroll
    for (int i = 0; i < TPW; i++) {
      const int tile = tile0 + i;
      if (tile >= ntiles) continue;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int at = tile_atoms[tile * 16 + J.drow[4 * g + v]];
        if (at < 0) continue;
        T *o = out + ((long long) at * nfo + fo) * N + c;
#pragma unroll
        for (int cb = 0; cb < NB; cb++) {
          const T val = js * acc[i][cb][v];
          o[cb * 16] = accumulate ? o[cb * 16] + val : val;
        }
      }
    }
  }
}

// ---- the jobs of a launch with one width of inputs and one of outputs, in the two shapes that few and many atom tiles need ----
// k_gemm_few: a wave owns ONE 16 x 16 tile of the output (an atom tile and a column block), so that a structure of a few
// atom tiles still puts a wave on every SIMD, and the segments of a job are dealt to S waves whose sums meet in LDS (in the
// order of the waves).  No operand passes through LDS and no wave waits for another before the end: both operands come from
// L1 / L2, 8 steps of them requested while the 8 before are multiplied, the description of a segment one request earlier.
// What bounds it: the L1 (16 kB of operands per 16 x 16 x 64 tile, as many cycles as its matrix instructions take with all
// four SIMDs busy) and, for jobs of one segment, the latency of a launch.  GRACE-3L, 96 atoms (8 tiles): 36 jobs of 47
// segments 80 us as k_gemm_jobs (36 blocks), 50 as k_gemm_wide, 25 so; 36 jobs of one segment 12.4 / 11.4 / 7.2 us.
template<class T, int KB, int NB, int S>
__global__ __launch_bounds__(64 * NB * S) void k_gemm_few(GemmJobs<T> J, GemmIO<T> io, const int *tile_atoms)
{
  typedef typename Mfma<T>::v4 v4;
  constexpr int KS = KB * 4, K = KB * 16, N = NB * 16, HS = KS > 8 ? 8 : KS, U = KS / HS, V = 16 / (int) sizeof(T);
  typedef T piece __attribute__((ext_vector_type(16 / sizeof(T))));
  __shared__ T part[S > 1 ? (S - 1) * NB * 256 : 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4, cb = wave % NB, pt = wave / NB;
  const int job = blockIdx.x, tile = blockIdx.y;
  const int sg0 = J.seg_off[job] + pt, sg1 = J.seg_off[job + 1];
  const int first = tile_atoms[tile * 16], mine = tile_atoms[tile * 16 + c];
  const int row = mine >= 0 ? mine : first;           // a row without an atom: computed from the tile's first, never stored
  const int nu = sg1 > sg0 ? (sg1 - sg0 + S - 1) / S * U : 0;      // units of HS steps of this wave
  const int fo = J.job_out[job], dst = J.job_dst[job];
  const T js = J.job_scale[job];
  T *out = io.out[dst] + fo * N + cb * 16 + c;
  const long long nfoN = (long long) io.nfo[dst] * N;
  int at[4];
#pragma unroll
  for (int v = 0; v < 4; v++) at[v] = tile_atoms[tile * 16 + J.drow[4 * g + v]];
  // what is added to the sum: requested first, added last (in fp32 a sum that starts from it is 20 % less accurate)
  v4 acc = {0, 0, 0, 0}, y = {0, 0, 0, 0};
  if (pt == 0) {
    const bool accumulate = io.accumulate >> dst & 1;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const long long o = (at[v] >= 0 ? at[v] : first) * nfoN;
      if (accumulate) y[v] = out[o];
      if (J.job_add && dst == 0) y[v] += J.job_add[job] * io.add[o + fo * N + cb * 16 + c];
    }
  }
  T xa[HS], wa[HS], xb[HS], wb[HS], sa = 0, sb = 0, scn = 0;
  int4 mn = {0, 0, 0, 0};
  auto describe = [&](int u) {
    const int sg = sg0 + (u / U) * S;
    mn = J.seg[sg];
    scn = J.seg_scale[sg];
  };
  auto load = [&](int u, T (&x)[HS], T (&w)[HS], T &sc) {
    const int src = mn.x, h = U == 1 ? 0 : u % U;
    const T *xp = io.X[src] + ((long long) row * io.nf[src] + mn.y) * K + (h * (HS / V) * 4 + g) * V;
    const T *wp = io.WF[src] + (((long long) mn.z * NB + cb) * KS + h * HS) * 64 + lane;
#pragma unroll
    for (int p = 0; p < HS / V; p++) {
      const piece q = *reinterpret_cast<const piece *>(xp + p * 4 * V);
#pragma unroll
      for (int e = 0; e < V; e++) x[p * V + e] = q[e];
    }
#pragma unroll
    for (int s = 0; s < HS; s++) w[s] = wp[s * 64];
    sc = scn;
    if (u + 1 < nu) describe(u + 1);
  };
  auto multiply = [&](const T (&x)[HS], const T (&w)[HS], T sc) {
#pragma unroll
    for (int s = 0; s < HS; s++) acc = Mfma<T>::mma(x[s] * sc, w[s], acc);
  };
  if (nu > 0) {
    describe(0);
    load(0, xa, wa, sa);
  }
  for (int u = 0; u < nu; u += 2) {
    if (u + 1 < nu) load(u + 1, xb, wb, sb);
    multiply(xa, wa, sa);
    if (u + 2 < nu) load(u + 2, xa, wa, sa);
    if (u + 1 < nu) multiply(xb, wb, sb);
  }
  if (S > 1) {
    if (pt > 0) {
#pragma unroll
      for (int v = 0; v < 4; v++) part[((pt - 1) * NB + cb) * 256 + v * 64 + lane] = acc[v];
    }
    lds_barrier();
    if (pt > 0) return;
#pragma unroll
    for (int q = 0; q < S - 1; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) acc[v] += part[(q * NB + cb) * 256 + v * 64 + lane];
  }
#pragma unroll
  for (int v = 0; v < 4; v++)
    if (at[v] >= 0) out[at[v] * nfoN] = js * acc[v] + y[v];
}

// k_gemm_wide (64 channels in, 64 out): a wave owns two atom tiles (one in fp32) and all 64 columns, the four waves of a block share the
// weight tile of a segment in LDS (two tiles of 32 kB in fp64, one filled while the other is read).  The rows of the next
// segment are requested into the registers that hold this one's, each piece as soon as its last product has been issued,
// and the next weight tile waits in registers until the products are done: every load has a whole segment (8192 cycles of
// matrix work in fp64) to arrive, which k_gemm_jobs, whose loads stood at the head of every segment, left exposed.
// GRACE-3L, 3001 atoms fp64: 72 jobs of 23 segments 1281 -> 857 us (49 TF; the rows of its source are read once: 2.6 GB, 0.5
// ms at the copy rate), 1685 jobs of one segment 1119 -> 909 us (writes 2.6 GB).
// fp32 matrix instructions take half as long, so more waves have to stand behind the same loads: with one tile a wave holds 117
// registers and four of them share a SIMD.  The two largest reduces of 10 000 atoms (reduce_4_L2, reduce_3_L2),
// fp32: 1.43 and 1.29 ms, against 1.67 and 1.51 with two tiles (198 registers, two waves), 2.97 and 2.70 with two tiles forced
// into three waves (75 registers spilled), 1.95 and 1.76 as k_gemm_jobs; the pass 91.5, 94.9, 102.1 and 101.8 ms.
// Jobs of one segment walk `reps` groups of atom tiles with the tile they have staged.
template<class T> constexpr int gemm_wide_tiles() { return sizeof(T) == 4 ? 1 : 2; }
template<class T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2))) void k_gemm_wide(GemmJobs<T> J, GemmIO<T> io, const int *tile_atoms, int ntiles,
                                                                                        int reps)
{
  typedef typename Mfma<T>::v4 v4;
  constexpr int KS = 16, K = 64, N = 64, NB = 4, MT = gemm_wide_tiles<T>(), V = 16 / (int) sizeof(T), NP = KS / V, WT = NB * KS * 64, WP = WT / V / 256;
  typedef T piece __attribute__((ext_vector_type(16 / sizeof(T))));
  __shared__ __align__(16) T wl[2][WT];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int job = blockIdx.x;
  const int sg0 = J.seg_off[job], nseg = J.seg_off[job + 1] - sg0;
  const int fo = J.job_out[job], dst = J.job_dst[job];
  const T js = J.job_scale[job];
  T *out = io.out[dst];
  const int nfo = io.nfo[dst];
  const bool accumulate = io.accumulate >> dst & 1;
  auto tile_of = [&](int rep, int i) { return ((blockIdx.y * reps + rep) * 4 + wave) * MT + i; };
  // groups of atom tiles this block walks (jobs of one segment), or segments
  const int left = ntiles - (int) blockIdx.y * reps * 4 * MT, ngroups = left >= reps * 4 * MT ? reps : (left + 4 * MT - 1) / (4 * MT);
  const int steps = reps > 1 ? ngroups : nseg;
  int row[MT];
  auto rows_of = [&](int rep) {
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int tile = tile_of(rep, i), tc = tile < ntiles ? tile : ntiles - 1;
      const int first = tile_atoms[tc * 16], mine = tile_atoms[tc * 16 + c];
      row[i] = mine >= 0 ? mine : first;              // rows without an atom: never stored
    }
  };
  v4 acc[MT][NB];
  T x[MT][KS];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int cb = 0; cb < NB; cb++) acc[i][cb] = v4{0, 0, 0, 0};
  };
  // What is added to the sums (value (cb, v) of a tile at x[i][4 cb + v]): requested into the registers of the operands as the
  // last segment frees them.  (Sums that start from it are as quick and, in fp32, 20 % less accurate.)
  auto added_request = [&](int rep, int q) {
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int tile = tile_of(rep, i), tc = tile < ntiles ? tile : ntiles - 1;
      const int at = tile_atoms[tc * 16 + J.drow[4 * g + q % 4]];
      const long long o = ((long long) (at >= 0 ? at : tile_atoms[tc * 16]) * nfo + fo) * N + c + (q / 4) * 16;
      x[i][q] = out[o];
    }
  };
  auto store = [&](int rep) {
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int tile = tile_of(rep, i);
      if (tile >= ntiles) continue;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int at = tile_atoms[tile * 16 + J.drow[4 * g + v]];
        if (at < 0) continue;
        const long long o = ((long long) at * nfo + fo) * N + c;
#pragma unroll
        for (int cb = 0; cb < NB; cb++) out[o + cb * 16] = accumulate ? js * acc[i][cb][v] + x[i][4 * cb + v] : js * acc[i][cb][v];
      }
    }
  };
  // fp32: the sum of every segment is added to the total by itself.  One long chain of accumulations over the segments of
  // joined contractions was 5 % less accurate than the separate launches (forces of 701 and 1500 atoms against fp64).
  v4 total[MT][NB];
  auto take = [&]() {
    if (sizeof(T) == 4) {
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int cb = 0; cb < NB; cb++) total[i][cb] += acc[i][cb];
      clear();
    }
  };
  clear();
  if (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int cb = 0; cb < NB; cb++) total[i][cb] = v4{0, 0, 0, 0};
  }
  if (nseg == 0) {                                    // a job that only clears
    for (int rep = 0; rep < (reps > 1 ? ngroups : 1); rep++) {
      if (accumulate) {
#pragma unroll
        for (int q = 0; q < KS; q++) added_request(rep, q);
      }
      store(rep);
    }
    return;
  }
  piece wn[WP];
  auto weights_request = [&](const int4 &m) {
    const T *wf = io.WF[m.x] + (long long) m.z * WT;
#pragma unroll
    for (int p = 0; p < WP; p++) wn[p] = *reinterpret_cast<const piece *>(wf + (p * 256 + threadIdx.x) * V);
  };
  auto weights_store = [&](int buf) {
#pragma unroll
    for (int p = 0; p < WP; p++) *reinterpret_cast<piece *>(&wl[buf][(p * 256 + threadIdx.x) * V]) = wn[p];
  };
  const T *xp[MT];
  auto sources = [&](const int4 &m) {
    const T *X = io.X[m.x];
    const int nf = io.nf[m.x];
#pragma unroll
    for (int i = 0; i < MT; i++) xp[i] = X + ((long long) row[i] * nf + m.y) * K + g * V;
  };
  auto x_request = [&](int p) {
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const piece q = *reinterpret_cast<const piece *>(xp[i] + p * 4 * V);
#pragma unroll
      for (int e = 0; e < V; e++) x[i][p * V + e] = q[e];
    }
  };
  int4 m = J.seg[sg0];
  T sc = J.seg_scale[sg0];
  rows_of(0);
  weights_request(m);
  sources(m);
#pragma unroll
  for (int p = 0; p < NP; p++) x_request(p);
  weights_store(0);
  for (int t = 0; t < steps; t++) {
    if (reps == 1 || t == 0) lds_barrier();
    const bool more = t + 1 < steps;
    const T scn = reps == 1 && more ? J.seg_scale[sg0 + t + 1] : sc;
    if (more) {
      if (reps == 1) {
        m = J.seg[sg0 + t + 1];
        weights_request(m);
      } else {
        rows_of(t + 1);
      }
      sources(m);
    }
    const T *wq = wl[reps == 1 ? t & 1 : 0] + lane;
    T w[2][NB];
#pragma unroll
    for (int cb = 0; cb < NB; cb++) w[0][cb] = wq[cb * KS * 64];
#pragma unroll
    for (int s = 0; s < KS; s++) {
      if (s + 1 < KS) {
#pragma unroll
        for (int cb = 0; cb < NB; cb++) w[(s + 1) & 1][cb] = wq[(cb * KS + s + 1) * 64];
      }
#pragma unroll
      for (int i = 0; i < MT; i++) {
        const T xs = x[i][s] * sc;
#pragma unroll
        for (int cb = 0; cb < NB; cb++) acc[i][cb] = Mfma<T>::mma(xs, w[s & 1][cb], acc[i][cb]);
      }
      if (more) {
        if ((s + 1) % V == 0) x_request(s / V);
      } else if (accumulate) {
        added_request(0, s);       // launches with several groups add nothing
      }
    }
    if (reps > 1) {
      store(t);
      clear();
    } else {
      if (nseg > 1) take();
      if (more) weights_store((t + 1) & 1);
    }
    sc = scn;
  }
  if (sizeof(T) == 4 && nseg > 1) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int cb = 0; cb < NB; cb++) acc[i][cb] = total[i][cb];
  }
  if (reps == 1) store(0);
}

// Block index -> (function q, atom group) for grids of nq * 8 * ceil(groups / 8) blocks.  Workgroups go to the 8 XCDs
// round-robin by linear index and every XCD has its own L2: the blocks of one atom group (all its functions q) are
// given consecutive indices on ONE XCD, so that the per-atom tensors they share are fetched into one L2 once.
__device__ inline void xcd_block(int nq, int &q, int &group)
{
  const int L = blockIdx.x, xcd = L & 7, rest = L >> 3;
  q = rest % nq;
  group = (rest / nq) * 8 + xcd;
}

struct ProdDev {
  // forward: terms sorted by output (CSR off over nout; only live outputs have terms)
  const int *off, *l, *r;
  const double *c;
  // reverse: terms by left operand (loff over nleft) and by right operand (roff over nright)
  const int *loff, *l_o, *l_r;
  const double *l_c;
  const int *roff, *r_o, *r_l;
  const double *r_c;
  int nout, nleft, nright;
};

// out[a][o][k] = sum_t c_t L[a][l_t][k] R[a][r_t][k]      grid: xcd_block over (nout, atom groups), block = C x AT
template<class T> __global__ void k_prod_fwd(ProdDev P, const T *L, const T *R, T *out, int natoms, int C, int sl, int sr)
{
  const int k = threadIdx.x % C, al = threadIdx.x / C;
  int o, ag;
  xcd_block(P.nout, o, ag);
  const int at = ag * (blockDim.x / C) + al;
  if (at >= natoms) return;
  const T *La = L + (long long) at * sl * C + k, *Ra = R + (long long) at * sr * C + k;
  T acc = (T) 0;
  for (int t = P.off[o]; t < P.off[o + 1]; t++) acc += (T) P.c[t] * La[(long long) P.l[t] * C] * Ra[(long long) P.r[t] * C];
  out[((long long) at * P.nout + o) * C + k] = acc;
}

// gL[a][q][k] += sum_{t: l_t = q} c_t g[a][o_t][k] R[a][r_t][k]   (side 0), gR likewise with L (side 1)
// grid (nleft or nright, atom groups)
template<class T> __global__ void k_prod_bwd(ProdDev P, int side, const T *other, const T *g, T *gX, int natoms, int C, int so,
                                             int sx)
{
  const int k = threadIdx.x % C, al = threadIdx.x / C;
  int q, ag;
  xcd_block(side == 0 ? P.nleft : P.nright, q, ag);
  const int at = ag * (blockDim.x / C) + al;
  if (at >= natoms) return;
  const int *off = side == 0 ? P.loff : P.roff, *oo = side == 0 ? P.l_o : P.r_o, *ot = side == 0 ? P.l_r : P.r_l;
  const double *cc = side == 0 ? P.l_c : P.r_c;
  if (off[q] == off[q + 1]) return;
  const T *Oa = other + (long long) at * so * C + k, *ga = g + (long long) at * P.nout * C + k;
  T acc = (T) 0;
  for (int t = off[q]; t < off[q + 1]; t++) acc += (T) cc[t] * ga[(long long) oo[t] * C] * Oa[(long long) ot[t] * C];
  gX[((long long) at * sx + q) * C + k] += acc;
}

template<class T> struct ReduceDev {
  // per source s: collected functions fn[s][c] (unique), weights in fragment order
  //   WF[s][mu][c][cb][ks][lane]  = W_s[mu][c][n = frag_k(g, ks)][k = cb 16 + lane % 16] (norm folded, k >= nrho zero)
  const T *WF[4];
  const int *fn[4];
  int ncol[4], nin[4], stride[4];    // collected functions, (padded) channels, functions per atom of the source
  int nsrc, nrho, nbr;               // width of the result, its 16-column blocks
  int sel, ostride, ooff;            // array of the result (0: fp64 rows, 1: rows of T) and its row: array[atom * ostride + ooff + k]
  int drow[16];                      // accumulator row of (lane / 16, register)
};
constexpr int kReduceSet = 8;        // reduces of one launch
template<class T> struct ReduceSet { ReduceDev<T> r[kReduceSet]; };

// out[atom][k] = sum_s sum_c sum_n W_s[mu][c][n][k] X_s[atom][fn c][n] on the matrix cores.  Grid (tiles of 16 atoms, reduces
// of the set, parts): the kReduceWaves waves of the `nparts` blocks of a (tile, reduce) split its (s, c) list, partial tiles are
// summed through LDS; with several parts they go to part_sums [reduce][part][tile][16][32] and k_reduce_sum adds them.
// KBA / KBF: 16-channel blocks of source 0 (A) and of the other sources.
// A wave waits some 2 us for the operands of one collected function, so what bounds few atoms is the length of a wave's
// list: 89 functions over one block of eight waves took 34 us with 128 atoms.
constexpr int kReduceWaves = 8;    // waves of a k_reduce_fwd block
template<class T, int KBA, int KBF>
__global__ __launch_bounds__(64 * kReduceWaves) void k_reduce_fwd(ReduceSet<T> set, const int *mu, const int *tile_atoms, const T *X0, const T *X1,
                                                    const T *X2, const T *X3, double *out0, T *out1, int nparts, double *part_sums)
{
  typedef typename Mfma<T>::v4 v4;
  constexpr int KSM = (KBA > KBF ? KBA : KBF) * 4;
  __shared__ double part[kReduceWaves][2][16][17];
  const ReduceDev<T> &R = set.r[blockIdx.y];
  const int tile = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int arow = tile_atoms[tile * 16 + c];
  const int a0 = tile_atoms[tile * 16];
  const int m = mu[a0];
  const T *X[4] = {X0, X1, X2, X3};
  v4 acc[2] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
  int s = 0, cc = wave + kReduceWaves * blockIdx.z;
  while (true) {
    while (s < R.nsrc && cc >= R.ncol[s]) cc -= R.ncol[s++];
    if (s >= R.nsrc) break;
    const int ks = (s == 0 ? KBA : KBF) * 4, K = ks * 4;
    const T *wf = R.WF[s] + ((long long) m * R.ncol[s] + cc) * R.nbr * ks * 64 + lane;
    T x[KSM];
    if (arow >= 0) {
      const T *xp = X[s] + ((long long) arow * R.stride[s] + R.fn[s][cc]) * K;
#pragma unroll
      for (int q = 0; q < KSM; q++) x[q] = q < ks ? xp[frag_k<T>(g, q)] : (T) 0;
    } else {
#pragma unroll
      for (int q = 0; q < KSM; q++) x[q] = (T) 0;
    }
#pragma unroll
    for (int cb = 0; cb < 2; cb++)
      if (cb < R.nbr) {
#pragma unroll
        for (int q = 0; q < KSM; q++)
          if (q < ks) acc[cb] = Mfma<T>::mma(x[q], wf[(cb * ks + q) * 64], acc[cb]);
      }
    cc += kReduceWaves * nparts;
  }
#pragma unroll
  for (int cb = 0; cb < 2; cb++)
#pragma unroll
    for (int v = 0; v < 4; v++) part[wave][cb][R.drow[4 * g + v]][c] = (double) acc[cb][v];
  __syncthreads();
  double *sums = part_sums + (((long long) blockIdx.y * nparts + blockIdx.z) * gridDim.x + tile) * (16 * 32);
  for (int e = threadIdx.x; e < 16 * R.nrho; e += 64 * kReduceWaves) {
    const int r = e / R.nrho, k = e % R.nrho;
    const int at = tile_atoms[tile * 16 + r];
    if (at < 0) continue;
    double v = 0.0;
    for (int w = 0; w < kReduceWaves; w++) v += part[w][k >> 4][r][k & 15];
    const long long to = (long long) at * R.ostride + R.ooff + k;
    if (nparts > 1) sums[r * 32 + k] = v;
    else if (R.sel == 0) out0[to] = v;
    else out1[to] = (T) v;
  }
}

// the parts of k_reduce_fwd, added in their order: grid (tiles, reduces of the set), 512 threads
template<class T>
__global__ __launch_bounds__(512) void k_reduce_sum(ReduceSet<T> set, const int *tile_atoms, const double *part_sums, int nparts, double *out0, T *out1)
{
  const ReduceDev<T> &R = set.r[blockIdx.y];
  const int tile = blockIdx.x, r = threadIdx.x >> 5, k = threadIdx.x & 31;
  const int at = tile_atoms[tile * 16 + r];
  if (at < 0 || k >= R.nrho) return;
  const double *p = part_sums + ((long long) blockIdx.y * nparts * gridDim.x + tile) * (16 * 32) + threadIdx.x;
  double v = 0.0;
#pragma unroll 4
  for (int q = 0; q < nparts; q++) v += p[(long long) q * gridDim.x * (16 * 32)];
  const long long to = (long long) at * R.ostride + R.ooff + k;
  if (R.sel == 0) out0[to] = v;
  else out1[to] = (T) v;
}

struct RowMap { int r[16]; };    // accumulator row of (lane / 16, register)

// One adjoint row of the reverse of a set of reduces: function fn of source s, its 16-channel blocks cb0 .. cb0 + nb - 1 (nb <= 2),
// fed by up to two reduces (ncon; 0: the row is written as zeros): their result rows g_sel[atom * stride + off + k], k < nout,
// nks MFMA steps each (step q takes k = 4 q + lane / 16).  Weights [mu][con][cb < 2][step < 8][lane] from w on.
struct ReduceBwdJob {
  int s, fn, nin, stride_out, cb0, nb, ncon;
  int sel[2], stride[2], off[2], nout[2], nks[2];
  long long w, wmu;    // first weight, weights of one element
};

// G_s[atom][fn][n] (+)= sum over the job's reduces of sum_k g[atom][k] W_s[mu][c][n][k]; overwrite: the rows are written.
// Grid (jobs, groups of tiles), a wave per job and `tpw` tiles of 16 atoms: the weights of a job fed by one reduce stay in
// registers for its tiles (of one element, mostly).  As a wave per (job, tile) the kernel was bound by the latency of its
// chain tile -> element -> weights in 64-thread blocks: see launch_reduce_bwd for the figures.
template<class T>
__global__ __launch_bounds__(256) void k_reduce_bwd(const ReduceBwdJob *__restrict__ jobs, const T *__restrict__ W, RowMap drow, const int *__restrict__ mu,
                                                    const int *__restrict__ tile_atoms, int ntiles, int tpw, const double *__restrict__ g0,
                                                    const T *__restrict__ g1, T *G0, T *G1, T *G2, T *G3, int overwrite)
{
  typedef typename Mfma<T>::v4 v4;
  const ReduceBwdJob J = jobs[blockIdx.x];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int t0 = (blockIdx.y * 4 + wave) * tpw, t1 = min(ntiles, t0 + tpw);
  if (t0 >= t1) return;
  T *G = J.s == 0 ? G0 : J.s == 1 ? G1 : J.s == 2 ? G2 : G3;
  T w[2][8];
  int held = -1;    // element whose weights w holds (jobs fed by one reduce)
  for (int t = t0; t < t1; t++) {
    const int arow = tile_atoms[t * 16 + c];
    const int m = __builtin_amdgcn_readfirstlane(mu[__builtin_amdgcn_readfirstlane(arow)]);    // a tile's first entry is an atom
    v4 acc[2] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
#pragma unroll
    for (int q = 0; q < 2; q++) {
      if (q >= J.ncon) continue;
      T x[8];
#pragma unroll
      for (int k4 = 0; k4 < 8; k4++) {
        const int k = 4 * k4 + g;
        x[k4] = (T) 0;
        if (k4 < J.nks[q] && arow >= 0 && k < J.nout[q]) {
          const long long at = (long long) arow * J.stride[q] + J.off[q] + k;
          x[k4] = J.sel[q] == 0 ? (T) g0[at] : g1[at];
        }
      }
      if (J.ncon > 1 || held != m) {
        const T *wp = W + J.w + m * J.wmu + q * (2 * 8 * 64) + lane;
#pragma unroll
        for (int cb = 0; cb < 2; cb++)
#pragma unroll
          for (int k4 = 0; k4 < 8; k4++) w[cb][k4] = cb < J.nb && k4 < J.nks[q] ? wp[(cb * 8 + k4) * 64] : (T) 0;
        held = m;
      }
#pragma unroll
      for (int cb = 0; cb < 2; cb++)
        if (cb < J.nb) {
#pragma unroll
          for (int k4 = 0; k4 < 8; k4++)
            if (k4 < J.nks[q]) acc[cb] = Mfma<T>::mma(x[k4], w[cb][k4], acc[cb]);
        }
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int at = __shfl(arow, drow.r[4 * g + v], 64);
      if (at < 0) continue;
      T *out = G + ((long long) at * J.stride_out + J.fn) * J.nin + J.cb0 * 16 + c;
#pragma unroll
      for (int cb = 0; cb < 2; cb++)
        if (cb < J.nb) out[cb * 16] = overwrite ? acc[cb][v] : out[cb * 16] + acc[cb][v];
    }
  }
}


// gX[atom][f][c] = sum of the parts of chain_bwd_part (part p at parts + p * stride), plus what gX holds for the functions of
// keep (the reduces' adjoints)
template<class T> __global__ void k_chain_sum(const T *__restrict__ parts, long long stride, int nparts, unsigned long long keep, int nf, int C,
                                              long long total, T *__restrict__ gX)
{
  const long long q = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (q >= total) return;
  T v = keep >> ((q / C) % nf) & 1 ? gX[q] : (T) 0;
  for (int p = 0; p < nparts; p++) v += parts[p * stride + q];
  gX[q] = v;
}

struct EnergyDev {
  const double *W[7];         // [n_in][n_out]
  double norm[7];
  int nin[7], nout[7];
  int nlay, act, ln, nrho, width;    // width: largest layer width (LDS row of the kernel)
  int wlds;                   // weights staged in LDS (sum of n_in n_out values, twice: as stored and transposed), or 0
  double out_scale;
  const double *shift;        // [nel]
};

// Readout networks of one hidden layer and up to 16 inputs (every GRACE-1L and 2L readout this repository configures): 16 lanes per
// atom, lane p takes the hidden units p, p + 16, ... with all inputs of its atom in registers, so that no lane of the group reads
// what another one wrote.  k_energy and the first k_energy_2l give a wave to an atom, exchange every layer through LDS and are
// bound by that chain of round trips: 22.6 us for 128 atoms, 28 for 8192, 128 for 65 536 (GRACE-1L), 81 for 32 000 (GRACE-2L).
// Here 7.4, 10, 43 and 38 us.
constexpr int kReadoutInputs = 16;
constexpr int kReadoutLds = 4096;            // doubles of weights that a block stages: hidden widths up to 240
constexpr unsigned kReadoutBlocks = 1024;    // blocks of 16 atoms; a block of a larger pass walks on and keeps its weights
inline bool readout_fits(int nlay, int nin, int nhid, int nout)
{
  return nlay == 2 && nin >= 1 && nin <= kReadoutInputs && nout == 1 && nhid <= kReadoutLds / (kReadoutInputs + 1);
}
inline size_t readout_lds(int nhid) { return (size_t) (kReadoutInputs + 1) * nhid * sizeof(double); }
inline unsigned readout_blocks(int natoms) { return std::min((unsigned) (natoms + 15) / 16, kReadoutBlocks); }

// weights of the two layers -> LDS: [16][nhid] (rows beyond the inputs are zero), then the nhid weights of the output
__device__ inline void readout_stage(double *lds, const double *W0, const double *W1, int nin, int nhid)
{
  for (int e = threadIdx.x; e < (kReadoutInputs + 1) * nhid; e += blockDim.x)
    lds[e] = e < nin * nhid ? W0[e] : e < kReadoutInputs * nhid ? 0.0 : W1[e - kReadoutInputs * nhid];
  __syncthreads();
}
// sum over the 16 lanes of an atom
__device__ inline double readout_sum(double v)
{
  for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
  return v;
}
// Output of the network for the input x of lane p (the inputs of lanes beyond the network's are zero), and, with want_grad, gscale
// times its derivative by that input.  All 64 lanes of the wave arrive here.
__device__ inline double readout_net(const double *lds, int nhid, double norm0, double norm1, int act, double x, int p, int want_grad, double gscale,
                                     double &grad)
{
  double xs[kReadoutInputs], g[kReadoutInputs];
#pragma unroll
  for (int a = 0; a < kReadoutInputs; a++) { xs[a] = __shfl(x, a, 16); g[a] = 0.0; }
  const double *w1 = lds + kReadoutInputs * nhid;
  double e = 0.0;
  for (int j = p; j < nhid; j += 16) {
    double w[kReadoutInputs], s = 0.0;
#pragma unroll
    for (int a = 0; a < kReadoutInputs; a++) { w[a] = lds[a * nhid + j]; s += xs[a] * w[a]; }
    s *= norm0;
    double v, dv;
    if (act == 1) {
      v = tanh(s);
      dv = 1.0 - v * v;
    } else {
      const double d = 1.0 + exp(-s), sg = 1.0 / d;
      v = s / d;
      dv = sg * (1.0 + s * (1.0 - sg));
    }
    e += v * w1[j];
    const double t = gscale * w1[j] * norm1 * dv * norm0;
#pragma unroll
    for (int a = 0; a < kReadoutInputs; a++) g[a] += t * w[a];
  }
  e = readout_sum(e) * norm1;
  if (want_grad) {
    // every step halves the inputs that a lane still adds up: lane p is left with input p
#pragma unroll
    for (int o = 8; o > 0; o >>= 1)
#pragma unroll
      for (int a = 0; a < o; a++) {
        const double mine = p & o ? g[a + o] : g[a], other = p & o ? g[a] : g[a + o];
        g[a] = mine + __shfl_xor(other, o, 16);
      }
    grad = g[0];
  }
  return e;
}
// the legacy layer norm in front of the network (fused_cpu.h:666-682): x q, q = 1 / sqrt(mean x^2 + 1e-16), and the reverse
__device__ inline double readout_ln(double x, int nin) { return 1.0 / sqrt(readout_sum(x * x) / nin + 1e-16); }
__device__ inline double readout_ln_bwd(double g, double x, double q, int nin) { return q * (g - x * readout_sum(g * x) * q * q / nin); }
// energies of the atoms of a block without structure records: one addition per block
__device__ inline void readout_add(double esum, double *energy)
{
  __shared__ double eblk[4];
  esum += __shfl_xor(esum, 16, 64);
  esum += __shfl_xor(esum, 32, 64);
  if ((threadIdx.x & 63) == 0) eblk[threadIdx.x >> 6] = esum;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(energy + record_of(nullptr, blockIdx.x), eblk[0] + eblk[1] + eblk[2] + eblk[3]);
}

// as k_energy below
static __global__ __launch_bounds__(256) void k_energy_hidden(EnergyDev M, const int *__restrict__ mu, int a0, int natoms, const double *__restrict__ rho,
                                                              double *__restrict__ grho, double *eatom_chunk, double *energy, int want_grad,
                                                              const int *sid)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *lds = reinterpret_cast<double *>(smem_raw);
  const int p = threadIdx.x & 15, nin = M.nrho - 1;
  readout_stage(lds, M.W[0], M.W[1], nin, M.nout[0]);
  double esum = 0.0;
  for (int b0 = blockIdx.x * 16; b0 < natoms; b0 += gridDim.x * 16) {    // uniform over the block
    const int at = b0 + (threadIdx.x >> 4);
    const bool ok = at < natoms;
    const double *r = rho + (long long) (ok ? at : 0) * M.nrho;
    const double x0 = p < nin ? r[p + 1] : 0.0;
    const double q = M.ln ? readout_ln(x0, nin) : 1.0;
    double g;
    const double e = readout_net(lds, M.nout[0], M.norm[0], M.norm[1], M.act, x0 * q, p, want_grad, M.out_scale, g);
    if (want_grad && M.ln) g = readout_ln_bwd(g, x0, q, nin);
    if (!ok) continue;    // no exchange between lanes below
    if (p == 0) {
      const double Ei = (e + r[0]) * M.out_scale + M.shift[mu[a0 + at]];
      if (eatom_chunk) eatom_chunk[at] = Ei;
      if (!energy) {}    // ordered mode: the records are summed from the per-atom energies afterwards
      else if (sid) atomicAdd(energy + record_of(sid, a0 + at), Ei);
      else esum += Ei;
    }
    if (!want_grad) continue;
    double *gr = grho + (long long) at * M.nrho;
    if (p == 0) gr[0] = M.out_scale;
    if (p < nin) gr[p + 1] = g;
  }
  if (!sid && energy) readout_add(esum, energy);
}

constexpr int kEnergyAtomsPerBlock = 16;    // atoms of one block of k_energy (4 waves, 4 atoms each)

// E_i = (MLP(rho[1:]) + rho[0]) out_scale + shift[mu_i] and dE/drho, fp64, one wave per atom (fused_1l.cpp:378-427;
// legacy RMS layer norm fused_cpu.h:666-682).  A block of 4 waves shares the staged weights and walks
// kEnergyAtomsPerBlock atoms; WLDS: the weights of the network sit in LDS (as stored and transposed), else they are
// read from global memory.  A layer with fewer than 33 outputs splits each dot product over 64 / outputs lanes (the
// last layer's single output: all 64).  Without structure records the block adds its energies to the total with one
// atomic.  dynamic LDS: M.wlds + 4 x (2 nlay + 4) x width doubles.
template<bool WLDS>
static __global__ __launch_bounds__(256) void k_energy(EnergyDev M, const int *mu, int a0, int natoms, const double *rho, double *grho,
                                                         double *eatom_chunk, double *energy, int want_grad, const int *sid)
{
  // LDS rows of W = M.width values per wave: nlay + 1 activations, nlay pre-activations, 2 adjoint buffers, x0
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int W = M.width;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double *wl0 = reinterpret_cast<double *>(smem_raw);
  double *act_ = wl0 + (WLDS ? M.wlds : 0) + wave * (2 * M.nlay + 4) * W, *pre_ = act_ + (M.nlay + 1) * W, *gbuf_ = pre_ + M.nlay * W,
         *x0 = gbuf_ + 2 * W;
#define act(L_, k_) act_[(L_) * W + (k_)]
#define pre(L_, k_) pre_[(L_) * W + (k_)]
#define gbuf(L_, k_) gbuf_[(L_) * W + (k_)]
  // the rows of a wave are its own: a wave-level barrier orders its LDS writes before the reads of its other lanes
#define GR_WAVE_SYNC()                                        \
  do {                                                        \
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");    \
    __builtin_amdgcn_wave_barrier();                          \
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");    \
  } while (0)
  // as stored [a][c] for the forward pass and transposed [c][a] for the reverse: one round of coalesced loads per block
  // instead of a dependent chain of them per layer and atom
  const double *wf[7], *wt[7];
  {
    double *wl = wl0;
    for (int L = 0; L < M.nlay; L++) {
      const int sz = M.nin[L] * M.nout[L];
      if (WLDS) {
        for (int e = threadIdx.x; e < sz; e += 256) {
          const double v = M.W[L][e];
          wl[e] = v;
          wl[sz + (e % M.nout[L]) * M.nin[L] + e / M.nout[L]] = v;
        }
        wf[L] = wl;
        wt[L] = wl + sz;
        wl += 2 * sz;
      } else {
        wf[L] = M.W[L];
        wt[L] = nullptr;
      }
    }
  }
  __syncthreads();
  const int n0 = M.nrho - 1;
  // lanes that share one output of a layer: the largest power of two g with outputs x g <= 64
  auto group = [](int nout_) {
    int g = 1;
    while (g < 64 && nout_ * (g * 2) <= 64) g *= 2;
    return g;
  };
  double esum = 0.0;                                // lane 0: energies of this wave's atoms (no structure records)
  for (int k4 = 0; k4 < kEnergyAtomsPerBlock / 4; k4++) {
    const int at = blockIdx.x * kEnergyAtomsPerBlock + k4 * 4 + wave;
    if (at >= natoms) break;                        // uniform over the wave; no block barrier inside the loop
    const double *r = rho + (long long) at * M.nrho;
    GR_WAVE_SYNC();                                 // the rows of the previous atom are no longer read
    for (int k = lane; k < n0; k += 64) act(0, k) = r[k + 1];
    GR_WAVE_SYNC();
    double q = 0.0;
    if (M.ln) {
      double ms = 0.0;
      for (int k = lane; k < n0; k += 64) { x0[k] = act(0, k); ms += act(0, k) * act(0, k); }
      for (int o = 32; o > 0; o >>= 1) ms += __shfl_xor(ms, o, 64);
      q = 1.0 / sqrt(ms / n0 + 1e-16);
      for (int k = lane; k < n0; k += 64) act(0, k) *= q;
      GR_WAVE_SYNC();
    }
    for (int L = 0; L < M.nlay; L++) {
      const int no = M.nout[L], ni = M.nin[L], g = group(no), p = lane % g;
      for (int c0 = 0; c0 < no; c0 += 64 / g) {     // every lane walks the loop: the exchanges below need the whole wave
        const int c = c0 + lane / g;
        double s = 0.0;
        if (c < no) {
#pragma unroll 4
          for (int a = p; a < ni; a += g) s += act(L, a) * wf[L][a * no + c];
        }
        for (int o = g >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (c < no && p == 0) {
          s *= M.norm[L];
          pre(L, c) = s;
          act(L + 1, c) = (L < M.nlay - 1) ? (M.act == 1 ? tanh(s) : s / (1.0 + exp(-s))) : s;
        }
      }
      GR_WAVE_SYNC();
    }
    const double Ei = (act(M.nlay, 0) + r[0]) * M.out_scale + M.shift[mu[a0 + at]];
    if (lane == 0) {
      if (eatom_chunk) eatom_chunk[at] = Ei;
      if (!energy) {}    // ordered mode: the records are summed from the per-atom energies afterwards
      else if (sid) atomicAdd(energy + record_of(sid, a0 + at), Ei);
      else esum += Ei;
    }
    if (!want_grad) continue;
    int cur = 0;
    if (lane == 0) gbuf(0, 0) = M.out_scale;
    GR_WAVE_SYNC();
    for (int L = M.nlay - 1; L >= 0; L--) {
      if (L < M.nlay - 1) {
        for (int c = lane; c < M.nout[L]; c += 64) {
          const double v = pre(L, c);
          if (M.act == 1) {
            const double t = act(L + 1, c);
            gbuf(cur, c) *= 1.0 - t * t;
          } else {
            const double sg = 1.0 / (1.0 + exp(-v));
            gbuf(cur, c) *= sg * (1.0 + v * (1.0 - sg));
          }
        }
        GR_WAVE_SYNC();
      }
      {
        const int no = M.nout[L], ni = M.nin[L], g = group(ni), p = lane % g;
        for (int b0 = 0; b0 < ni; b0 += 64 / g) {
          const int a = b0 + lane / g;
          double s = 0.0;
          if (a < ni) {
            if (WLDS) {
#pragma unroll 4
              for (int c = p; c < no; c += g) s += gbuf(cur, c) * wt[L][c * ni + a];
            } else {
#pragma unroll 4
              for (int c = p; c < no; c += g) s += gbuf(cur, c) * wf[L][(long long) a * no + c];
            }
          }
          for (int o = g >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
          if (a < ni && p == 0) gbuf(cur ^ 1, a) = s * M.norm[L];
        }
      }
      cur ^= 1;
      GR_WAVE_SYNC();
    }
    if (M.ln) {
      double t = 0.0;
      for (int k = lane; k < n0; k += 64) t += gbuf(cur, k) * x0[k];
      for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
      for (int k = lane; k < n0; k += 64) gbuf(cur, k) = q * (gbuf(cur, k) - x0[k] * t * q * q / n0);
      GR_WAVE_SYNC();
    }
    double *g = grho + (long long) at * M.nrho;
    if (lane == 0) g[0] = M.out_scale;
    for (int k = lane; k < n0; k += 64) g[k + 1] = gbuf(cur, k);
  }
  if (!sid && energy) {    // one atomic per block (every wave leaves the loop above and arrives here)
    __shared__ double eblk[4];
    if (lane == 0) eblk[wave] = esum;
    __syncthreads();
    if (threadIdx.x == 0) {
      const double e = eblk[0] + eblk[1] + eblk[2] + eblk[3];
      if (e != 0.0) atomicAdd(energy + record_of(nullptr, blockIdx.x), e);
    }
  }
#undef GR_WAVE_SYNC
#undef act
#undef pre
#undef gbuf
}

// ---------------------------------------------------------------------------------------------------------------
// UQ head (uqv6, gamma only)
// ---------------------------------------------------------------------------------------------------------------
constexpr int kUqMaxSrc = 8, kUqMaxBlk = 3;
template<class T> struct UqDev {
  const T *X[kUqMaxSrc];      // per-atom tensors of the reduces' sources [atom][function][channel]
  const int *ci[kUqMaxSrc];   // collected functions of each source
  int nfun[kUqMaxSrc], cpad[kUqMaxSrc], nin[kUqMaxSrc], nc[kUqMaxSrc], off[kUqMaxSrc];    // functions per atom, padded / real channels, collected, first basis index
  int blk[kUqMaxSrc];         // invariant block of the source (1L: rho = 0; 2L: I2 = 0, rho = 1; 3L: layer)
  int nsrc, nblk, rp, D, K;
  int row0, d_basis;          // this launch holds rows row0 .. row0 + d_basis of the basis (off[] counts from row0)
  int carry_in, carry_out;    // 3L, one launch per layer: add the projection and block norms kept by the earlier layers / keep them and stop
  double *zacc, *n2acc;       // [atom][rp], [atom][kUqMaxBlk]: the kept raw projection and squared block norms
  double density_scale;
  const double *R;            // [d_basis][rp]
  const double *cen;          // [nel][K][D]
  const double *icov;         // [nel][K][D][D]
  const int *ncl;             // [nel]
  const double *thr;          // [nel][K]
};

// gamma, sigma, cluster of one atom per block (libgrace/include/grace/fused_cpu.h:1290-1312 basis, :1375-1412 GMM;
// libgrace/src/fused_1l.cpp:616-636, fused_2l.cpp:1156-1186): basis B = per invariant block the collected functions of
// the reduce's sources, n-outer and c-inner per source; phi = ((B / |B|) R, log |B| scale, log |B_block| scale ...);
// nearest centroid of the atom's element, Mahalanobis distance over the cluster's threshold.  fp64 throughout.
// GRACE-3L (libgrace/src/fused_3l.cpp:1156-1201) evaluates the rows of one layer per launch, right after that layer's
// rho reduce while its tensors exist: raw projection and squared block norms are carried in zacc / n2acc.
// block: 256 threads; dynamic LDS: d_basis + 4 rp + 2 D doubles.
template<class T>
__global__ __launch_bounds__(256) void k_uq(UqDev<T> U, const int *mu, int natoms, double *gamma, double *sigma, double *cluster)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *Bsh = reinterpret_cast<double *>(smem_raw);       // [d_basis]
  double *Zp = Bsh + U.d_basis;                             // [4][rp] partial projections
  double *f = Zp + 4 * U.rp;                                // [D]
  double *dl = f + U.D;                                     // [D]
  __shared__ double wsum[4], bsum[4][kUqMaxBlk];
  __shared__ int kstar;
  const int at = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (at >= natoms) return;
  // ---- basis and the norms of its blocks
  double n2[kUqMaxBlk];
#pragma unroll
  for (int b = 0; b < kUqMaxBlk; b++) n2[b] = 0.0;
  for (int s = 0; s < U.nsrc; s++) {
    const T *x = U.X[s] + (long long) at * U.nfun[s] * U.cpad[s];
    const int w = U.nin[s] * U.nc[s];
    double acc = 0.0;
    for (int r = t; r < w; r += 256) {
      const int n = r / U.nc[s], c = r % U.nc[s];
      const double v = (double) x[U.ci[s][c] * U.cpad[s] + n];
      Bsh[U.off[s] + r] = v;
      acc += v * v;
    }
#pragma unroll
    for (int b = 0; b < kUqMaxBlk; b++)
      if (U.blk[s] == b) n2[b] += acc;
  }
#pragma unroll
  for (int b = 0; b < kUqMaxBlk; b++) {
    for (int o = 32; o > 0; o >>= 1) n2[b] += __shfl_xor(n2[b], o, 64);
    if (lane == 0) bsum[wave][b] = n2[b];
  }
  __syncthreads();
  double nb2[kUqMaxBlk], tot = 0.0;
#pragma unroll
  for (int b = 0; b < kUqMaxBlk; b++) {
    nb2[b] = bsum[0][b] + bsum[1][b] + bsum[2][b] + bsum[3][b];
    if (U.carry_in) nb2[b] += U.n2acc[(long long) at * kUqMaxBlk + b];
    tot += nb2[b];
  }
  const double nrm = sqrt(tot);
  // ---- projection Z = B R: column d = t mod rp, rows split over the 256 / rp (at most 4 used) thread groups
  {
    const int ng = 256 / U.rp > 4 ? 4 : 256 / U.rp, gq = t / U.rp, d = t % U.rp;
    if (gq < ng) {
      double z = 0.0;
      for (int b = gq; b < U.d_basis; b += ng) z += Bsh[b] * U.R[(long long) (U.row0 + b) * U.rp + d];
      Zp[gq * U.rp + d] = z;
    }
    __syncthreads();
    if (t < U.D) {
      if (t < U.rp) {
        double z = 0.0;
        for (int q = 0; q < ng; q++) z += Zp[q * U.rp + t];
        if (U.carry_in) z += U.zacc[(long long) at * U.rp + t];
        if (U.carry_out) U.zacc[(long long) at * U.rp + t] = z;
        f[t] = z / (nrm + 1.0e-12);
      } else {    // density channels: the whole basis, then its blocks (one block: the same norm again)
        const int p = t - U.rp;
        double dn = nrm;
#pragma unroll
        for (int b = 0; b < kUqMaxBlk; b++)
          if (p == 1 + b) dn = sqrt(nb2[b]);
        f[t] = log(dn + 1.0e-12) * U.density_scale;
      }
    }
    if (U.carry_out) {    // the same for every thread of the block
#pragma unroll
      for (int b = 0; b < kUqMaxBlk; b++)
        if (t == b) U.n2acc[(long long) at * kUqMaxBlk + b] = nb2[b];
      return;
    }
    __syncthreads();
  }
  // ---- nearest centroid of the element (the first of equal distances)
  const int m = mu[at];
  if (t == 0) {
    int kb = 0;
    double best = 1.0e300;
    for (int q = 0; q < U.ncl[m]; q++) {
      const double *c = U.cen + ((long long) m * U.K + q) * U.D;
      double d2 = 0.0;
      for (int p = 0; p < U.D; p++) d2 += (f[p] - c[p]) * (f[p] - c[p]);
      if (d2 < best) { best = d2; kb = q; }
    }
    kstar = kb;
  }
  __syncthreads();
  const int kq = kstar;
  for (int p = t; p < U.D; p += 256) dl[p] = f[p] - U.cen[((long long) m * U.K + kq) * U.D + p];
  __syncthreads();
  // ---- sigma^2 = delta^T S delta
  const double *S = U.icov + ((long long) m * U.K + kq) * U.D * U.D;
  double part = 0.0;
  for (int p = t; p < U.D; p += 256) {
    double y = 0.0;
    for (int q = 0; q < U.D; q++) y += S[(long long) p * U.D + q] * dl[q];
    part += dl[p] * y;
  }
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  __syncthreads();
  if (lane == 0) wsum[wave] = part;
  __syncthreads();
  if (t == 0) {
    const double sg = sqrt(wsum[0] + wsum[1] + wsum[2] + wsum[3] + 1.0e-8);
    const double th = U.thr[(long long) m * U.K + kq];
    sigma[at] = sg;
    gamma[at] = sg / (th > 1.0e-10 ? th : 1.0e-10);
    cluster[at] = (double) kq;
  }
}

// Two unit vectors that span the plane normal to the unit vector u: e1 = a x u / |a x u| with a the coordinate axis on
// which u has its smallest component, e2 = u x e1.  A pure function of u: the kernel that stores tangential gradients
// and the kernel that turns their adjoints into a force compute the same pair.
__device__ inline void tangent_basis(const double *u, double *e1, double *e2)
{
  const double ax = fabs(u[0]), ay = fabs(u[1]), az = fabs(u[2]);
  double a[3] = {0.0, 0.0, 0.0};
  if (ax <= ay && ax <= az) a[0] = 1.0;
  else if (ay <= az) a[1] = 1.0;
  else a[2] = 1.0;
  const double c0 = a[1] * u[2] - a[2] * u[1], c1 = a[2] * u[0] - a[0] * u[2], c2 = a[0] * u[1] - a[1] * u[0];
  const double inv = 1.0 / sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  e1[0] = c0 * inv; e1[1] = c1 * inv; e1[2] = c2 * inv;
  e2[0] = u[1] * e1[2] - u[2] * e1[1]; e2[1] = u[2] * e1[0] - u[0] * e1[2]; e2[2] = u[0] * e1[1] - u[1] * e1[0];
}

// ---------------------------------------------------------------------------------------------------------------
// bond backward: forces and virial
// ---------------------------------------------------------------------------------------------------------------
template<class T> struct BondBwdArgs {
  const long long *eoff;
  const int *ej;
  const double *rh, *r, *rc;
  const T *Rz, *dRz;          // [E][noutp]
  const int *erow, *emu;      // RowsOf::pairs: as ScatterArgs
  const T *z;
  RadialTable<T> tb;          // tb.F set: value and derivative of the radial functions come from the tables, Rz / dRz are not read
  const T *gA;                // [chunk atoms][nlm][C]
  double *f;                  // [n][3]  (+=, atomics)
  double *virial;             // [6]     (+=, atomics) of the record that the atom uses (record_of)
  const int *sid;             // [n] structure of each atom, or null
  double *vatom;              // [n][9] per-atom virial xx yy zz xy xz yz yx zx zy (+=, atomics), or null: half of a bond's (-r rhat) (x) fv to each of its atoms
  // ordered mode (both set, no atomics, vatom null): fedge[e][3] = force of bond e on its central atom; fcen[i][9] = sum of
  // these over the bonds of atom i, then the six virial sums of its bonds; k_ordered_forces / k_ordered_records finish
  double *fedge, *fcen;
  // sums of a bond left by the reverse pair kernels of the layers above ([e][3]: against Y dR, D1 R and D2 R as px, p1, p2 here),
  // or null: their part of the bond's force is finished with this layer's, in one addition to each of its atoms
  const double *bsum;
  int ordered_add;            // ordered mode: add to what fedge / fcen hold (a later layer of the same pass) instead of storing
  int a0;
  int C, nl, nlm, noutp;
  int tiles;                  // tiles of 16 bonds of a round (bond_bwd_tiles)
  int drow[16];               // accumulator row of (lane / 16, register)
  ShCoef sh;
};

// Waves per SIMD that k_bond_bwd is compiled for.  In fp32 it waits for its chain of loads, not for HBM or the atomics (without
// them it is no faster), and left alone it takes 173 registers where 168 let a third wave in: tables, 65 536 atoms 1.85 -> 1.39 ms,
// 3999 of GRACE-2L 183 -> 147 us; paired rows, 20 000 atoms 571 -> 536 us.  A fourth wave spills 42 registers (2.03 ms).  Rows of
// their own serve small structures, which have one block per CU anyway (500 atoms 20.4 -> 21.9 us); from lmax 5 on, with 64
// channels and in fp64 three waves spill.  Of the forms compiled for three waves one spills, tables at 32 channels and lmax 4 (two
// registers): the unit vector of a bond is read again behind its tiles and the addresses of a row's harmonics are formed where
// they are used, 32 768 atoms 725 -> 665 us, 3999 atoms of 78 bonds 153 -> 142, paired rows, 8192 atoms 178 -> 163 (21 and 16 spilled).
template<class T> constexpr int bond_bwd_waves(int kb, int nl, RowsOf rows) { return sizeof(T) == 4 && kb <= 2 && nl <= 5 && rows != RowsOf::bonds ? 3 : 1; }

// Tiles of 16 bonds whose harmonics a wave evaluates at once, a bond per lane, and waves of a block.  One tile at a time leaves 48
// lanes idle in the harmonics, half of the vector instructions of a tile in fp32.  Two tiles: paired rows, 8192 atoms fp32 198 -> 178 us,
// tables, 3999 atoms of 78 bonds 156 -> 153; in fp64, where the harmonics of two tiles leave LDS for six waves of a CU, 203 -> 225 us
// (tables, 4001 atoms), 21 -> 25 (128 atoms).  Up to two atoms per CU (few) four waves of one tile each are quicker than two of two,
// one tile / two, 58 bonds, us: lmax 4, 32 channels, 128 atoms 17.4 / 20.0, 432 21.0 / 22.5, 686 32.3 / 24.5; lmax 6 20.5 / 24.7, 26.2 /
// 30.5, 39.8 / 33.4; with tables 19.6 / 21.9, 23.4 / 25.4, 27.4 / 28.9.
template<class T> constexpr int bond_bwd_tiles(bool few) { return sizeof(T) == 4 && !few ? 2 : 1; }
// Values of a bond in LDS, its harmonics and their two gradient components: odd, so that the 16 bonds of a tile, which are read at
// once, start in different banks.  As 3 nlm values, which is even from lmax 1 on for every second lmax and 48 at lmax 3: 3456 atoms of 58
// bonds, lmax 3 fp64, paired rows of 16 channels 97.7 -> 70.0 us, of 32 113.6 -> 92.2, of 64 223.5 -> 204.4.
constexpr int bond_bwd_row(int nlm) { return 3 * nlm | 1; }

// One block per atom; a wave takes rounds of HT tiles of 16 bonds.  Per tile and l two tile GEMMs on the matrix cores,
//   P[m][b] = sum_n gA[l*l + m][n] Rz[b][l][n],   Q[m][b] = sum_n gA[l*l + m][n] dRz[b][l][n]      (K = channels)
// with the bonds as columns: lane (g, c) of the wave ends up with the rows m = drow[4 g + v] of bond c, so the sums over
// m are four terms in the lane and two exchanges between the lane groups, and lane c < 16 -- the lane that evaluated
// the harmonics of bond c and holds its geometry in registers -- finishes the bond:
//   g_d = sum_lm G[b][lm][d] P[lm][b],  dE/dx = sum_lm Y[b][lm] Q[lm][b],
//   fv = dE/dx / rc rhat + (g - (g . rhat) rhat) / r;  f_i += fv, f_j -= fv, virial += (-r rhat) (x) fv
// (fused_cpu.h:836-860,1027-1050; fused_1l.cpp:46-51 of the reference).  Only the part of g normal to the bond enters,
// g - (g . rhat) rhat = (g . e1) e1 + (g . e2) e2 for an orthonormal pair e1, e2 normal to the bond (tangent_basis), so
// the harmonics' gradients are kept as their two components along e1 and e2: two sums per bond instead of three, and a
// third less LDS per block (three blocks per CU instead of two).  gA of the atom sits in LDS as [lm][C + 2]
// (the pad spreads the rows over the banks); the radial rows of l + 1 are requested before the products of l.
// KB = channels / 16, NL = lmax + 1.  dynamic LDS: nlm (C + 2) + 4 tiles x 16 bonds x bond_bwd_row(nlm) values.
// l = 0 has no gradient: its radial function is neither read nor evaluated, its derivative is (a tenth of the rows at lmax 4).  With
// that, the harmonics of a bond in one row and fewer address instructions: paired rows, 8192 atoms fp64 280 -> 254 us, fp32 226 ->
// 198; tables, 3999 atoms fp32 166 -> 156, 4001 atoms fp64 211 -> 204, and the tiles two at a time above.
// RowsOf::tables: the B operands are formed from the radial tables (lane (g, c): the eight columns l C + 8 g + s of bond c, four table
// entries each, value and derivative from the same four; requested for l + 1 before the products of l).
template<class T, int KB, int NL, RowsOf ROWS> __global__ __launch_bounds__(256, bond_bwd_waves<T>(KB, NL, ROWS)) void k_bond_bwd(BondBwdArgs<T> a)
{
  const int HT = sizeof(T) == 4 ? a.tiles : 1, NW = 4 / HT;
  constexpr bool TAB = ROWS == RowsOf::tables, PAIRS = ROWS == RowsOf::pairs;
  typedef typename Mfma<T>::v4 v4;
  constexpr int KS = KB * 4, C = KB * 16, CS = C + 2, NLM = NL * NL, HS = bond_bwd_row(NLM);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *gAl = reinterpret_cast<T *>(smem_raw);                          // [NLM][CS]
  T *Hsh = gAl + NLM * CS;                                           // [NW waves][16 HT][HS]: harmonics, gradient . e1, gradient . e2
  __shared__ double red[4][9];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int i = a.a0 + blockIdx.x;
  const long long e0 = a.eoff[i], e1_ = a.eoff[i + 1];
  {
    const T *gAi = a.gA + (long long) blockIdx.x * NLM * C;
    for (int q = t; q < NLM * C; q += 64 * NW) gAl[(q / C) * CS + q % C] = gAi[q];
  }
  __syncthreads();
  T *Hw = Hsh + wave * HT * 16 * HS;
  int mrow[4];
  const T *hrow0 = Hw + c * HS;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    mrow[v] = a.drow[4 * g + v];
  }
  double fi[3] = {0, 0, 0}, vir[6] = {0, 0, 0, 0, 0, 0};
  const int ntile = (int) ((e1_ - e0 + 15) / 16);
  for (int round = wave; round * HT < ntile; round += NW) {
    const long long er = e0 + (long long) round * HT * 16;
    const int nr = (int) (e1_ - er < 16 * HT ? e1_ - er : 16 * HT);      // bonds of the round
    // rows read by this lane: without tables step s of lane group g is channel 8 (s / 2) + 2 g + s % 2 (CH), so that the
    // four lane groups read 64 consecutive bytes of a bond's row in one instruction; with tables channel g KS + s
#define CH(s_) (TAB ? (s_) : 8 * ((s_) >> 1) + ((s_) & 1))
    const T *rp = nullptr, *dp = nullptr;
    T x[2][KS], dx[2][KS];
    // tables: interval, offset and species weights of bond c, and the entries of l = 0
    // (four columns at a time: the entries of the next four are requested before the products of these four)
    constexpr int KH = 4;
    T raw[4][TAB ? KH : 1], zc[TAB || PAIRS ? KS : 1];
    TableBond<T> tt{};
    TableRow<T> trow{};
    // four columns from column `col` of the lane's eight on
    auto request = [&](int col) {
      constexpr int V = 16 / (int) sizeof(T);
      typedef T piece __attribute__((ext_vector_type(16 / sizeof(T))));
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int q = 0; q < KH / V; q++) {
          const piece w = *reinterpret_cast<const piece *>(table_entry<NL * C>(trow, e) + col + q * V);
#pragma unroll
          for (int s = 0; s < V; s++) raw[e][q * V + s] = w[s];
        }
    };
    // the first rows (table entries) of the tile from bond eb on: of l = 0, whose gradient is zero, the derivative alone
    auto begin = [&](long long eb) {
      const long long e = eb + (eb + c < e1_ ? c : 0);
      if constexpr (TAB) {
        double t;
        const int tk = table_interval(a.tb.x[e], a.tb.N, t);
        tt = table_bond<T>(t, a.tb.N);
        trow = table_row<T, NL * C>(a.tb, tk, g * KS);
        const int mu = a.tb.emu[e];
#pragma unroll
        for (int s = 0; s < KS; s++) zc[s] = a.tb.z[mu * C + g * KS + s];
        request(0);
      } else {
        const long long row = PAIRS ? (long long) a.erow[e] : e;
        rp = a.Rz + row * a.noutp + 2 * g;
        dp = a.dRz + row * a.noutp + 2 * g;
#pragma unroll
        for (int s = 0; s < KS; s++) dx[0][s] = dp[CH(s)];
        if constexpr (PAIRS) {
          const int mu = a.emu[e];
#pragma unroll
          for (int s = 0; s < KS; s++) zc[s] = a.z[mu * C + 2 * g + CH(s)];
        }
      }
    };
    begin(er);
    // geometry of bond `lane` (lanes below nr), kept for the end of the round
    double u0 = 0, u1 = 0, u2 = 1, br = 1, brc = 1;
    double e1[3] = {1, 0, 0}, e2[3] = {0, 1, 0};
    int jj = 0;
    if (lane < nr) {
      const long long e = er + lane;
      u0 = a.rh[3 * e]; u1 = a.rh[3 * e + 1]; u2 = a.rh[3 * e + 2];
      br = a.r[e]; brc = a.rc[e]; jj = a.ej[e];
      const double u[3] = {u0, u1, u2};
      tangent_basis(u, e1, e2);
      T *h = Hw + lane * HS;
      sh_eval<true, T, NL - 1>(a.sh, u0, u1, u2, h, h + NLM, e1, e2, h + 2 * NLM);
    }
    // LDS writes of this wave visible to its other lanes (its harmonics are private to the wave)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double px_r = 0, p1_r = 0, p2_r = 0;      // of bond er + lane
    for (int ht = 0; ht < HT; ht++) {
      const long long eb = er + 16 * ht;
      if (sizeof(T) == 4 && eb >= e1_) break;
      const bool colok = eb + c < e1_;                // B operand column = bond c of the tile
      double px = 0, p1 = 0, p2 = 0;
#pragma unroll
      for (int l = 0; l < NL; l++) {
        const int cur = TAB ? 0 : (l & 1), nxt = cur ^ 1;
        if constexpr (!TAB) {
          if (l + 1 < NL) {
#pragma unroll
            for (int s = 0; s < KS; s++) { x[nxt][s] = rp[(l + 1) * C + CH(s)]; dx[nxt][s] = dp[(l + 1) * C + CH(s)]; }
          }
        }
        v4 aP = {0, 0, 0, 0}, aQ = {0, 0, 0, 0};
        // A operand: row m = c of gA_l^T, k = g KS + s
        const T *ga = gAl + (l * l + (c < 2 * l + 1 ? c : 0)) * CS + (TAB ? g * KS : 2 * g);
        if constexpr (TAB) {
#pragma unroll
          for (int hb = 0; hb < KS; hb += KH) {
            T xv[KH], dxv[KH];
#pragma unroll
            for (int s = 0; s < KH; s++) {
              const TableCubic<T> cubic = table_cubic(raw[0][s], raw[1][s], raw[2][s], raw[3][s], tt);
              xv[s] = l > 0 ? table_value(cubic, tt) * zc[hb + s] : (T) 0;
              dxv[s] = table_slope(cubic, tt) * zc[hb + s];
            }
            // the next four columns: of this l, or the first four of l + 1
            if (hb + KH < KS) request(l * C + hb + KH);
            else if (l + 1 < NL) request((l + 1) * C);
#pragma unroll
            for (int s = 0; s < KH; s++) {
              const T w = c < 2 * l + 1 ? ga[hb + s] : (T) 0;
              if (l > 0) aP = Mfma<T>::mma(w, xv[s], aP);
              aQ = Mfma<T>::mma(w, dxv[s], aQ);
            }
          }
        } else {
#pragma unroll
          for (int s = 0; s < KS; s++) {
            const T w = c < 2 * l + 1 ? ga[CH(s)] : (T) 0;
            T dxs = dx[cur][s];
            if constexpr (PAIRS) dxs *= zc[s];
            if (l > 0) {
              T xs = x[cur][s];
              if constexpr (PAIRS) xs *= zc[s];
              aP = Mfma<T>::mma(w, xs, aP);
            }
            aQ = Mfma<T>::mma(w, dxs, aQ);
          }
        }
        // rows m > 2 l hold zeros (their operand is zero) and take the harmonics of m = 0; what a column without a bond gives is not used
        if (colok)      // ends a scheduling region: without it the l of a tile run into each other and spill (740 -> 1180 us)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          int m = mrow[v];
          asm volatile("" : "+v"(m));      // or the compiler keeps (and spills) an address per l and v ahead of the tiles
          const T *h = hrow0 + (m < 2 * l + 1 ? m : 0) + ht * 16 * HS + l * l;
          px += (double) (h[0] * aQ[v]);
          if (l > 0) {
            p1 += (double) (h[NLM] * aP[v]);
            p2 += (double) (h[2 * NLM] * aP[v]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (sizeof(T) == 4 && ht + 1 < HT && eb + 16 < e1_) begin(eb + 16);
      // sum over the four lane groups (the rows m of a bond are spread over them); lane group ht keeps the sums of tile ht
      px += __shfl_xor(px, 16, 64); p1 += __shfl_xor(p1, 16, 64); p2 += __shfl_xor(p2, 16, 64);
      px += __shfl_xor(px, 32, 64); p1 += __shfl_xor(p1, 32, 64); p2 += __shfl_xor(p2, 32, 64);
      if (sizeof(T) == 8 || g == ht) { px_r = px; p1_r = p1; p2_r = p2; }
    }
    if (TAB) px_r *= (double) a.tb.N;      // the slopes are per interval
    if (lane < nr) {
      if (sizeof(T) == 4) {      // read again: held over the tiles they are 6 of the 168 registers
        int again = 0;
        asm volatile("" : "+s"(again));
        const long long e = er + lane + again;
        u0 = a.rh[3 * e]; u1 = a.rh[3 * e + 1]; u2 = a.rh[3 * e + 2];
      }
      if (a.bsum) {
        const double *b = a.bsum + 3 * (er + lane);
        px_r += b[0]; p1_r += b[1]; p2_r += b[2];
      }
      const double dEdr = px_r / brc, t1 = p1_r / br, t2 = p2_r / br;
      const double fv[3] = {dEdr * u0 + t1 * e1[0] + t2 * e2[0], dEdr * u1 + t1 * e1[1] + t2 * e2[1], dEdr * u2 + t1 * e1[2] + t2 * e2[2]};
      for (int d = 0; d < 3; d++) {
        fi[d] += fv[d];
        if (a.fedge) a.fedge[3 * (er + lane) + d] = (a.ordered_add ? a.fedge[3 * (er + lane) + d] : 0.0) + fv[d];
        else atomicAdd(&a.f[3 * (long long) jj + d], -fv[d]);
      }
      const double ddx = -u0 * br, ddy = -u1 * br, ddz = -u2 * br;
      vir[0] += ddx * fv[0]; vir[1] += ddy * fv[1]; vir[2] += ddz * fv[2];
      vir[3] += ddx * fv[1]; vir[4] += ddx * fv[2]; vir[5] += ddy * fv[2];
      if (a.vatom) {    // the neighbour's half (add_vatom, libgrace/include/grace/fused_cpu.h:1075-1087); the atom's own below
        double *vj = a.vatom + 9 * (long long) jj;
        atomicAdd(vj, 0.5 * ddx * fv[0]); atomicAdd(vj + 1, 0.5 * ddy * fv[1]); atomicAdd(vj + 2, 0.5 * ddz * fv[2]);
        atomicAdd(vj + 3, 0.5 * ddx * fv[1]); atomicAdd(vj + 4, 0.5 * ddx * fv[2]); atomicAdd(vj + 5, 0.5 * ddy * fv[2]);
        // the components below the diagonal (the centroid form, kk/grace_1l_kk_impl.h:1344-1349), for both atoms of the bond
        double *vi = a.vatom + 9 * (long long) i;
        const double yx = 0.5 * ddy * fv[0], zx = 0.5 * ddz * fv[0], zy = 0.5 * ddz * fv[1];
        atomicAdd(vj + 6, yx); atomicAdd(vj + 7, zx); atomicAdd(vj + 8, zy);
        atomicAdd(vi + 6, yx); atomicAdd(vi + 7, zx); atomicAdd(vi + 8, zy);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  double vsum[9] = {fi[0], fi[1], fi[2], vir[0], vir[1], vir[2], vir[3], vir[4], vir[5]};
#pragma unroll
  for (int k = 0; k < 9; k++)
    for (int o = 32; o > 0; o >>= 1) vsum[k] += __shfl_xor(vsum[k], o, 64);
  if (lane == 0)
    for (int k = 0; k < 9; k++) red[wave][k] = vsum[k];
  __syncthreads();
  if (t < 9) {
    double s = red[0][t];
    for (int w = 1; w < NW; w++) s += red[w][t];
    if (a.fcen) a.fcen[9 * (long long) i + t] = (a.ordered_add ? a.fcen[9 * (long long) i + t] : 0.0) + s;
    else if (e1_ > e0) {
      if (t < 3) atomicAdd(&a.f[3 * (long long) i + t], s);
      else {
        atomicAdd(&a.virial[record_of(a.sid, i) + t - 3], s);
        if (a.vatom) atomicAdd(&a.vatom[9 * (long long) i + t - 3], 0.5 * s);
      }
    }
  }
}
#undef CH

// ---------------------------------------------------------------------------------------------------------------
// ordered (atomic-free) sums of the forces, the virial and the energy: same bits on every run
// ---------------------------------------------------------------------------------------------------------------
// bonds per neighbour atom: count[ej[e]] += 1 (integer atomics: the result does not depend on their order)
static __global__ void k_tlist_count(const long long *n_edges, const int *ej, int *count)
{
  const long long e = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (e < *n_edges) atomicAdd(&count[ej[e]], 1);
}
// bond numbers by neighbour atom, in arrival order (k_tlist_sort orders every row)
static __global__ void k_tlist_fill(const long long *n_edges, const int *ej, const long long *toff, int *cursor, int *raw)
{
  const long long e = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (e < *n_edges) {
    const int j = ej[e];
    raw[toff[j] + atomicAdd(&cursor[j], 1)] = (int) e;
  }
}
// One wave per atom k (owned atoms, then ghosts): its row of bond numbers in ascending order, by counting for every
// entry the entries below it (a row is a few hundred entries at most).
static __global__ void k_tlist_sort(int n_nodes, const long long *toff, const int *raw, int *sorted)
{
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (k >= n_nodes) return;
  const long long t0 = toff[k];
  const int *row = raw + t0;
  const int len = (int) (toff[k + 1] - t0);
  for (int p = lane; p < len; p += 64) {
    const int mine = row[p];
    int rank = 0;
    for (int q = 0; q < len; q++) rank += row[q] < mine;
    sorted[t0 + rank] = mine;
  }
}
// One wave per atom k: f[k] = fcen[k] (owned atoms) - sum of fedge over the bonds that have k as their neighbour, the
// sorted row taken by the lanes in turn and the lane sums added in a fixed tree.
static __global__ void k_ordered_forces(int n_nodes, int n, const long long *toff, const int *sorted, const double *fedge, const double *fcen, double *f)
{
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (k >= n_nodes) return;
  const long long t0 = toff[k];
  const int len = (int) (toff[k + 1] - t0);
  double s[3] = {0, 0, 0};
  for (int p = lane; p < len; p += 64) {
    const double *fe = fedge + 3 * (long long) sorted[t0 + p];
    s[0] += fe[0]; s[1] += fe[1]; s[2] += fe[2];
  }
#pragma unroll
  for (int d = 0; d < 3; d++)
    for (int o = 32; o > 0; o >>= 1) s[d] += __shfl_xor(s[d], o, 64);
  if (lane < 3) f[3 * (long long) k + lane] = (k < n ? fcen[9 * (long long) k + lane] : 0.0) - s[lane];
}
// One block per structure: record (energy, virial[6]) = sums of eatom[i] and fcen[i][3 .. 9] over its atoms, which are
// the range [lower_bound(s), lower_bound(s + 1)) of the non-decreasing sid (null: one structure, all atoms); every
// thread adds its atoms in ascending order, the thread sums are added in a fixed tree.
static __global__ __launch_bounds__(256) void k_ordered_records(int n, const int *sid, const double *eatom, const double *fcen, int with_virial, double *rec)
{
  __shared__ double part[256][7];
  const int s = blockIdx.x, t = threadIdx.x;
  int lo = 0, hi = n;
  if (sid) {
    auto lower = [&](int key) {
      int a = 0, b = n;
      while (a < b) {
        const int m = (a + b) >> 1;
        if (sid[m] < key) a = m + 1;
        else b = m;
      }
      return a;
    };
    lo = lower(s);
    hi = lower(s + 1);
  }
  double v[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int i = lo + t; i < hi; i += 256) {
    v[0] += eatom[i];
    if (with_virial)
      for (int k = 0; k < 6; k++) v[1 + k] += fcen[9 * (long long) i + 3 + k];
  }
  for (int k = 0; k < 7; k++) part[t][k] = v[k];
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o)
      for (int k = 0; k < 7; k++) part[t][k] += part[t + o][k];
    __syncthreads();
  }
  if (t < 7) rec[8 * (long long) s + t] = part[0][t];
}

}    // namespace grhip
