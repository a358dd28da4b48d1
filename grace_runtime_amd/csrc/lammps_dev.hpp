// The LAMMPS pair-style call with every per-atom array in device memory (the RunInput of the reference's GPU engines,
// libgrace/include/grace/kk/grace_1l_kk.h:80-103: x, f, type, ilist, numneigh and the 2-d neighbour view of a KOKKOS
// pair style).  The full neighbour list is turned into the engine's CSR list with bond vectors by two kernels (count,
// fill) without leaving the device; the owner map stands in for the exchange of the reference on one rank, with an
// exchange installed the ghosts stay atoms of their own.
#pragma once

#include "engine_common.hpp"

namespace grhip {

struct LmpListDev {
  const int *type;         // [nall] 1-based atom types
  const double *x;         // [nall][3]
  const int *numneigh;     // [nlocal], by atom
  const int *neighbors;    // element (i, k) at i stride_i + k stride_k
  long long stride_i, stride_k;
  const int *owner;        // [nall] owned atom of every ghost, or null
  const int *idx;          // [nlocal] engine row of an owned atom of a mapped type, else -1
  const int *atom;         // [n] owned atom of engine row q
  const unsigned char *mapped;    // [ntypes + 1] type has a model element
  int n, nlocal, nall, neighmask;
  int nodes;               // 1: ghosts are atoms of their own (an exchange moves their rows): a neighbour keeps its index
};

// FILL = false: count[q] = bonds of row q to atoms of mapped types; *err = 1: neighbour index outside the atoms,
// 2: a ghost without a usable owner.  FILL = true: j and rij of those bonds from offset[q] on, in list order, and named[] = the
// atom that the list names (an owned atom or a ghost).
// One wave per row, a lane per entry of the list: a thread that walked its row alone waited for one entry after the other
// (4001 atoms of 80 entries: 135 us for either form; now 6 and 7 us).
template<bool FILL>
__global__ __launch_bounds__(256) void k_lmp_rows(LmpListDev L, int *count, int *err, const long long *offset, int *j, double *rij, int *named)
{
  const int lane = threadIdx.x & 63;
  const int q = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= L.n) return;
  const int i = L.atom[q];
  const double xi0 = L.x[3 * (long long) i], xi1 = L.x[3 * (long long) i + 1], xi2 = L.x[3 * (long long) i + 2];
  const int nn = L.numneigh[i];
  const int *row = L.neighbors + i * L.stride_i;
  long long w = FILL ? offset[q] : 0;
  for (int k0 = 0; k0 < nn; k0 += 64) {
    const int k = k0 + lane;
    bool bond = false;
    int a = 0, o = 0;
    if (k < nn) {
      a = row[k * L.stride_k] & L.neighmask;
      o = a;
      if (a < 0 || a >= L.nall) {
        if (!FILL) *err = 1;
      } else if (L.mapped[L.type[a]]) {
        bond = true;
        if (!L.nodes) {
          if (a >= L.nlocal) o = L.owner ? L.owner[a] : -1;
          if (o < 0 || o >= L.nlocal || L.idx[o] < 0 || L.type[o] != L.type[a]) {
            if (!FILL) *err = 2;
            bond = false;
          } else {
            o = L.idx[o];
          }
        }
      }
    }
    const unsigned long long m = __ballot(bond);
    if (FILL && bond) {
      const long long p = w + __popcll(m & ((1ull << lane) - 1ull));
      j[p] = o;
      named[p] = a;
      rij[3 * p] = L.x[3 * (long long) a] - xi0;
      rij[3 * p + 1] = L.x[3 * (long long) a + 1] - xi1;
      rij[3 * p + 2] = L.x[3 * (long long) a + 2] - xi2;
    }
    w += __popcll(m);
  }
  if (!FILL && lane == 0) count[q] = (int) w;
}

// The bond vectors of a kept list from new positions: one wave per row, a lane per bond.  The rows of the 2-d view, the types
// and the owners do not change between two reneighbourings and are not read again (4001 atoms, 312 000 bonds: 135 us as the
// second pass of the conversion, now 5.6 us).
static __global__ __launch_bounds__(256) void k_lmp_vectors(const int *__restrict__ atom, int n, const long long *__restrict__ offset,
                                                            const int *__restrict__ named, const double *__restrict__ x, double *__restrict__ rij)
{
  const int lane = threadIdx.x & 63;
  const int q = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= n) return;
  const long long i = atom[q];
  const double xi0 = x[3 * i], xi1 = x[3 * i + 1], xi2 = x[3 * i + 2];
  for (long long p = offset[q] + lane, e = offset[q + 1]; p < e; p += 64) {
    const long long a = named[p];
    rij[3 * p] = x[3 * a] - xi0;
    rij[3 * p + 1] = x[3 * a + 1] - xi1;
    rij[3 * p + 2] = x[3 * a + 2] - xi2;
  }
}

// buffers of the converted list, kept between calls
struct LammpsDeviceList {
  DevBuf idx, atom, mapped, count, err, offset, j, rij, named;
  int64_t nb = 0;
  // what the kept list was made for: a call that says "same list" and matches it only renews the bond vectors
  bool kept = false;
  int n = 0, nlocal = 0, nall = 0, inum = 0, nodes = 0, neighmask = 0;
  long long stride_i = 0, stride_k = 0;
  const void *neighbors = nullptr, *type = nullptr, *numneigh = nullptr, *owner = nullptr;
  uint64_t serial = 0;
};

}    // namespace grhip
