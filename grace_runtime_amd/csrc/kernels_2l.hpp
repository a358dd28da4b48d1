// HIP kernels of the second message-passing layer of GRACE-2L for gfx950.
//
//   k_sh_edges     Y_lm and the gradient of its polynomial extension for every edge, once per pass, written coalesced
//   k_fill_slot    the species weights zB0[mu_j] as one more "message function" of every atom
//   k_pair_fwd     P[slot][lm][n] = sum_b Y_lm(b) R1_l(b)[n] M_jb[slot][n]: the neighbour gather of the messages
//                  (slots 0 .. nI-1: the equivariant message I_j; slot nI: zB0, which gives B0)
//                  (atom_yi / atom_scatter, libgrace/include/grace/fused_cpu.h:947-1025)
//   k_pair_bwd_mfma, k_pair_bwd[_async]  its reverse: per-bond force of layer 2, dE/dI_j added to the neighbour's row
//                  (bond_yi_bwd_g, bond_yi_commit, bond_scatter_bwd_t, bond_force: fused_cpu.h:836-942,1027-1050); the first
//                  forms the sums over m on the matrix cores, the others on the vector unit
//   k_energy_2l_hidden, k_energy_2l    readout with the two RMSNorms, fp64 (libgrace/src/fused_2l.cpp:548-615)
//
// The vector kernels of the reverse run one block per atom with one thread per (slot, channel): a thread keeps its 2l+1 .. nlm
// adjoints in registers and walks the atom's bonds; everything that is the same for the whole block (neighbour index, Y, G of
// the bond) is read through uniform addresses.
#pragma once

#include "kernels_1l.hpp"

namespace grhip {

// One thread per edge: YG[e] = (Y[nlm], D1[nlm], D2[nlm]) (row width W = 3 nlm), or Y[nlm] alone (W = nlm, no
// gradients), in rows of `stride` >= W values, the rest of a row zero.  D1 = G . e1, D2 = G . e2 are the components of the gradient G of the polynomial extension of Y along the
// tangent vectors of the bond (tangent_basis): the bond force only uses the part of sum_lm gY_lm G_lm normal to the bond,
// g - (g . rhat) rhat = (g . e1) e1 + (g . e2) e2, so two components per harmonic carry all of it.
// The lanes write their rows into an LDS tile, the block copies the tile out in consecutive addresses.
// block: 64 threads; dynamic LDS: 64 * (W + 1) values.
template<class T> __global__ void k_sh_edges(ShCoef sh, const double *rh, const long long *n_edges, int nlm, int grad, T *YG, int stride)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *tile = reinterpret_cast<T *>(smem_raw);
  const int W = grad ? 3 * nlm : nlm, t = threadIdx.x;
  const long long ne = *n_edges, e0 = blockIdx.x * 64ll, e = e0 + t;
  if (e0 >= ne) return;
  if (e < ne) {
    const double *u = rh + 3 * e;
    T *row = tile + t * (W + 1);
    if (grad) {
      double e1[3], e2[3];
      tangent_basis(u, e1, e2);
      sh_eval<true, T>(sh, u[0], u[1], u[2], row, row + nlm, e1, e2, row + 2 * nlm);
    } else {
      sh_eval<false, T>(sh, u[0], u[1], u[2], row, nullptr);
    }
  }
  __syncthreads();
  const int rows = (int) (ne - e0 < 64 ? ne - e0 : 64);
  T *out = YG + e0 * stride;
  for (int q = t; q < rows * stride; q += 64) {
    const int r = q / stride, col = q % stride;
    out[q] = col < W ? tile[r * (W + 1) + col] : (T) 0;
  }
}

// M[atom][slot][n] = z[mu_atom][n] by the first `fill_blocks` blocks; the others clear what the reverse pair kernel adds to (two
// arrays of 8-byte words, 4 a thread).  As two fills of their own the arrays cost 3 us each below some thousand atoms.
constexpr int kClearWords = 4;
template<class T> __global__ __launch_bounds__(256) void k_fill_slot(const int *mu, const T *z, T *M, int natoms, int nslot, int slot, int C, unsigned fill_blocks,
                                                                     unsigned long long *clear0, long long n0, unsigned long long *clear1, long long n1)
{
  if (blockIdx.x >= fill_blocks) {
    const long long first = (long long) (blockIdx.x - fill_blocks) * (256 * kClearWords) + threadIdx.x;
#pragma unroll
    for (int w = 0; w < kClearWords; w++) {
      const long long q = first + w * 256;
      if (q < n0) clear0[q] = 0;
      else if (q < n0 + n1) clear1[q - n0] = 0;
    }
    return;
  }
  const long long q = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (q >= (long long) natoms * C) return;
  const int at = (int) (q / C), n = (int) (q % C);
  M[((long long) at * nslot + slot) * C + n] = z[mu[at] * C + n];
}
constexpr int kPairChunk = 8;    // bonds staged in LDS at a time by the pair kernel that stages through registers
constexpr size_t kPairLdsMax = 158 * 1024;    // dynamic LDS a pair kernel may ask for

// Block -> (atom, slot group).  ngrp == 0: a (atoms, groups) grid.  ngrp > 0: a 1-d grid of 8 ceil(atoms / 8) ngrp
// blocks laid out so that the groups of one atom are blocks b, b + 8, b + 16 ...: workgroups go to the 8 XCDs in turn,
// so those blocks run on ONE XCD shortly after each other and find the atom's radial rows and harmonics in its L2.
__device__ inline bool pair_block(int ngrp, int natoms, int &atom, int &grp)
{
  if (ngrp == 0) {
    atom = blockIdx.x;
    grp = blockIdx.y;
    return true;
  }
  const int b = blockIdx.x, q = b >> 3;
  grp = q % ngrp;
  atom = (q / ngrp) * 8 + (b & 7);
  return atom < natoms;
}

// Stages what a chunk of nb bonds (edges base .. base + nb) needs into LDS with all loads in flight at once: the
// neighbour rows M_j[slot][n] of this thread, the radial rows (contiguous in memory, or row erow[e] of bond e), and touches the harmonics of the
// chunk (the first yuse values of every row of ylen) so that the uniform (scalar) reads of the bond loop find them in
// the L2.
template<class T>
__device__ inline T pair_stage(const int *__restrict__ ej, const T *__restrict__ M, const T *__restrict__ R1, const T *__restrict__ dR1,
                               const T *__restrict__ Yu, int ylen, int yuse, long long base, int nb, int nslot, int C, int nrow, bool active, int slot,
                               int n, T *Msh, T *Rsh, T *dRsh, int NT, const int *__restrict__ erow)
{
  const int t = threadIdx.x;
  T mv[kPairChunk];
#pragma unroll
  for (int b = 0; b < kPairChunk; b++) {
    const int j = b < nb ? ej[base + b] : 0;
    mv[b] = (active && b < nb) ? M[((long long) j * nslot + slot) * C + n] : (T) 0;
  }
  if (erow) {
    for (int b = 0; b < nb; b++) {
      const long long row = (long long) erow[base + b] * nrow;
      for (int q = t; q < nrow; q += blockDim.x) {
        Rsh[b * nrow + q] = R1[row + q];
        if (dR1) dRsh[b * nrow + q] = dR1[row + q];
      }
    }
  } else {
    const T *rs = R1 + base * nrow, *drs = dR1 ? dR1 + base * nrow : nullptr;
    for (int q = t; q < nb * nrow; q += blockDim.x) {
      Rsh[q] = rs[q];
      if (drs) dRsh[q] = drs[q];
    }
  }
  T touch = (T) 0;
  const T *yu = Yu + base * ylen;
  const int per = (yuse + 7) / 8;    // 64-byte pieces of a row that the bond loop reads
  for (int q = t; q < nb * per; q += blockDim.x) touch += yu[(q / per) * ylen + (q % per) * 8];
#pragma unroll
  for (int b = 0; b < kPairChunk; b++) Msh[b * NT + t] = mv[b];
  return touch;
}

// sums of 4 values per lane over the wave with 7 exchanges: afterwards lanes 0, 1, 2, 3 hold the totals of
// v0, v2, v1, v3
__device__ inline double wave_sum4(double v0, double v1, double v2, double v3, int lane)
{
  const bool b0 = lane & 1, b1 = lane & 2;
  double a = b0 ? v2 : v0, b = b0 ? v3 : v1;
  const double sa = b0 ? v0 : v2, sb = b0 ? v1 : v3;
  a += __shfl_xor(sa, 1, 64);
  b += __shfl_xor(sb, 1, 64);
  double c = b1 ? b : a;
  const double sc = b1 ? a : b;
  c += __shfl_xor(sc, 2, 64);
#pragma unroll
  for (int o = 4; o < 64; o <<= 1) c += __shfl_xor(c, o, 64);
  return c;
}

// grid: (atoms, slot groups); block: spb * C threads rounded up to a wave, spb slots per block (a kernel argument);
// dynamic LDS: kPairChunk * (NT + 2 nl C) values.  Every block adds the force of its slots to the bond's two atoms.
// The atoms are a chunk of the structure: eoff, gP start at the chunk's first atom a0; ej, M, gM, f, sid, the harmonics
// and the radial rows are indexed by the atom's or the bond's number in the structure.
// gP: adjoint of P of the atom.
//   S_l = sum_m Y_lm gP[lm],  T_l,k = sum_m D_k,lm gP[lm], k = 1, 2 (tangential gradients)   (per thread: slot, n)
//   dE/dI_j[slot][n] += sum_l R1_l S_l                                        (slots < nI)
//   dE/dx = sum_{slot,n,l} S_l dR1_l M_j,   g_k = sum_{slot,n,l} T_l,k R1_l M_j
//   fv = dE/dx / rc rhat + (g_1 e1 + g_2 e2) / r  (= the reference's dE/dx / rc rhat + (g - (g . rhat) rhat) / r with
//   g the Cartesian sum);  f_i += fv, f_j -= fv, virial += (-r rhat) (x) fv
// ORD (ordered sums): no floating-point atomics.  The message adjoint of bond e goes to ord.gMe[e - ord.e_base][slot][n],
// the force that the block's slot group gives the bond to ord.fedge[e][group][3], the sums over the atom's bonds to
// ord.fcen[a0 + i][group][9] (ord.ngrp groups: with one group these are the engine's per-bond and per-atom stores, with
// several k_ordered_combine adds the groups in turn); the sums over the waves of a block are added in the order of the waves.
template<class T> struct PairOrdered {
  T *gMe;
  double *fedge, *fcen;
  long long e_base;
  int ngrp;
};
template<class T, int NLM, bool ORD = false>
__global__ void k_pair_bwd(const long long *__restrict__ eoff, const int *__restrict__ ej, const T *__restrict__ YG,
                           const T *__restrict__ R1, const T *__restrict__ dR1, const T *__restrict__ M, const T *__restrict__ gP,
                           const double *__restrict__ rh, const double *__restrict__ rlen, const double *__restrict__ rcut,
                           T *__restrict__ gM, double *__restrict__ f, double *__restrict__ virial, int nslot, int nI, int C, int nl,
                           int noutp, T *__restrict__ sink, int one, const int *__restrict__ sid, int spb, int ngrp, int natoms, int a0,
                           double *__restrict__ vatom, int ystr, const int *__restrict__ erow, PairOrdered<T> ord)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double bsum[kPairChunk][4];
  __shared__ double bwave[ORD ? kPairChunk : 1][ORD ? 16 : 1][4];    // ORD: the sums of every wave (at most 16 waves)
  int i, grp;
  if (!pair_block(ngrp, natoms, i, grp)) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, NT = blockDim.x;
  T *Msh = reinterpret_cast<T *>(smem_raw), *Rsh = Msh + kPairChunk * NT, *dRsh = Rsh + kPairChunk * noutp;
  const int slot_raw = grp * spb + t / C;
  const bool active = t < spb * C && slot_raw < nslot;
  const int slot = active ? slot_raw : 0, n = t % C;
  const int nlm = nl * nl;
  const long long e0 = eoff[i], e1 = eoff[i + 1];
  T g[NLM];
  {
    const T *gp = gP + ((long long) i * nslot + slot) * nlm * C + n;
#pragma unroll
    for (int q = 0; q < NLM; q++) g[q] = (active && q < nlm) ? gp[(long long) q * C] : (T) 0;
  }
  double fi[3] = {0, 0, 0}, vir[6] = {0, 0, 0, 0, 0, 0};
  T touch = (T) 0;
  for (long long base = e0; base < e1; base += kPairChunk) {
    const int nb = (int) (e1 - base < kPairChunk ? e1 - base : kPairChunk);
    __syncthreads();
    touch += pair_stage<T>(ej, M, R1, dR1, YG, ystr, nlm * 3, base, nb, nslot, C, noutp, active, slot, n, Msh, Rsh, dRsh, NT, erow);
    if (t < kPairChunk * 4) bsum[t >> 2][t & 3] = 0.0;
    __syncthreads();
    for (int b = 0; b < nb; b++) {
      const long long e = base + b;
      const T m = Msh[b * NT + t];
      const T *r = Rsh + b * noutp + n, *dr = dRsh + b * noutp + n;
      const T *yg = YG + e * ystr;
      T sI = (T) 0, dE = (T) 0, t1 = (T) 0, t2 = (T) 0;
      // every l is the body of a loop that runs `one` (= 1, a kernel argument) times: its uniform loads then stay inside
      // it (all harmonics of a bond at once need more scalar registers than there are)
#pragma unroll
      for (int l = 0; l <= kKernMaxL; l++)
        if (l * l < NLM) for (int it = 0; it < one; it++) {
          T S = (T) 0, a1 = (T) 0, a2 = (T) 0;
#pragma unroll
          for (int mm = 0; mm < 2 * l + 1; mm++) {
            const T gv = g[l * l + mm];
            S += yg[l * l + mm] * gv; a1 += yg[nlm + l * l + mm] * gv; a2 += yg[2 * nlm + l * l + mm] * gv;
          }
          const T rl = r[l * C], drl = dr[l * C];
          sI += rl * S;
          dE += drl * S;
          t1 += rl * a1; t2 += rl * a2;
        }
      if (active && slot < nI) {
        if (ORD) ord.gMe[((e - ord.e_base) * nI + slot) * C + n] = sI;
        else atomicAdd(&gM[((long long) ej[e] * nI + slot) * C + n], sI);
      }
      const double c = wave_sum4((double) (dE * m), (double) (t1 * m), (double) (t2 * m), 0.0, lane);
      if (lane < 3) {    // lanes 0..2: dE/dx, g . e2, g . e1  (order v0, v2, v1, v3)
        if (ORD) bwave[b][wave][lane] = c;
        else atomicAdd(&bsum[b][lane], c);
      }
    }
    __syncthreads();
    if (ORD && t < nb)
      for (int k = 0; k < 3; k++) {
        double sw = 0.0;
        for (int w = 0; w < (NT >> 6); w++) sw += bwave[t][w][k];
        bsum[t][k] = sw;
      }
    if (t < nb) {
      const long long e = base + t;
      const double *u = rh + 3 * e;
      const double r = rlen[e], rc = rcut[e];
      const double dEdr = bsum[t][0] / rc, g1 = bsum[t][2] / r, g2 = bsum[t][1] / r;
      double e1[3], e2[3], fv[3];
      tangent_basis(u, e1, e2);
      for (int d = 0; d < 3; d++) fv[d] = dEdr * u[d] + g1 * e1[d] + g2 * e2[d];
      const int jj = ej[e];
      for (int d = 0; d < 3; d++) {
        fi[d] += fv[d];
        if (ORD) ord.fedge[3 * (e * ord.ngrp + grp) + d] = fv[d];
        else atomicAdd(&f[3 * (long long) jj + d], -fv[d]);
      }
      const double ddx = -u[0] * r, ddy = -u[1] * r, ddz = -u[2] * r;
      vir[0] += ddx * fv[0]; vir[1] += ddy * fv[1]; vir[2] += ddz * fv[2];
      vir[3] += ddx * fv[1]; vir[4] += ddx * fv[2]; vir[5] += ddy * fv[2];
      if (!ORD && vatom) {    // per-atom virial: the neighbour's half of this bond (fused_cpu.h:1075-1087 of the reference)
        double *vj = vatom + 9 * (long long) jj;
        atomicAdd(vj, 0.5 * ddx * fv[0]); atomicAdd(vj + 1, 0.5 * ddy * fv[1]); atomicAdd(vj + 2, 0.5 * ddz * fv[2]);
        atomicAdd(vj + 3, 0.5 * ddx * fv[1]); atomicAdd(vj + 4, 0.5 * ddx * fv[2]); atomicAdd(vj + 5, 0.5 * ddy * fv[2]);
        // the components below the diagonal (the centroid form, kk/grace_1l_kk_impl.h:1344-1349), for both atoms of the bond
        double *vi = vatom + 9 * (long long) (a0 + i);
        const double yx = 0.5 * ddy * fv[0], zx = 0.5 * ddz * fv[0], zy = 0.5 * ddz * fv[1];
        atomicAdd(vj + 6, yx); atomicAdd(vj + 7, zx); atomicAdd(vj + 8, zy);
        atomicAdd(vi + 6, yx); atomicAdd(vi + 7, zx); atomicAdd(vi + 8, zy);
      }
    }
  }
  // the finishing threads t < kPairChunk sit in wave 0
  if (wave == 0) {
    double vsum[9] = {fi[0], fi[1], fi[2], vir[0], vir[1], vir[2], vir[3], vir[4], vir[5]};
#pragma unroll
    for (int k = 0; k < 9; k++)
      for (int o = 32; o > 0; o >>= 1) vsum[k] += __shfl_xor(vsum[k], o, 64);
    if (ORD) {
      if (lane == 0)
        for (int k = 0; k < 9; k++) ord.fcen[9 * ((long long) (a0 + i) * ord.ngrp + grp) + k] = vsum[k];
    } else if (lane == 0 && e1 > e0) {
      for (int k = 0; k < 3; k++) atomicAdd(&f[3 * (long long) (a0 + i) + k], vsum[k]);
      for (int k = 0; k < 6; k++) atomicAdd(&virial[record_of(sid, a0 + i) + k], vsum[3 + k]);
      if (vatom)
        for (int k = 0; k < 6; k++) atomicAdd(&vatom[9 * (long long) (a0 + i) + k], 0.5 * vsum[3 + k]);
    }
  }
  if (touch == (T) 1.2345e300) sink[0] = touch;    // keeps the touching loads alive
}

// Ordered sums with several slot groups per atom: fedge[e][3] (=, or += with add) the sum over the groups, in their order, of
// fpart[e][group][3] for the bonds [e_base, e_end), and fcen[i][9] likewise of cpart[i][group][9] for the atoms [a0, a0 + natoms).
static __global__ void k_ordered_combine(const double *__restrict__ fpart, const double *__restrict__ cpart, int ngrp, long long e_base,
                                         const long long *__restrict__ e_end_dev, long long e_count, int a0, int natoms, int add,
                                         double *__restrict__ fedge, double *__restrict__ fcen)
{
  const long long e_end = e_count >= 0 ? e_base + e_count : *e_end_dev;
  const long long ne3 = 3 * (e_end - e_base), t = blockIdx.x * (long long) blockDim.x + threadIdx.x;
  if (t < ne3) {
    const long long e = e_base + t / 3;
    const int d = (int) (t % 3);
    double s = add ? fedge[3 * e + d] : 0.0;
    for (int g = 0; g < ngrp; g++) s += fpart[3 * (e * ngrp + g) + d];
    fedge[3 * e + d] = s;
  } else if (t < ne3 + 9ll * natoms) {
    const long long q = t - ne3, i = a0 + q / 9;
    const int k = (int) (q % 9);
    double s = add ? fcen[9 * i + k] : 0.0;
    for (int g = 0; g < ngrp; g++) s += cpart[9 * (i * ngrp + g) + k];
    fcen[9 * i + k] = s;
  }
}

// Ordered sums: gM[j][slot][n] += sum of gMe[e - e_base][slot][n] over the bonds e in [e_base, e_end) that have j as their
// neighbour, in ascending order of e (sorted: the bonds by neighbour atom, each row ascending; ncol = nI C columns).
// One block per atom j; a thread owns columns, so no two threads add to one value.
template<class T>
__global__ void k_ordered_gm(const long long *__restrict__ toff, const int *__restrict__ sorted, const T *__restrict__ gMe, long long e_base,
                             const long long *__restrict__ e_end_dev, long long e_count, int ncol, T *__restrict__ gM)
{
  const int j = blockIdx.x;
  const long long t0 = toff[j], t1 = toff[j + 1];
  const long long e_end = e_count >= 0 ? e_base + e_count : *e_end_dev;
  for (int col = threadIdx.x; col < ncol; col += blockDim.x) {
    T s = (T) 0;
    for (long long p = t0; p < t1; p++) {
      const long long e = sorted[p];
      if (e >= e_base && e < e_end) s += gMe[(e - e_base) * ncol + col];
    }
    gM[(long long) j * ncol + col] += s;
  }
}

// acc[f] += y[f] x_l(f) for the functions f = l^2 + m of one slot, y[f] being value f % 16 of every row of 16 lanes of y[f / 16]: the
// multiply-add takes its factor from another lane of the row (row_newbcast) at no cost.  One asm statement per 16 functions: it
// opens with the wait states of a DPP operand behind a vector instruction that wrote it, which the compiler does not count.
#define GR_BF(TY, K, X) "v_fmac_" TY "_dpp %" #K ", %[y], %[" #X "] row_newbcast:" #K " row_mask:0xf bank_mask:0xf\n\t"
#define GR_BF_0_1(TY) "s_nop 1\n\t" GR_BF(TY, 0, p)
#define GR_BF_0_4(TY) GR_BF_0_1(TY) GR_BF(TY, 1, q) GR_BF(TY, 2, q) GR_BF(TY, 3, q)
#define GR_BF_0_9(TY) GR_BF_0_4(TY) GR_BF(TY, 4, r) GR_BF(TY, 5, r) GR_BF(TY, 6, r) GR_BF(TY, 7, r) GR_BF(TY, 8, r)
#define GR_BF_0_16(TY) GR_BF_0_9(TY) GR_BF(TY, 9, s) GR_BF(TY, 10, s) GR_BF(TY, 11, s) GR_BF(TY, 12, s) GR_BF(TY, 13, s) GR_BF(TY, 14, s) GR_BF(TY, 15, s)
#define GR_BF_1_9(TY) "s_nop 1\n\t" GR_BF(TY, 0, p) GR_BF(TY, 1, p) GR_BF(TY, 2, p) GR_BF(TY, 3, p) GR_BF(TY, 4, p) GR_BF(TY, 5, p) GR_BF(TY, 6, p) GR_BF(TY, 7, p) GR_BF(TY, 8, p)
#define GR_BF_1_16(TY) GR_BF_1_9(TY) GR_BF(TY, 9, q) GR_BF(TY, 10, q) GR_BF(TY, 11, q) GR_BF(TY, 12, q) GR_BF(TY, 13, q) GR_BF(TY, 14, q) GR_BF(TY, 15, q)
#define GR_BF_2_4(TY) "s_nop 1\n\t" GR_BF(TY, 0, p) GR_BF(TY, 1, p) GR_BF(TY, 2, p) GR_BF(TY, 3, p)
#define GR_BF_2_16(TY) GR_BF_2_4(TY) GR_BF(TY, 4, q) GR_BF(TY, 5, q) GR_BF(TY, 6, q) GR_BF(TY, 7, q) GR_BF(TY, 8, q) GR_BF(TY, 9, q) GR_BF(TY, 10, q) GR_BF(TY, 11, q) GR_BF(TY, 12, q) GR_BF(TY, 13, q) GR_BF(TY, 14, q) GR_BF(TY, 15, q)
#define GR_BF_3_1(TY) "s_nop 1\n\t" GR_BF(TY, 0, p)
#define GR_BO_1(a) "+v"((a)[0])
#define GR_BO_4(a) GR_BO_1(a), "+v"((a)[1]), "+v"((a)[2]), "+v"((a)[3])
#define GR_BO_9(a) GR_BO_4(a), "+v"((a)[4]), "+v"((a)[5]), "+v"((a)[6]), "+v"((a)[7]), "+v"((a)[8])
#define GR_BO_16(a) GR_BO_9(a), "+v"((a)[9]), "+v"((a)[10]), "+v"((a)[11]), "+v"((a)[12]), "+v"((a)[13]), "+v"((a)[14]), "+v"((a)[15])
#define GR_BFMA(B, N, Y, ...)                                                                    \
  {                                                                                              \
    if constexpr (sizeof(T) == 8) asm(GR_BF_##B##_##N("f64") : GR_BO_##N(a + 16 * B) : [y] "v"(Y), __VA_ARGS__); \
    else asm(GR_BF_##B##_##N("f32") : GR_BO_##N(a + 16 * B) : [y] "v"(Y), __VA_ARGS__);  \
  }
template<int NL, class T> __device__ inline __attribute__((always_inline)) void bcast_fma(T *a, const T *y, const T *x)
{
  if constexpr (NL == 1) GR_BFMA(0, 1, y[0], [p] "v"(x[0]))
  if constexpr (NL == 2) GR_BFMA(0, 4, y[0], [p] "v"(x[0]), [q] "v"(x[1]))
  if constexpr (NL == 3) GR_BFMA(0, 9, y[0], [p] "v"(x[0]), [q] "v"(x[1]), [r] "v"(x[2]))
  if constexpr (NL >= 4) GR_BFMA(0, 16, y[0], [p] "v"(x[0]), [q] "v"(x[1]), [r] "v"(x[2]), [s] "v"(x[3]))
  if constexpr (NL == 5) GR_BFMA(1, 9, y[1], [p] "v"(x[4]))
  if constexpr (NL >= 6) GR_BFMA(1, 16, y[1], [p] "v"(x[4]), [q] "v"(x[5]))
  if constexpr (NL == 6) GR_BFMA(2, 4, y[2], [p] "v"(x[5]))
  if constexpr (NL == 7) GR_BFMA(2, 16, y[2], [p] "v"(x[5]), [q] "v"(x[6]))
  if constexpr (NL == 7) GR_BFMA(3, 1, y[3], [p] "v"(x[6]))
}

// ---- the neighbour gather
// P[slot][lm][n] of an atom = sum over its bonds of Y_lm R1_l[n] M_j[slot][n], the bonds in their order.
// A wave owns `width` channels of NQ `rows` slots (a lane: one channel, slots s0 + q rows + lane / width, q < NQ) and walks the bonds
// alone: no LDS, no barrier.  The rows of the bond after the one being worked on are in flight; addresses are a uniform base
// in scalar registers and a constant offset of the lane; the harmonics come as one value per lane and reach the
// multiply-adds through their lane-broadcast operand.
// Against its predecessor (a block per atom and group of slots, operands staged in LDS by chunks of four bonds, harmonics through
// scalar loads, a thread per slot and channel): a radial row is read once for NQ slots instead of from LDS for each, and no wave
// waits for another.  GRACE-2L, 8000 atoms fp64 456 -> 332 us, 3999 atoms fp32 150 -> 85; GRACE-3L, 72 slots, 701 atoms fp32 583 ->
// 395, 3001 atoms fp64 3.53 -> 3.26 ms, 96 atoms 127 -> 99 us.  What bounds it: instruction issue (in fp64 the 42 multiply-adds of a
// slot, channel and bond at lmax 5 are 1.1 of the 3.26 ms, the stores of P 0.8): with the rows of all neighbours, or all radial
// rows, the same it is at most 12 % faster.  Two bonds ahead instead of one: the same; one slot per lane instead of two: 1.6 x the time.
// Behind the form through LDS in one range only: fp64, a row per bond, 5 slots of 32 channels, lmax 4, whose waves
// fit the GPU once up to 2048 atoms (2000 atoms 90 -> 82 us, 3456 142 -> 150, 5488 206 -> 214, 8192 297 -> 286).
template<class T> struct PairFwdArgs {
  const long long *eoff;
  const int *ej, *erow;    // erow: radial row of every bond (k_edge_pairs), or null: row e
  const T *Y, *R1, *M;
  T *P;
  int nslot, C, noutp, ystride, natoms;
  int width, rows, chunks;    // lanes of a slot; slots side by side in a wave; waves that share the channels of a slot
  int waves, wpb, ngrp;       // waves of an atom, of a block; blocks of an atom
};
// Slots of a lane: what leaves room for the rows of two bonds with two waves per SIMD in fp64, three in fp32 (701 atoms, 72 slots:
// 3 slots and three waves 395 us, 4 slots and two waves 444, 2 slots and four 428)
constexpr int pair_fwd_slots(int nlm, size_t value_bytes)
{
  const int q = (value_bytes == 8 ? 80 : 110) / nlm;
  return q < 1 ? 1 : q > 4 ? 4 : q;
}

template<class T, int NL, int NQ>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 3 : 2) void k_pair_fwd(PairFwdArgs<T> a)
{
  constexpr int NLM = NL * NL, NY = (NLM + 15) / 16, SETS = 2;
  int i, grp;
  if (!pair_block(a.ngrp, a.natoms, i, grp)) return;
  const int lane = threadIdx.x & 63, w = grp * a.wpb + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);    // wave of the atom
  if (w >= a.waves) return;
  const int h = lane / a.width, n = (w % a.chunks) * a.width + lane - h * a.width, s0 = (w / a.chunks) * NQ * a.rows;
  const bool active = h < a.rows && n < a.C;
  const unsigned nc = active ? n : 0;
  unsigned mo[NQ], yo[NY];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int s = s0 + q * a.rows + h;
    mo[q] = ((active && s < a.nslot ? s : 0) * a.C + nc) * (unsigned) sizeof(T);
  }
#pragma unroll
  for (int k = 0; k < NY; k++) yo[k] = (16 * k + (lane & 15) < NLM ? 16 * k + (lane & 15) : NLM - 1) * (unsigned) sizeof(T);
  unsigned ro[NL];
#pragma unroll
  for (int l = 0; l < NL; l++) ro[l] = (l * a.C + nc) * (unsigned) sizeof(T);
  // a uniform base in scalar registers and the lane's offset: the empty statement keeps the compiler from adding the two ahead
  typedef const char __attribute__((address_space(1))) *bytes_t;
  typedef const T __attribute__((address_space(1))) *value_t;
  auto uniform = [](const T *p) {
    bytes_t b = (bytes_t) p;
    asm("" : "+s"(b));
    return b;
  };
  auto load = [](bytes_t base, unsigned offset) {
    asm("" : "+v"(offset) : "s"(base));
    return *(value_t) (base + offset);
  };
  const long long e0 = a.eoff[i], e1 = a.eoff[i + 1];
  const int nb = (int) (e1 - e0);
  T acc[NQ][NLM];
#pragma unroll
  for (int q = 0; q < NQ; q++)
#pragma unroll
    for (int f = 0; f < NLM; f++) acc[q][f] = (T) 0;
  if (nb > 0) {
    // the neighbour and radial row of the bond requested next are read one request ahead
    const int *rowlist = a.erow ? a.erow : a.ej;
    int jn = a.ej[e0], rn = rowlist[e0];
    T r[SETS][NL], m[SETS][NQ], y[SETS][NY];
    auto request = [&](int b, T (&rr)[NL], T (&mm)[NQ], T (&yy)[NY]) {      // behind the last bond: the last bond again
      const long long e = e0 + (b < nb ? b : nb - 1), next = e0 + (b + 1 < nb ? b + 1 : nb - 1);
      const bytes_t Rb = uniform(a.R1 + (a.erow ? rn : e) * a.noutp), Mb = uniform(a.M + (long long) jn * (a.nslot * a.C)), Yb = uniform(a.Y + e * a.ystride);
      jn = a.ej[next];
      rn = rowlist[next];
#pragma unroll
      for (int l = 0; l < NL; l++) rr[l] = load(Rb, ro[l]);
#pragma unroll
      for (int q = 0; q < NQ; q++) mm[q] = load(Mb, mo[q]);
#pragma unroll
      for (int k = 0; k < NY; k++) yy[k] = load(Yb, yo[k]);
    };
#pragma unroll
    for (int k = 0; k < SETS; k++) request(k, r[k], m[k], y[k]);
    for (int b = 0; b < nb; b += SETS) {
#pragma unroll
      for (int k = 0; k < SETS; k++) {
        __builtin_amdgcn_sched_barrier(0);
        if (b + k < nb) {
#pragma unroll
          for (int q = 0; q < NQ; q++) {
            T x[NL];
#pragma unroll
            for (int l = 0; l < NL; l++) x[l] = r[k][l] * m[k][q];
            bcast_fma<NL>(acc[q], y[k], x);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        request(b + k + SETS, r[k], m[k], y[k]);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int s = s0 + q * a.rows + h;
    if (!active || s >= a.nslot) continue;
    T *o = a.P + ((long long) i * a.nslot + s) * NLM * a.C + n;
#pragma unroll
    for (int f = 0; f < NLM; f++) __builtin_nontemporal_store(acc[q][f], &o[(long long) f * a.C]);
  }
}

template<class T, int NL, int NQ> inline void launch_pair_fwd_q(PairFwdArgs<T> a, hipStream_t stream)
{
  a.chunks = (a.C + 63) / 64;
  a.width = (a.C + a.chunks - 1) / a.chunks;
  a.rows = 64 / a.width;
  a.waves = a.chunks * ((a.nslot + NQ * a.rows - 1) / (NQ * a.rows));
  a.ngrp = (a.waves + 3) / 4;
  a.wpb = (a.waves + a.ngrp - 1) / a.ngrp;
  hipLaunchKernelGGL((k_pair_fwd<T, NL, NQ>), dim3((unsigned) ((a.natoms + 7) / 8 * 8 * a.ngrp)), dim3(64 * a.wpb), 0, stream, a);
}
// Slots of a lane at NL and C: the groups of slots even; where every wave would have a SIMD to itself anyway (simds: of the
// GPU) more waves with fewer slots (107 atoms of GRACE-2L: 31.4 us with three slots, 28.1 with two, 28.3 with one)
template<class T, int NL> inline void launch_pair_fwd_l(const PairFwdArgs<T> &a, int simds, hipStream_t stream)
{
  constexpr int MAXQ = pair_fwd_slots(NL * NL, sizeof(T));
  const int chunks = (a.C + 63) / 64, rows = a.C < 64 ? 64 / a.C : 1, need = (a.nslot + rows - 1) / rows;
  int nq = 1;
  for (; nq < MAXQ; nq++)
    if ((long long) a.natoms * chunks * ((need + nq - 1) / nq) <= simds) break;
  const int groups = (need + nq - 1) / nq;
  nq = (need + groups - 1) / groups;
  if constexpr (MAXQ >= 4) if (nq == 4) return launch_pair_fwd_q<T, NL, 4>(a, stream);
  if constexpr (MAXQ >= 3) if (nq == 3) return launch_pair_fwd_q<T, NL, 3>(a, stream);
  if constexpr (MAXQ >= 2) if (nq == 2) return launch_pair_fwd_q<T, NL, 2>(a, stream);
  launch_pair_fwd_q<T, NL, 1>(a, stream);
}
template<class T> inline void launch_pair_fwd(const PairFwdArgs<T> &a, int nl, int simds, hipStream_t stream)
{
  if (a.natoms == 0) return;
  switch (nl) {
    case 1: return launch_pair_fwd_l<T, 1>(a, simds, stream);
    case 2: return launch_pair_fwd_l<T, 2>(a, simds, stream);
    case 3: return launch_pair_fwd_l<T, 3>(a, simds, stream);
    case 4: return launch_pair_fwd_l<T, 4>(a, simds, stream);
    case 5: return launch_pair_fwd_l<T, 5>(a, simds, stream);
    case 6: return launch_pair_fwd_l<T, 6>(a, simds, stream);
    default: return launch_pair_fwd_l<T, 7>(a, simds, stream);
  }
}

// ---- the reverse pair kernel with asynchronous staging
// The chunk after the one being worked on is copied from global memory straight into a second LDS buffer while the
// waves compute (global_load_lds: no registers, no wait until the end of the chunk), so the memory latency of the
// neighbour rows no longer stands between two chunks.
__device__ inline void lds_load_word(const void *src, void *lds_wave_base)
{
  __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *) src, (void __attribute__((address_space(3))) *) lds_wave_base, 4, 0, 0);
}

// The waves of a block copy nbytes (a multiple of 16, both ends 16-byte aligned) from global memory to LDS: pieces of
// 1 kB are dealt to the waves, a lane moves 16 bytes; the data lands at dst in the order it has at src.
__device__ inline void block_copy_async(const void *src, void *dst, int nbytes, int wave, int nw, int lane)
{
  for (int p = wave; p * 1024 < nbytes; p += nw) {
    const int q = p * 64 + lane;
    if (q * 16 < nbytes)
      __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *) (reinterpret_cast<const char *>(src) + 16 * (size_t) q),
                                       (void __attribute__((address_space(3))) *) (reinterpret_cast<char *>(dst) + 1024 * (size_t) p), 16, 0, 0);
  }
}

// the same for nb rows of nbytes each (multiples of 16), row b from src + row[b] * nbytes, one after another at dst
__device__ inline void block_copy_rows_async(const void *src, const int *__restrict__ row, void *dst, int nb, int nbytes, int wave, int nw, int lane)
{
  const int ppr = nbytes >> 4, total = nb * ppr;    // 16-byte pieces of a row, of the chunk
  for (int p = wave; p * 64 < total; p += nw) {
    const int q = p * 64 + lane;
    if (q < total) {
      const int b = q / ppr;
      __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1))) *) (reinterpret_cast<const char *>(src) + (long long) row[b] * nbytes + 16 * (q - b * ppr)),
                                       (void __attribute__((address_space(3))) *) (reinterpret_cast<char *>(dst) + 1024 * (size_t) p), 16, 0, 0);
    }
  }
}

__device__ inline void wait_async_loads() { __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// k_pair_bwd with asynchronous staging and chunks of CH bonds; same arguments, grid and block.
// dynamic LDS: 2 CH (NT + 2 noutp) values.
template<class T, int NLM, int CH>
__global__ void k_pair_bwd_async(const long long *__restrict__ eoff, const int *__restrict__ ej, const T *__restrict__ YG,
                                 const T *__restrict__ R1, const T *__restrict__ dR1, const T *__restrict__ M, const T *__restrict__ gP,
                                 const double *__restrict__ rh, const double *__restrict__ rlen, const double *__restrict__ rcut,
                                 T *__restrict__ gM, double *__restrict__ f, double *__restrict__ virial, int nslot, int nI, int C, int nl,
                                 int noutp, T *__restrict__ sink, int one, const int *__restrict__ sid, int spb, int ngrp, int natoms, int a0,
                                 double *__restrict__ vatom, int ystr, const int *__restrict__ erow)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ double bsum[2][CH][4];
  __shared__ __align__(16) double g_rh[2][CH * 3], g_r[2][CH], g_rc[2][CH];
  __shared__ __align__(16) int g_j[2][CH];
  int i, grp;
  if (!pair_block(ngrp, natoms, i, grp)) return;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, NT = blockDim.x, nw = NT >> 6;
  T *Msh = reinterpret_cast<T *>(smem_raw), *Rsh = Msh + 2 * CH * NT, *dRsh = Rsh + 2 * CH * noutp;
  const int slot_raw = grp * spb + t / C;
  const bool active = t < spb * C && slot_raw < nslot;
  const int slot = active ? slot_raw : 0, n = t % C;
  const int nlm = nl * nl;
  // threads of the block with a slot: the first nact (slots grp spb .. of the atom's rows, C values each)
  const int nact = (nslot - grp * spb < spb ? nslot - grp * spb : spb) * C;
  const long long e0 = eoff[i], e1 = eoff[i + 1];
  const int nchunk = (int) ((e1 - e0 + CH - 1) / CH);
  T g[NLM];
  {
    const T *gp = gP + ((long long) i * nslot + slot) * nlm * C + n;
#pragma unroll
    for (int q = 0; q < NLM; q++) g[q] = (active && q < nlm) ? gp[(long long) q * C] : (T) 0;
  }
  for (int q = t; q < 2 * CH * NT; q += NT) Msh[q] = (T) 0;
  if (t < 2 * CH * 4) (&bsum[0][0][0])[t] = 0.0;
  __syncthreads();
  // stage(c): everything chunk c needs, into buffer c & 1
  auto stage = [&](int c) {
    const long long base = e0 + (long long) c * CH;
    const int nb = (int) (e1 - base < CH ? e1 - base : CH), buf = c & 1;
    // the rows of the block's slots are contiguous in M_j and in the buffer: nact values per bond
    for (int b = 0; b < nb; b++)
      block_copy_async(M + ((long long) ej[base + b] * nslot + grp * spb) * C, Msh + (size_t) (buf * CH + b) * NT, nact * (int) sizeof(T), (wave + b) % nw,
                       nw, lane);
    if (erow) {
      block_copy_rows_async(R1, erow + base, Rsh + (size_t) buf * CH * noutp, nb, noutp * (int) sizeof(T), (wave + 1) % nw, nw, lane);
      block_copy_rows_async(dR1, erow + base, dRsh + (size_t) buf * CH * noutp, nb, noutp * (int) sizeof(T), (wave + 2) % nw, nw, lane);
    } else {
      block_copy_async(R1 + base * noutp, Rsh + (size_t) buf * CH * noutp, nb * noutp * (int) sizeof(T), (wave + 1) % nw, nw, lane);
      block_copy_async(dR1 + base * noutp, dRsh + (size_t) buf * CH * noutp, nb * noutp * (int) sizeof(T), (wave + 2) % nw, nw, lane);
    }
    if (wave == 0) {
      if (lane < nb * 6) lds_load_word(reinterpret_cast<const char *>(rh + 3 * base) + 4 * lane, &g_rh[buf][0]);
      if (lane < nb * 2) lds_load_word(reinterpret_cast<const char *>(rlen + base) + 4 * lane, &g_r[buf][0]);
      if (lane < nb * 2) lds_load_word(reinterpret_cast<const char *>(rcut + base) + 4 * lane, &g_rc[buf][0]);
      if (lane < nb) lds_load_word(reinterpret_cast<const char *>(ej + base) + 4 * lane, &g_j[buf][0]);
    }
  };
  double fi[3] = {0, 0, 0}, vir[6] = {0, 0, 0, 0, 0, 0};
  T touch = (T) 0;
  // round c stages chunk c + 1 and works on chunk c (round -1 only stages)
  for (int c = -1; c < nchunk; c++) {
    const long long base = e0 + (long long) c * CH;
    const int nb = c < 0 ? 0 : (int) (e1 - base < CH ? e1 - base : CH), buf = c & 1;
    T tv = (T) 0;
    if (c + 1 < nchunk) {
      stage(c + 1);
      // the harmonics of the next chunk, one 64-byte piece per thread, so that its uniform reads find them in the L2
      const long long nbase = base + CH;
      const int nnb = (int) (e1 - nbase < CH ? e1 - nbase : CH), per = (nlm * 3 + 7) / 8;
      if (t < nnb * per) tv = YG[(nbase + t / per) * ystr + (t % per) * 8];
    }
    for (int b = 0; b < nb; b++) {
      const long long e = base + b;
      const T m = Msh[(size_t) (buf * CH + b) * NT + t];
      const T *r = Rsh + (size_t) (buf * CH + b) * noutp + n, *dr = dRsh + (size_t) (buf * CH + b) * noutp + n;
      const T *yg = YG + e * ystr;
      T sI = (T) 0, dE = (T) 0, t1 = (T) 0, t2 = (T) 0;
#pragma unroll
      for (int l = 0; l <= kKernMaxL; l++)
        if (l * l < NLM) for (int it = 0; it < one; it++) {
          T S = (T) 0, a1 = (T) 0, a2 = (T) 0;
#pragma unroll
          for (int mm = 0; mm < 2 * l + 1; mm++) {
            const T gv = g[l * l + mm];
            S += yg[l * l + mm] * gv; a1 += yg[nlm + l * l + mm] * gv; a2 += yg[2 * nlm + l * l + mm] * gv;
          }
          const T rl = r[l * C], drl = dr[l * C];
          sI += rl * S;
          dE += drl * S;
          t1 += rl * a1; t2 += rl * a2;
        }
      if (active && slot < nI) atomicAdd(&gM[((long long) g_j[buf][b] * nI + slot) * C + n], sI);
      const double cs = wave_sum4((double) (dE * m), (double) (t1 * m), (double) (t2 * m), 0.0, lane);
      if (lane < 3) atomicAdd(&bsum[buf][b][lane], cs);    // lanes 0..2: dE/dx, g . e2, g . e1  (order v0, v2, v1, v3)
    }
    touch += tv;
    wait_async_loads();
    __syncthreads();
    // the forces of the chunk: threads 0 .. nb - 1 while the other waves go on; bsum[buf] is clear again before the
    // chunk after the next adds to it (a barrier lies between)
    if (t < nb) {
      const double *u = &g_rh[buf][3 * t];
      const double r = g_r[buf][t], rc = g_rc[buf][t];
      const double dEdr = bsum[buf][t][0] / rc, g1 = bsum[buf][t][2] / r, g2 = bsum[buf][t][1] / r;
      bsum[buf][t][0] = bsum[buf][t][1] = bsum[buf][t][2] = 0.0;
      double e1v[3], e2v[3], fv[3];
      tangent_basis(u, e1v, e2v);
      for (int d = 0; d < 3; d++) fv[d] = dEdr * u[d] + g1 * e1v[d] + g2 * e2v[d];
      const int jj = g_j[buf][t];
      for (int d = 0; d < 3; d++) {
        fi[d] += fv[d];
        atomicAdd(&f[3 * (long long) jj + d], -fv[d]);
      }
      const double ddx = -u[0] * r, ddy = -u[1] * r, ddz = -u[2] * r;
      vir[0] += ddx * fv[0]; vir[1] += ddy * fv[1]; vir[2] += ddz * fv[2];
      vir[3] += ddx * fv[1]; vir[4] += ddx * fv[2]; vir[5] += ddy * fv[2];
      if (vatom) {    // per-atom virial: the neighbour's half of this bond (fused_cpu.h:1075-1087 of the reference)
        double *vj = vatom + 9 * (long long) jj;
        atomicAdd(vj, 0.5 * ddx * fv[0]); atomicAdd(vj + 1, 0.5 * ddy * fv[1]); atomicAdd(vj + 2, 0.5 * ddz * fv[2]);
        atomicAdd(vj + 3, 0.5 * ddx * fv[1]); atomicAdd(vj + 4, 0.5 * ddx * fv[2]); atomicAdd(vj + 5, 0.5 * ddy * fv[2]);
        // the components below the diagonal (the centroid form, kk/grace_1l_kk_impl.h:1344-1349), for both atoms of the bond
        double *vi = vatom + 9 * (long long) (a0 + i);
        const double yx = 0.5 * ddy * fv[0], zx = 0.5 * ddz * fv[0], zy = 0.5 * ddz * fv[1];
        atomicAdd(vj + 6, yx); atomicAdd(vj + 7, zx); atomicAdd(vj + 8, zy);
        atomicAdd(vi + 6, yx); atomicAdd(vi + 7, zx); atomicAdd(vi + 8, zy);
      }
    }
  }
  if (wave == 0) {
    double vsum[9] = {fi[0], fi[1], fi[2], vir[0], vir[1], vir[2], vir[3], vir[4], vir[5]};
#pragma unroll
    for (int k = 0; k < 9; k++)
      for (int o = 32; o > 0; o >>= 1) vsum[k] += __shfl_xor(vsum[k], o, 64);
    if (lane == 0 && e1 > e0) {
      for (int k = 0; k < 3; k++) atomicAdd(&f[3 * (long long) (a0 + i) + k], vsum[k]);
      for (int k = 0; k < 6; k++) atomicAdd(&virial[record_of(sid, a0 + i) + k], vsum[3 + k]);
      if (vatom)
        for (int k = 0; k < 6; k++) atomicAdd(&vatom[9 * (long long) (a0 + i) + k], 0.5 * vsum[3 + k]);
    }
  }
  if (touch == (T) 1.2345e300) sink[0] = touch;    // keeps the touching loads alive
}

// ---- the reverse pair kernel on the matrix cores
// For one atom the adjoints gP[slot][lm][n] are fixed while the bonds change, so per l the three sums over m
//   S_l, T_l,1, T_l,2 [bond][column] = sum_m (Y, D1, D2)[bond][l, m] gP[l, m][column],   column = (slot, n),
// are products of a [16 bonds][2l + 1] tile of the harmonics with a [2l + 1][16 columns] tile of the adjoints: MFMA
// 16x16x4 with the bonds as rows, K = 2l + 1 in steps of 4 (the unused k of the last step are zero in the harmonics).
// Per accumulator value (bond, column, l) four multiply-adds remain for the vector unit:
//   sI += R_l S_l;  U_l += S_l m,  V_l,k += T_l,k m  (m = the neighbour's message value; summed over the wave's slots)
// and per (bond, n, l) three:  dE/dx += dR_l U_l,  g_k += R_l V_l,k.
//
// A wave owns 16 channels of up to kPairMfmaSlots slots of one atom and works alone: nothing is staged for the block and no barrier
// stands inside its loop.  Only the adjoint tiles, which every bond reads, sit in LDS ([slot][lm][16], its own area); the
// harmonics, the radial rows and the message rows of the neighbours come from memory into registers in the layout in which
// they are used.  The harmonics of the next l are requested before the products of one, the neighbours' rows of the next chunk as
// soon as the last products have used this chunk's and before the atomic additions of this chunk are sent (the counter of
// outstanding memory operations is in order: a load behind an atomic waits for it); the longest l comes first, so that the
// first loads behind the atomics have its products to arrive under.
// fp32 and fp64 matrix instructions do not run beside vector instructions of another wave of the SIMD (2000 x 4 fp64 MFMA of one wave
// 243 us, 128 000 fp64 multiply-adds of another 292, both together 525), so what counts is their sum: l = 0, whose harmonic is
// a constant without gradient, takes no matrix step, the last function of an even l (5 = 4 + 1, 9 = 8 + 1) is added by the vector unit
// through its lane-broadcast operand instead of a step of its own (27 steps for three sums at lmax 5 instead of 36), and
// addresses are a uniform base and a constant offset.  Kernel alone, before / now: GRACE-2L, 8000 atoms fp64 1.11 / 1.00 ms, 3999 atoms
// fp32 396 / 341 us; GRACE-3L, 72 slots, 3001 atoms fp64 9.2 / 9.05 ms, 36 slots 4.62 / 4.39, 72 slots, 701 atoms fp32 1.63 / 1.54, 96 atoms
// 0.318 / 0.300.  The vector kernels are behind everywhere.  What bounds it: in fp64 the matrix and vector work (5.2 of the 9.05
// ms) next to the atomic additions, which are written through (1.6 ms of it); which neighbour's rows are read makes no difference.
// Radial rows one l ahead: 2 % in fp32 rows per bond, spills elsewhere; contiguous ranges of atoms per XCD 8 % slower.
// grid: as k_pair_bwd (pair_block, groups of wpb spw slots); block: 64 (C / 16) wpb threads, dynamic LDS per wave:
// (spw NLM + 3) 16 values.
template<class T> struct PairMfmaArgs {
  const long long *eoff;
  const int *ej, *erow;    // erow: radial row of every bond (k_edge_pairs), or null: row e
  const T *YG, *R1, *dR1, *M, *gP;
  T *gM;
  double *bsum;            // [E][3] += sums of the bonds (BondBwdArgs)
  int nslot, nI, C, noutp, ngrp, natoms, ystr;
  int spw, wpb;    // slots of a wave; groups of spw slots of a block
  int drow[16];    // accumulator row of (lane / 16, register)
};

// Matrix steps of l (four k each): l odd, the last holds three; l even, the function left over goes to the vector unit
constexpr int pair_mfma_steps(int l) { return (l + 1) / 2; }
constexpr bool pair_mfma_rest(int l) { return l > 0 && l % 2 == 0; }
// value of lane Q of every row of 16 lanes
template<int Q> __device__ inline double row_bcast(double x)
{
  long long v = __builtin_bit_cast(long long, x);
  v = __builtin_amdgcn_update_dpp(v, v, 0x150 + Q, 0xf, 0xf, true);
  return __builtin_bit_cast(double, v);
}
template<int Q> __device__ inline float row_bcast(float x)
{
  const int v = __builtin_bit_cast(int, x);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(v, v, 0x150 + Q, 0xf, 0xf, true));
}
// slots of a wave: the message values, their adjoints and the adjoint tiles of 4 x 36 functions are what fits two waves per
// SIMD in fp64 (registers and LDS)
constexpr int kPairMfmaSlots = 4;
inline size_t pair_mfma_wave_lds(int nl, int spw, size_t value_bytes) { return ((size_t) spw * nl * nl + 3) * 16 * value_bytes; }

// A wave walks the bonds of its atom, 16 at a time.  Per chunk the l are taken in the order NL - 1, 1, 2 .. NL - 2: the
// longest first, since the loads behind the atomic additions of the chunk before wait for those.
template<class T, int NL, int NQ, bool PAIRS> __device__ inline void pair_bwd_wave(const PairMfmaArgs<T> &a, int i, int s0, int n0, const T *Bw)
{
  typedef typename Mfma<T>::v4 v4;
  typedef const char __attribute__((address_space(1))) *bytes_t;
  typedef const T __attribute__((address_space(1))) *value_t;
  constexpr int NLM = NL * NL, NS = NL - 1, TS = (int) sizeof(T);
  constexpr bool EARLY = NS >= 3;    // the message rows are read for the last time by the products of the last step
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int C = a.C;
  auto scalar = [](long long x) {
    return (long long) (unsigned) __builtin_amdgcn_readfirstlane((int) x) | (long long) __builtin_amdgcn_readfirstlane((int) (x >> 32)) << 32;
  };
  const long long e0 = scalar(a.eoff[i]), e1 = scalar(a.eoff[i + 1]);
  const int nchunk = (int) ((e1 - e0 + 15) / 16);
  if (nchunk == 0) return;
  int rows[4];
#pragma unroll
  for (int v = 0; v < 4; v++) rows[v] = a.drow[4 * g + v];
  const int myrow = a.drow[4 * g + (c & 3)];             // the bond whose sums lane (g, c < 4) ends up with
  // a uniform base in scalar registers and an offset of the lane, in bytes: the empty statements keep the compiler from adding
  // the two ahead of their use (it would keep, and spill, an address per l)
  auto uniform = [](const T *p) {
    bytes_t b = (bytes_t) p;
    asm("" : "+s"(b));
    return b;
  };
  auto load = [](bytes_t b, unsigned offset, int values) {
    asm("" : "+v"(offset) : "s"(b));
    return *(value_t) (b + offset + values * TS);
  };
  // The chunk requested next: its first bond, the neighbours of the lane's four bonds, their radial rows (PAIRS: addresses, else
  // bytes from the chunk's first) and, in bytes from the chunk's first, the lane's row of the harmonics and the row whose left-over
  // functions it holds for its row of 16 lanes.  Bonds beyond the last read the last, what they give is not used.
  const int *rowlist = PAIRS ? a.erow : a.ej;
  long long base = e0;
  int jn[4];
  const T *pr[4];
  unsigned ro[4], yo = 0, yro = 0;
  auto next_bonds = [&](int ch) {
    base = e0 + 16ll * ch;
    const int last = e1 - 1 - base > 15 ? 15 : (int) (e1 - 1 - base);      // negative behind the last chunk
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = rows[v] < last ? rows[v] : last;
      jn[v] = a.ej[base + r];
      if (PAIRS) pr[v] = a.R1 + (long long) rowlist[base + r] * a.noutp + n0 + c;
      else ro[v] = (unsigned) ((r < 0 ? 0 : r) * a.noutp + n0 + c) * TS;
    }
    const int ry = c < last ? c : last, rr = myrow < last ? myrow : last;
    if (last < 0) base = e1 - 1;
    yo = (unsigned) ((ry < 0 ? 0 : ry) * a.ystr + g) * TS;
    yro = (unsigned) ((rr < 0 ? 0 : rr) * a.ystr) * TS;
  };
  auto request_r = [&](T (&R)[4], T (&dR)[4], int l) {
    if (PAIRS) {
      const long long d = reinterpret_cast<const char *>(a.dR1) - reinterpret_cast<const char *>(a.R1) + (long long) l * C * TS;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        R[v] = pr[v][l * C];
        dR[v] = *reinterpret_cast<const T *>(reinterpret_cast<const char *>(pr[v]) + d);
      }
    } else {
      const bytes_t Rb = uniform(a.R1 + base * a.noutp + l * C), dRb = uniform(a.dR1 + base * a.noutp + l * C);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        R[v] = load(Rb, ro[v], 0);
        dR[v] = load(dRb, ro[v], 0);
      }
    }
  };
  T m[NQ][4];
  auto request_m = [&](int q) {
#pragma unroll
    for (int v = 0; v < 4; v++) m[q][v] = a.M[((long long) jn[v] * a.nslot + s0 + q) * C + n0 + c];
  };
  // an offset of zero that the compiler cannot see through: LDS reads stay where they are used
  auto opaque = []() {
    int z = 0;
    asm volatile("" : "+v"(z));
    return z;
  };
  // keeps the accumulation of x where it stands: the compiler otherwise moves the multiply-adds of all l behind the loop, to
  // the branch that uses their sum, and spills every matrix product
  auto pin = [](T &x) { asm volatile("" : "+v"(x)); };
  // y[k][s]: the lane's operand of matrix step s; for l even y[k][steps]: the left-over function of its bond `myrow`
  auto request_y = [&](T (&y)[3][4], int l) {
    const bytes_t Yb = uniform(a.YG + base * a.ystr);
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
      for (int s = 0; s < pair_mfma_steps(l); s++) y[k][s] = load(Yb, yo, k * NLM + l * l + 4 * s);
      if (pair_mfma_rest(l)) y[k][pair_mfma_steps(l)] = load(Yb, yro, k * NLM + l * l + 2 * l);
    }
  };
  auto order = [](int t) { return t == 0 ? NL - 1 : t; };
  const T *Bl = Bw + g * 16 + c;
  const T y00 = a.YG[e0 * a.ystr];                        // the harmonic of l = 0: the same for every bond
  next_bonds(0);
  T y[3][4], yn[3][4], R[4], dR[4], R0[4], dR0[4];
  if (NS > 0) request_y(y, order(0));
#pragma unroll
  for (int q = 0; q < NQ; q++) request_m(q);
  for (int ch = 0; ch < nchunk; ch++) {
    const int nb = (int) (e1 - e0 - 16ll * ch < 16 ? e1 - e0 - 16ll * ch : 16);
    int jc[4];
#pragma unroll
    for (int v = 0; v < 4; v++) jc[v] = jn[v];
    T sI[NQ][4];
    T pE[4], p1[4], p2[4];
#pragma unroll
    for (int q = 0; q < NQ; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) sI[q][v] = (T) 0;
#pragma unroll
    for (int v = 0; v < 4; v++) pE[v] = p1[v] = p2[v] = (T) 0;
    // l = 0: no gradient, and a sum that is the same for every bond
    auto add_l0 = [&]() {
      const int bz = opaque();
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        const T s = y00 * Bw[bz + q * NLM * 16 + c];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          sI[q][v] += R0[v] * s;
          pE[v] += dR0[v] * (s * m[q][v]);
          pin(sI[q][v]); pin(pE[v]);
        }
      }
    };
    if (NS == 0) {
      request_r(R0, dR0, 0);
      next_bonds(ch + 1);
      add_l0();
    }
#pragma unroll
    for (int t = 0; t < NS; t++) {
      const int l = order(t);
      // the radial rows of this l arrive under its first products, the harmonics of the next step under all of them
      request_r(R, dR, l);
      if (l == 1) request_r(R0, dR0, 0);
      if (t + 1 == NS) next_bonds(ch + 1);
      request_y(yn, order(t + 1 < NS ? t + 1 : 0));
      const int bz = opaque();
      __builtin_amdgcn_sched_barrier(0);
      if (!pair_mfma_rest(l)) {    // the fourth k of the last step: zero in the harmonics (the adjoint row read there is another one)
        const int last = pair_mfma_steps(l) - 1;
#pragma unroll
        for (int k = 0; k < 3; k++) y[k][last] = g < 3 ? y[k][last] : (T) 0;
      }
      T U[4] = {0, 0, 0, 0}, V1[4] = {0, 0, 0, 0}, V2[4] = {0, 0, 0, 0};
      const int rest = pair_mfma_steps(l);
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        v4 aS = {0, 0, 0, 0}, a1 = {0, 0, 0, 0}, a2 = {0, 0, 0, 0};
        if (pair_mfma_rest(l)) {
          const T b = Bw[bz + (q * NLM + l * l + 2 * l) * 16 + c];
          T yq[3];
#pragma unroll
          for (int k = 0; k < 3; k++) {
            yq[k] = y[k][rest];
            if (TS == 8) pin(yq[k]);        // in fp64 the twelve broadcast values of an l would be spilled: formed for every slot
          }
          aS = v4{row_bcast<0>(yq[0]) * b, row_bcast<1>(yq[0]) * b, row_bcast<2>(yq[0]) * b, row_bcast<3>(yq[0]) * b};
          a1 = v4{row_bcast<0>(yq[1]) * b, row_bcast<1>(yq[1]) * b, row_bcast<2>(yq[1]) * b, row_bcast<3>(yq[1]) * b};
          a2 = v4{row_bcast<0>(yq[2]) * b, row_bcast<1>(yq[2]) * b, row_bcast<2>(yq[2]) * b, row_bcast<3>(yq[2]) * b};
        }
#pragma unroll
        for (int s = 0; s < pair_mfma_steps(l); s++) {
          const T bq = Bl[bz + (q * NLM + l * l + 4 * s) * 16];
          aS = Mfma<T>::mma(y[0][s], bq, aS);
          a1 = Mfma<T>::mma(y[1][s], bq, a1);
          a2 = Mfma<T>::mma(y[2][s], bq, a2);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
          sI[q][v] += R[v] * aS[v];
          U[v] += aS[v] * m[q][v];
          V1[v] += a1[v] * m[q][v];
          V2[v] += a2[v] * m[q][v];
          pin(sI[q][v]); pin(U[v]); pin(V1[v]); pin(V2[v]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (EARLY && t + 1 == NS) request_m(q);
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        pE[v] += dR[v] * U[v];
        p1[v] += R[v] * V1[v];
        p2[v] += R[v] * V2[v];
        pin(pE[v]); pin(p1[v]); pin(p2[v]);
      }
      if (l == 1) add_l0();
#pragma unroll
      for (int k = 0; k < 3; k++)
#pragma unroll
        for (int q = 0; q < 4; q++) y[k][q] = yn[k][q];
    }
    if (!EARLY) {
#pragma unroll
      for (int q = 0; q < NQ; q++) request_m(q);
    }
    __builtin_amdgcn_sched_barrier(0);
    // dE/dI of the neighbours
#pragma unroll
    for (int v = 0; v < 4; v++) {
      if (rows[v] >= nb) continue;
      T *gm = a.gM + ((long long) jc[v] * a.nI + s0) * C + n0 + c;
#pragma unroll
      for (int q = 0; q < NQ; q++)
        if (s0 + q < a.nI) atomicAdd(&gm[q * C], sI[q][v]);
    }
    // the three sums of the lane's four bonds over the 16 columns: 12 values, halved twice while exchanged, so that
    // lane c holds the sums of register v = c % 4
    double w[12];
#pragma unroll
    for (int v = 0; v < 4; v++) { w[v] = (double) pE[v]; w[4 + v] = (double) p1[v]; w[8 + v] = (double) p2[v]; }
    const bool b0 = c & 1, b1 = c & 2;
    double h[6];
#pragma unroll
    for (int q = 0; q < 6; q++) {
      const double keep = b0 ? w[2 * q + 1] : w[2 * q], give = b0 ? w[2 * q] : w[2 * q + 1];
      h[q] = keep + __shfl_xor(give, 1, 64);
    }
    double z[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const double keep = b1 ? h[2 * q + 1] : h[2 * q], give = b1 ? h[2 * q] : h[2 * q + 1];
      z[q] = keep + __shfl_xor(give, 2, 64);
      z[q] += __shfl_xor(z[q], 4, 64);
      z[q] += __shfl_xor(z[q], 8, 64);
    }
    if (c < 4 && myrow < nb) {
      double *b = a.bsum + 3 * (e0 + 16ll * ch + myrow);
#pragma unroll
      for (int q = 0; q < 3; q++) atomicAdd(&b[q], z[q]);
    }
  }
}

template<class T, int NL, bool PAIRS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 3 : 2))) void k_pair_bwd_mfma(PairMfmaArgs<T> a)
{
  constexpr int NLM = NL * NL;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int i, grp;
  if (!pair_block(a.ngrp, a.natoms, i, grp)) return;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int c = lane & 15, g = lane >> 4, nbk = a.C >> 4;
  T *Bw = reinterpret_cast<T *>(smem_raw) + (size_t) wave * (a.spw * NLM + 3) * 16;
  const int n0 = (wave % nbk) * 16, s0 = (grp * a.wpb + wave / nbk) * a.spw;      // channels and slots of the wave
  const int nq = a.nslot - s0 < a.spw ? a.nslot - s0 : a.spw;
  if (nq > 0) {
    const T *gp = a.gP + ((long long) i * a.nslot + s0) * NLM * a.C + n0 + c;
    for (int row = g; row < nq * NLM; row += 4) Bw[row * 16 + c] = gp[(long long) row * a.C];
    if (g < 3) Bw[(nq * NLM + g) * 16 + c] = (T) 0;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (nq == 4) pair_bwd_wave<T, NL, 4, PAIRS>(a, i, s0, n0, Bw);
  else if (nq == 3) pair_bwd_wave<T, NL, 3, PAIRS>(a, i, s0, n0, Bw);
  else if (nq == 2) pair_bwd_wave<T, NL, 2, PAIRS>(a, i, s0, n0, Bw);
  else if (nq == 1) pair_bwd_wave<T, NL, 1, PAIRS>(a, i, s0, n0, Bw);
}

// Values per row of the harmonics and their two gradient components in memory: more than 3 nlm (the last matrix step of an odd
// lmax reads one value past the row's third part, which the kernel replaces by zero), a whole number of 16-byte pieces, and an
// odd number of pairs (fp64) or fours (fp32), which kept 16 rows in different banks while the kernel copied them to LDS
inline int pair_row_stride(int nlm, size_t value_bytes)
{
  int v = 3 * nlm + 3;
  if (value_bytes == 8) while (v % 4 != 2) v++;
  else while (v % 8 != 4) v++;
  return v;
}

// Shape of a k_pair_bwd_mfma launch for nslot message functions of C channels in blocks of about `waves` waves: ok = false
// where the kernel does not apply (channels not in blocks of 16, lmax above 6)
struct PairMfmaPlan {
  bool ok = false;
  int spw = 0, wpb = 0, ngrp = 0, threads = 0, ystr = 0;
  size_t lds = 0;
};
inline PairMfmaPlan pair_mfma_plan(int nslot, int C, int nl, size_t value_bytes, int waves)
{
  PairMfmaPlan p;
  if (C % 16 != 0 || C > 128 || nl > 7 || nslot < 1) return p;
  const int nbk = C / 16, groups = (nslot + kPairMfmaSlots - 1) / kPairMfmaSlots;    // a wave per group and column block
  p.spw = (nslot + groups - 1) / groups;
  p.wpb = std::max(1, std::min(groups, waves / nbk));
  p.ngrp = (groups + p.wpb - 1) / p.wpb;
  p.threads = 64 * nbk * p.wpb;
  p.ystr = pair_row_stride(nl * nl, value_bytes);
  p.lds = pair_mfma_wave_lds(nl, p.spw, value_bytes) * (p.threads / 64);
  p.ok = p.lds <= kPairLdsMax && p.threads <= 512;
  return p;
}
// Waves of a block: those of one group of slots (blocks of 4 and 8 waves at 32 channels were 3 % slower, of 8 at 64 channels
// 4 %: a block keeps its place until its last wave is done)
inline int pair_mfma_waves(int asked) { return asked > 0 ? asked : 1; }

template<class T, bool PAIRS> inline auto pair_bwd_kernel(int nl) -> void (*)(PairMfmaArgs<T>)
{
  switch (nl) {
    case 1: return k_pair_bwd_mfma<T, 1, PAIRS>;
    case 2: return k_pair_bwd_mfma<T, 2, PAIRS>;
    case 3: return k_pair_bwd_mfma<T, 3, PAIRS>;
    case 4: return k_pair_bwd_mfma<T, 4, PAIRS>;
    case 5: return k_pair_bwd_mfma<T, 5, PAIRS>;
    case 6: return k_pair_bwd_mfma<T, 6, PAIRS>;
    default: return k_pair_bwd_mfma<T, 7, PAIRS>;
  }
}
// PAIRS: engines whose bonds may share radial rows (erow); without, erow is never set
template<class T, bool PAIRS> inline void launch_pair_bwd_mfma(const PairMfmaPlan &p, PairMfmaArgs<T> a, int nl, hipStream_t stream)
{
  void (*kern)(PairMfmaArgs<T>) = pair_bwd_kernel<T, false>(nl);
  if constexpr (PAIRS) if (a.erow) kern = pair_bwd_kernel<T, true>(nl);
  if (p.lds > 48 * 1024)
    HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int) p.lds));
  a.spw = p.spw;
  a.wpb = p.wpb;
  a.ngrp = p.ngrp;
  a.ystr = p.ystr;
  hipLaunchKernelGGL(kern, dim3((unsigned) ((a.natoms + 7) / 8 * 8 * p.ngrp)), dim3(p.threads), p.lds, stream, a);
}

struct Energy2Dev {
  const double *W[7];         // [n_in][n_out]
  double norm[7];
  int nin[7], nout[7];
  int nlay, act, ln, nrho, rms, width;    // width: largest layer width (LDS row of the kernel)
  double out_scale, eps;
  const double *shift;        // [nel]
  const double *lnI;          // [nrho - 1] scale of the only_nonlin RMSNorm of rho
  const double *ln0;          // [nrho]     scale of the full RMSNorm of I2
};

// as k_energy_2l below, by 16 lanes per atom: networks of one hidden layer (k_energy_hidden of GRACE-1L)
static __global__ __launch_bounds__(256) void k_energy_2l_hidden(Energy2Dev M, const int *__restrict__ mu, int natoms, const double *__restrict__ rho,
                                                                 const double *__restrict__ I2, double *__restrict__ grho, double *__restrict__ gI2,
                                                                 double *eatom, double *energy, int want_grad, const int *sid)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double *lds = reinterpret_cast<double *>(smem_raw);
  const int p = threadIdx.x & 15, nr = M.nrho, nin = nr - 1;
  readout_stage(lds, M.W[0], M.W[1], nin, M.nout[0]);
  const double lnI = p < nin ? M.lnI[p] : 0.0, ln0 = p < nin ? M.ln0[p + 1] : 0.0, lnF = M.ln0[0];
  double esum = 0.0;
  for (int b0 = blockIdx.x * 16; b0 < natoms; b0 += gridDim.x * 16) {    // uniform over the block
    const int at = b0 + (threadIdx.x >> 4);
    const bool ok = at < natoms;
    const double *r = rho + (long long) (ok ? at : 0) * nr, *i2 = I2 + (long long) (ok ? at : 0) * nr;
    const double rf = r[0], jf = i2[0], rp = p < nin ? r[p + 1] : 0.0, jp = p < nin ? i2[p + 1] : 0.0;    // channel 0, and channel p + 1
    const double s1 = M.rms ? sqrt(readout_sum(rp * rp) / nin + M.eps) : 1.0, s0 = M.rms ? sqrt((readout_sum(jp * jp) + jf * jf) / nr + M.eps) : 1.0;
    const double x0 = rp / s1 * lnI + jp / s0 * ln0;
    const double q = M.ln ? readout_ln(x0, nin) : 1.0;
    double g;
    const double e = readout_net(lds, M.nout[0], M.norm[0], M.norm[1], M.act, x0 * q, p, want_grad, M.out_scale, g);
    if (ok && p == 0) {
      const double Ei = (e + rf + jf / s0 * lnF) * M.out_scale + M.shift[mu[at]];
      if (eatom) eatom[at] = Ei;
      if (!energy) {}    // ordered sums: the records are added from eatom afterwards
      else if (sid) atomicAdd(energy + record_of(sid, at), Ei);
      else esum += Ei;
    }
    if (!want_grad) continue;
    if (M.ln) g = readout_ln_bwd(g, x0, q, nin);
    // RMSNorm reverses (y_k = x_k s_k / sigma)
    double t1 = 0.0, t0 = 0.0;
    if (M.rms) {
      t1 = readout_sum(g * lnI * rp);
      t0 = readout_sum(g * ln0 * jp) + M.out_scale * lnF * jf;
    }
    if (!ok) continue;    // no exchange between lanes below
    double *gr = grho + (long long) at * nr, *gi = gI2 + (long long) at * nr;
    if (p == 0) {
      gr[0] = M.out_scale;
      gi[0] = M.out_scale * lnF / s0 - jf * t0 / (nr * s0 * s0 * s0);
    }
    if (p < nin) {
      gr[p + 1] = g * lnI / s1 - rp * t1 / (nin * s1 * s1 * s1);
      gi[p + 1] = g * ln0 / s0 - jp * t0 / (nr * s0 * s0 * s0);
    }
  }
  if (!sid && energy) readout_add(esum, energy);
}

// E_i = (MLP(x) + rho[0] + I2[0] ln0[0] / s0) out_scale + shift,  x_k = rho[k] lnI[k-1] / s1 + I2[k] ln0[k] / s0,
// s1 = sqrt(mean rho[1:]^2 + eps), s0 = sqrt(mean I2^2 + eps); dE/drho, dE/dI2.  One wave per atom, fp64; a layer with
// fewer than 33 outputs splits each dot product over 64 / outputs lanes.
static __global__ void k_energy_2l(Energy2Dev M, const int *mu, int natoms, const double *rho, const double *I2, double *grho, double *gI2,
                            double *eatom, double *energy, int want_grad, const int *sid)
{
  // LDS rows of W = M.width values: nlay + 1 activations, nlay pre-activations, 2 adjoint buffers, x0
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int W = M.width;
  double *act_ = reinterpret_cast<double *>(smem_raw), *pre_ = act_ + (M.nlay + 1) * W, *gbuf_ = pre_ + M.nlay * W, *x0 = gbuf_ + 2 * W;
#define act(L_, k_) act_[(L_) * W + (k_)]
#define pre(L_, k_) pre_[(L_) * W + (k_)]
#define gbuf(L_, k_) gbuf_[(L_) * W + (k_)]
  const int at = blockIdx.x, lane = threadIdx.x;
  const double *r = rho + (long long) at * M.nrho, *i2 = I2 + (long long) at * M.nrho;
  const int nr = M.nrho, n0 = nr - 1;
  double ms1 = 0.0, ms0 = 0.0;
  for (int k = lane; k < nr; k += 64) {
    if (k > 0) ms1 += r[k] * r[k];
    ms0 += i2[k] * i2[k];
  }
  for (int o = 32; o > 0; o >>= 1) { ms1 += __shfl_xor(ms1, o, 64); ms0 += __shfl_xor(ms0, o, 64); }
  const double s1 = M.rms ? sqrt(ms1 / n0 + M.eps) : 1.0, s0 = M.rms ? sqrt(ms0 / nr + M.eps) : 1.0;
  for (int k = lane; k < n0; k += 64) act(0, k) = r[k + 1] / s1 * M.lnI[k] + i2[k + 1] / s0 * M.ln0[k + 1];
  __syncthreads();
  double q = 0.0;
  if (M.ln) {
    double ms = 0.0;
    for (int k = lane; k < n0; k += 64) { x0[k] = act(0, k); ms += act(0, k) * act(0, k); }
    for (int o = 32; o > 0; o >>= 1) ms += __shfl_xor(ms, o, 64);
    q = 1.0 / sqrt(ms / n0 + 1e-16);
    for (int k = lane; k < n0; k += 64) act(0, k) *= q;
    __syncthreads();
  }
  // lanes that share one output of a layer: the largest power of two g with outputs x g <= 64
  auto group = [](int nout_) {
    int g = 1;
    while (g < 64 && nout_ * (g * 2) <= 64) g *= 2;
    return g;
  };
  for (int L = 0; L < M.nlay; L++) {
    const int no = M.nout[L], ni = M.nin[L], g = group(no), p = lane % g;
    for (int c0 = 0; c0 < no; c0 += 64 / g) {    // every lane walks the loop: the exchanges need the whole wave
      const int c = c0 + lane / g;
      double s = 0.0;
      if (c < no) {
#pragma unroll 4
        for (int a = p; a < ni; a += g) s += act(L, a) * M.W[L][(long long) a * no + c];
      }
      for (int o = g >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (c < no && p == 0) {
        s *= M.norm[L];
        pre(L, c) = s;
        act(L + 1, c) = (L < M.nlay - 1) ? (M.act == 1 ? tanh(s) : s / (1.0 + exp(-s))) : s;
      }
    }
    __syncthreads();
  }
  const double Ei = (act(M.nlay, 0) + r[0] + i2[0] / s0 * M.ln0[0]) * M.out_scale + M.shift[mu[at]];
  if (lane == 0) {
    if (eatom) eatom[at] = Ei;
    if (energy) atomicAdd(energy + record_of(sid, at), Ei);    // null: ordered sums, the records are added from eatom afterwards
  }
  if (!want_grad) return;
  int cur = 0;
  if (lane == 0) gbuf(0, 0) = M.out_scale;
  __syncthreads();
  for (int L = M.nlay - 1; L >= 0; L--) {
    if (L < M.nlay - 1) {
      for (int c = lane; c < M.nout[L]; c += 64) {
        const double v = pre(L, c);
        if (M.act == 1) {
          const double tt = act(L + 1, c);
          gbuf(cur, c) *= 1.0 - tt * tt;
        } else {
          const double sg = 1.0 / (1.0 + exp(-v));
          gbuf(cur, c) *= sg * (1.0 + v * (1.0 - sg));
        }
      }
      __syncthreads();
    }
    {
      const int no = M.nout[L], ni = M.nin[L], g = group(ni), p = lane % g;
      for (int b0 = 0; b0 < ni; b0 += 64 / g) {
        const int a = b0 + lane / g;
        double s = 0.0;
        if (a < ni) {
#pragma unroll 4
          for (int c = p; c < no; c += g) s += gbuf(cur, c) * M.W[L][(long long) a * no + c];
        }
        for (int o = g >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (a < ni && p == 0) gbuf(cur ^ 1, a) = s * M.norm[L];
      }
    }
    cur ^= 1;
    __syncthreads();
  }
  if (M.ln) {
    double tt = 0.0;
    for (int k = lane; k < n0; k += 64) tt += gbuf(cur, k) * x0[k];
    for (int o = 32; o > 0; o >>= 1) tt += __shfl_xor(tt, o, 64);
    for (int k = lane; k < n0; k += 64) gbuf(cur, k) = q * (gbuf(cur, k) - x0[k] * tt * q * q / n0);
    __syncthreads();
  }
  // gbuf(cur, k-1) = dE/dx_k; RMSNorm reverses (y_k = x_k s_k / sigma)
  double t1 = 0.0, t0 = 0.0;
  if (M.rms) {
    for (int k = lane; k < nr; k += 64) {
      const double gy = k == 0 ? M.out_scale : gbuf(cur, k - 1);
      if (k > 0) t1 += gy * M.lnI[k - 1] * r[k];
      t0 += gy * M.ln0[k] * i2[k];
    }
    for (int o = 32; o > 0; o >>= 1) { t1 += __shfl_xor(t1, o, 64); t0 += __shfl_xor(t0, o, 64); }
  }
  double *gr = grho + (long long) at * nr, *gi = gI2 + (long long) at * nr;
  for (int k = lane; k < nr; k += 64) {
    const double gy = k == 0 ? M.out_scale : gbuf(cur, k - 1);
    gr[k] = k == 0 ? M.out_scale : gy * M.lnI[k - 1] / s1 - r[k] * t1 / (n0 * s1 * s1 * s1);
    gi[k] = gy * M.ln0[k] / s0 - i2[k] * t0 / (nr * s0 * s0 * s0);
  }
#undef act
#undef pre
#undef gbuf
}

}    // namespace grhip
